// Adjoint kernel: lnL and dlnL/dtheta for a batch of parameter vectors (FP64).
//
// The Kepler solve is differentiated implicitly: from E - e sin E = M,
//   dE/dM = 1/(1 - e cos E),  dE/de|_M = sin E/(1 - e cos E),
// so no derivative flows through the solver's iterations.  With
// D = 1 - e cos E, b = sqrt(1 - e^2), cos f = (cos E - e)/D, sin f = b sin E/D,
// the planet term mu = A (cos(f + w) + e cos w) has
//   dmu/dM = -A sin(f + w) b / D^2
//   dmu/de = -A sin(f + w) (b sin E / D^2 + sin E/(b D)) + A cos w
//   dmu/dw = -A (sin(f + w) + e sin w),   dmu/dA = cos(f + w) + e cos w.
// Without the moving average dlnL/dmu_i = r_i / err2_i and
// dlnL/dJ_k = J_k sum_{i in k} (r_i^2/err2_i^2 - 1/err2_i).
//
// MA(1) (moav01.model:7-15; per instrument for the intended semantics):
// eps_i = r_i + a_i eps_{i-1}, a_i = -c exp(-dt_i / tau), and lnL sums
// -(eps_i^2 / err2_i + ln err2_i) / 2.  Its adjoint lambda_i = dlnL/deps_i
// obeys the reverse recurrence lambda_i = -eps_i / err2_i + a_{i+1}
// lambda_{i+1}; then dlnL/dmu_i = -lambda_i, dlnL/dc = sum lambda_i
// eps_{i-1} da_i/dc and dlnL/dtau likewise, with eps in place of r in the
// jitter term.  The kernel makes two passes: the forward likelihood, which
// stores eps_i (scratch, one row per vector), then the epochs in reverse
// (tiles, then chunks), where the planet terms and their derivatives are
// recomputed and lambda comes from a suffix scan with the carry running
// backwards.
//
// Terms added after the moving average, S_i = sum_j zeta_j a_ij (activity
// columns) + sum_c A_c cos(f_c t_i + ph_c) (sinusoid, magnetic cycle): dlnL/dS_i
// is the final residual over err2_i and does not pass through the MA adjoint:
//   dS/dzeta_j = a_ij, dS/dA = cos M, dS/dph = -A sin M, dS/df = -A sin M t,
//   df/dP = -f/P.
//
// The natural-parameter gradients are then mapped to the block's
// parameterisation (block_repo.py:23-31) once per vector.
#include <cmath>
#include <cstdlib>
#include <mutex>

#include "emp_kernels.h"

using namespace emp;

struct GradLDS {
    double g[MAXD];            // gradient w.r.t. the full vector
    double nat[KMAX][5];       // per planet: (M*tau, M, e, w, A) sums
    double cosg[CMAX][3];      // per cosine term: (A, phase, frequency) sums
};

// Per-wave partial sums, added over a slot's waves in wave order at the end,
// so that the gradient does not depend on how the waves were scheduled.
// acc: offsets, jitters, MA coefficients and timescales (one entry per
// (set, order), order-minor; orders above 1 only in the EXT = 2 instances),
// then, with the terms added after the MA, the cosine terms and the activity
// coefficients.  nat: per planet the five natural-parameter sums, then the
// acceleration coefficients.
template <int EXT>
struct GradWave {
    static constexpr int QM = EXT == 2 ? 4 : 1;
    static constexpr int OFF = 0, JIT = IMAX, MAC = 2 * IMAX, MAT = MAC + IMAX * QM, COS = MAT + IMAX * QM;
    static constexpr int SAI = COS + (EXT >= 1 ? 3 * CMAX : 0);
    static constexpr int N = SAI + (EXT >= 1 ? SAIMAX : 0);
};
constexpr int WN_ACC = KMAX * 5, WN_N = KMAX * 5 + AMAX;
template <int EXT, int NW = NWAVES>
struct GradWaveLDS {
    double acc[NW][GradWave<EXT>::N];
    double nat[NW][WN_N];
};

// w times the derivatives of one planet's term at time t with respect to its
// natural parameters, added to a = (dmu/dM tau, dmu/dM, dmu/de, dmu/dw,
// dmu/dA).  With D = 1 - e cos E, b = sqrt(1 - e^2) (per planet, pc.bq):
// D cos f = cos E - e, D sin f = b sin E.
template <int PREC, class KTE>
__device__ __forceinline__ void planet_wgrad(const PlanetC& pc, const SinCosTab& tab, const KTE* kt, double t,
                                             double w, double (&a)[5], bool tp, int kmode) {
    double sE1[1], cE1[1], rD1[1];
    planet_sc<PREC, 1>(pc, tab, kt, {t}, sE1, cE1, rD1, tp, kmode);
    const double sE = sE1[0], cE = cE1[0], rD = rD1[0];
    const double e = pc.e;
    const double u = cE - e, v = pc.bq * sE;
    const double sfw = __builtin_fma(v, pc.cw, u * pc.sw) * rD;     // sin(f + w)
    const double cfw = __builtin_fma(u, pc.cw, -(v * pc.sw)) * rD;  // cos(f + w)
    const double wA = w * pc.K;
    const double ws = wA * sfw;
    const double dM = -(ws * pc.bq) * (rD * rD);
    const double tau = tp ? t - pc.tp : t;
    a[0] = __builtin_fma(dM, tau, a[0]);
    a[1] += dM;
    a[2] = __builtin_fma(-ws, sE * rD * __builtin_fma(pc.bq, rD, pc.ibq), __builtin_fma(wA, pc.cw, a[2]));
    a[3] = __builtin_fma(-wA, __builtin_fma(e, pc.sw, sfw), a[3]);
    a[4] = __builtin_fma(w, __builtin_fma(e, pc.cw, cfw), a[4]);
}

// (x, y) exchanged between lanes 32 apart by v_permlane32_swap, which swaps
// the upper half of its first operand with the lower half of its second:
// lanes 0-31 end with (x, x of lane + 32), lanes 32-63 with (y of lane - 32,
// y), so the sum holds x summed over the pair below and y above.
__device__ __forceinline__ double swap_add32(double x, double y) {
    const long long xi = __double_as_longlong(x), yi = __double_as_longlong(y);
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)xi, (unsigned)yi, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(xi >> 32), (unsigned)(yi >> 32), false, false);
    return __longlong_as_double(((long long)hi[0] << 32) | lo[0]) +
           __longlong_as_double(((long long)hi[1] << 32) | lo[1]);
}

// The same between lanes 16 apart within each half (v_permlane16_swap):
// x summed over the pair where lane bit 4 is 0, y where it is 1.
__device__ __forceinline__ double swap_add16(double x, double y) {
    const long long xi = __double_as_longlong(x), yi = __double_as_longlong(y);
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)xi, (unsigned)yi, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(xi >> 32), (unsigned)(yi >> 32), false, false);
    return __longlong_as_double(((long long)hi[0] << 32) | lo[0]) +
           __longlong_as_double(((long long)hi[1] << 32) | lo[1]);
}

// Sum of five per-lane values over the wave, scattered: the values are
// paired across lanes 32 apart as (v0, v4), (v1, v2), (v3, v3) (permlane
// swaps: each lane keeps the member its lane bit selects, summed with its
// partner's), those across lanes 16 apart as (v0|v4, v1|v2) and (v3, v3),
// the two results across lanes 8 apart (DPP), and the remaining value is
// summed over each aligned group of eight lanes.  The totals land at lanes
// 0 (v0), 16 (v1), 48 (v2), 8 (v3) and 32 (v4); red5_index(lane) names the
// value a lane holds, -1 for lanes that hold none.  Whole wave active.
__device__ __forceinline__ double wave_reduce5(const double (&v)[5], int lane) {
    const double a0 = swap_add32(v[0], v[4]);
    const double a1 = swap_add32(v[1], v[2]);
    const double a2 = swap_add32(v[3], v[3]);
    const double b0 = swap_add16(a0, a1);
    const double b1 = swap_add16(a2, a2);
    const bool h3 = lane & 8;
    double c = (h3 ? b1 : b0) + dpp_mov_f64<0x128>(h3 ? b0 : b1);   // row_ror 8: lane ^ 8
    c += dpp_mov_f64<0x141>(c);    // row_half_mirror: lane i with 7 - i of its group of 8
    c += dpp_mov_f64<0xB1>(c);     // quad_perm [1, 0, 3, 2]
    c += dpp_mov_f64<0x4E>(c);     // quad_perm [2, 3, 0, 1]
    return c;
}

// Nibble g of 0xF2F4F130 is the value lane 8 g holds (F: none).
__device__ __forceinline__ int red5_index(int lane) {
    const int i = (int)((0xF2F4F130u >> (4 * (lane >> 3))) & 0xFu);
    return ((lane & 7) || i == 0xF) ? -1 : i;
}

// Four values: (v0, v1) and (v2, v3) across lanes 32 apart, the pair across
// lanes 16 apart, then summed over each row of 16 lanes.  The totals land at
// lanes 0 (v0), 32 (v1), 16 (v2) and 48 (v3): red4_index(lane).
__device__ __forceinline__ double wave_reduce4(const double (&v)[4]) {
    const double a0 = swap_add32(v[0], v[1]);
    const double a1 = swap_add32(v[2], v[3]);
    double c = swap_add16(a0, a1);
    c += dpp_mov_f64<0x128>(c);
    c += dpp_mov_f64<0x141>(c);
    c += dpp_mov_f64<0xB1>(c);
    c += dpp_mov_f64<0x4E>(c);
    return c;
}

__device__ __forceinline__ int red4_index(int lane) {
    return (lane & 15) ? -1 : (int)((0x3120u >> (4 * (lane >> 4))) & 0xFu);
}

// The five sums added to dst[0..4], the first n of four to dst[0..n).
__device__ __forceinline__ void wave_reduce_add5(const double (&v)[5], double* dst, int lane, int ri) {
    const double c = wave_reduce5(v, lane);
    if (ri >= 0) dst[ri] += c;
}

__device__ __forceinline__ void wave_reduce_add4(const double (&v)[4], int n, double* dst, int ri4) {
    const double c = wave_reduce4(v);
    if (ri4 >= 0 && ri4 < n) dst[ri4] += c;
}

// Adds w = dlnL/dS_n times the derivatives of the terms added after the MA
// at epoch n (time t, instrument k): entry e of the cosine terms' sums, then of
// the activity coefficients' (from 3 CMAX on) at acc[e << cl].
template <int EXT, class SL>
__device__ __forceinline__ void post_accumulate(const ModelDev& md, const SL& sl, const SinCosTab& tab, double t,
                                                int n, int k, double w, double* acc, int cl) {
    if (md.sai_w) {
        const int b0 = md.sai_base[k], nc = md.sai_base[k + 1] - b0;
        for (int c = 0; c < nc; ++c) atomicAdd(&acc[(3 * CMAX + b0 + c) << cl], w * md.sai[(size_t)c * md.N + n]);
    }
    for (int c = 0; c < md.n_cos; ++c) {
        const double r = reduce_2pi(cos_phase(sl, c, t));
        double sn, cs;
        sincos_tab(tab, __builtin_fabs(r), sn, cs);
        const double dph = -sl.cosw[c][0] * (r < 0.0 ? -sn : sn);
        atomicAdd(&acc[(3 * c + 0) << cl], w * cs);
        atomicAdd(&acc[(3 * c + 1) << cl], w * dph);
        atomicAdd(&acc[(3 * c + 2) << cl], w * dph * t);
    }
}

// Adjoint of MA(q), q >= 2, for one chunk (epochs in reverse): with
// a_{n,c} the forward multipliers, lambda_n = u_n + sum_{c<q} a_{n+1+c,c}
// lambda_{n+1+c}, an affine map on the state (lambda_n, ..., lambda_{n+Q-1})
// whose companion matrix has first row (a_{n+1,0}, ..., a_{n+Q,Q-1}).  Maps
// are composed from the wave's last lane down (suffix), then across the
// slot's waves from the last one.  `carry` is the state after the chunk
// (updated to the state before it).  Reads the tile before the barrier.
template <int Q, int WPT, class SL>
__device__ __forceinline__ double lam_chunk_q(const ModelDev& md, const SL& sl, const TileLDS& tl, bool valid,
                                              int j, int tb, int tn, double t, int k, double u, int lane, int wave,
                                              int wsub, int& parity, double (&carry)[4]) {
    __shared__ double qtot[2][MAX_WAVES][Q * Q + Q];
    double m[Q][Q], v[Q];
#pragma unroll
    for (int a = 0; a < Q; ++a) {
        v[a] = 0.0;
#pragma unroll
        for (int b = 0; b < Q; ++b) m[a][b] = a == b ? 1.0 : 0.0;
    }
    if (valid) {
        const int q = md.ma_q, n = tb + j;
        const double* ph = sl.theta + md.off_ma + 2 * q * (md.ma_global ? 0 : k);
#pragma unroll
        for (int c = 0; c < Q; ++c) {
            double a = 0.0;
            const int n2 = n + 1 + c, j2 = j + 1 + c;
            if (c < q && n2 < md.N) {
                const int k2 = j2 < tn ? tl.ins[j2] : md.ins[n2];
                if (md.ma_global || k2 == k) {
                    const double t2 = j2 < tn ? tl.t[j2] : md.t[n2];
                    a = -(ph[2 * c] * exp(-__builtin_fabs(t2 - t) / ph[2 * c + 1]));
                }
            }
            m[0][c] = a;
        }
#pragma unroll
        for (int a = 1; a < Q; ++a)
#pragma unroll
            for (int b = 0; b < Q; ++b) m[a][b] = b == a - 1 ? 1.0 : 0.0;
        v[0] = u;
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        double pm[Q][Q], pv[Q];
#pragma unroll
        for (int a = 0; a < Q; ++a) {
#pragma unroll
            for (int b = 0; b < Q; ++b) pm[a][b] = __shfl_down(m[a][b], o, 64);
            pv[a] = __shfl_down(v[a], o, 64);
        }
        if (lane + o < 64) {
            double nm[Q][Q], nv[Q];
#pragma unroll
            for (int a = 0; a < Q; ++a) {
                double acc = v[a];
#pragma unroll
                for (int b = 0; b < Q; ++b) acc = __builtin_fma(m[a][b], pv[b], acc);
                nv[a] = acc;
#pragma unroll
                for (int c = 0; c < Q; ++c) {
                    double e = 0.0;
#pragma unroll
                    for (int b = 0; b < Q; ++b) e = __builtin_fma(m[a][b], pm[b][c], e);
                    nm[a][c] = e;
                }
            }
#pragma unroll
            for (int a = 0; a < Q; ++a) {
                v[a] = nv[a];
#pragma unroll
                for (int c = 0; c < Q; ++c) m[a][c] = nm[a][c];
            }
        }
    }
    double sin_[Q];
    if (WPT == 1) {
#pragma unroll
        for (int a = 0; a < Q; ++a) sin_[a] = carry[a];
    } else {
        if (lane == 0) {
#pragma unroll
            for (int a = 0; a < Q; ++a) {
#pragma unroll
                for (int b = 0; b < Q; ++b) qtot[parity][wave][a * Q + b] = m[a][b];
                qtot[parity][wave][Q * Q + a] = v[a];
            }
        }
        __syncthreads();
        const int w0 = wave - wsub;
        double s_all[Q];
#pragma unroll
        for (int a = 0; a < Q; ++a) s_all[a] = carry[a];
        for (int w = WPT - 1; w >= 0; --w) {
            if (w == wsub) {
#pragma unroll
                for (int a = 0; a < Q; ++a) sin_[a] = s_all[a];
            }
            const double* T = qtot[parity][w0 + w];
            double ns[Q];
#pragma unroll
            for (int a = 0; a < Q; ++a) {
                double acc = T[Q * Q + a];
#pragma unroll
                for (int b = 0; b < Q; ++b) acc = __builtin_fma(T[a * Q + b], s_all[b], acc);
                ns[a] = acc;
            }
#pragma unroll
            for (int a = 0; a < Q; ++a) s_all[a] = ns[a];
        }
#pragma unroll
        for (int a = 0; a < Q; ++a) carry[a] = s_all[a];
        parity ^= 1;
    }
    double st[Q];
#pragma unroll
    for (int a = 0; a < Q; ++a) {
        double acc = v[a];
#pragma unroll
        for (int b = 0; b < Q; ++b) acc = __builtin_fma(m[a][b], sin_[b], acc);
        st[a] = acc;
    }
    if (WPT == 1) {
#pragma unroll
        for (int a = 0; a < Q; ++a) carry[a] = __shfl(st[a], 0, 64);
    }
    return st[0];
}

// Per-lane sums of the per-instrument gradient terms (offset, jitter, MA(1)
// coefficient and timescale) of the lane's epochs, kept in registers while
// the lane's instrument stays the same and added to the wave's LDS sums when
// it changes (epochs grouped by instrument, as the per-instrument MA orders
// them, change instrument a few times per lane in a whole pass), instead of
// four same-address LDS atomics per epoch.
struct InsAcc {
    int k = -1;
    double off = 0.0, jit = 0.0, mac = 0.0, mat = 0.0;
    template <int EXT>
    __device__ __forceinline__ void flush(double* wacc) {
        using GW = GradWave<EXT>;
        if (k < 0) return;
        atomicAdd(&wacc[GW::OFF + k], off);
        atomicAdd(&wacc[GW::JIT + k], jit);
        atomicAdd(&wacc[GW::MAC + k * GW::QM], mac);
        atomicAdd(&wacc[GW::MAT + k * GW::QM], mat);
        off = jit = mac = mat = 0.0;
    }
    template <int EXT>
    __device__ __forceinline__ void to(int kk, double* wacc) {
        if (kk != k) {
            flush<EXT>(wacc);
            k = kk;
        }
    }
};

// The MA adjoint at one chunk of a tile taken in reverse: lambda of the
// lane's epoch from eps (the forward pass's scratch row), with the carry from
// the later epochs; returns w = dlnL/dmu = -lambda (0 for an invalid lane)
// after adding the epoch's offset, jitter, post-MA and MA-parameter terms.
template <int PREC, int WPT, int EXT, class SL>
__device__ __forceinline__ double ma_chunk_w(const ModelDev& md, const SL& sl, const TileLDS& tl, ScanLDS& sc,
                                             const double* eps, double* wacc, InsAcc& ia, bool valid, int j, int tb,
                                             int tn, int lane, int wave, int wsub, int& parity, double& lam_carry,
                                             double (&lq_carry)[4]) {
    using GW = GradWave<EXT>;
    constexpr bool POST = EXT >= 1;
    const bool maq = EXT == 2 && md.ma_q > 1;
    double u = 0.0, amul = 1.0, ie = 0.0, t = 0.0, ef = 0.0;
    int k = 0;
    if (valid) {
        t = tl.t[j];
        k = tl.ins[j];
        const double err2 = tl.s2[j] + sl.jit2[k];
        ie = rcp_path<PREC>(err2);
        const double e_i = eps[tb + j];
        ef = (POST && has_post(md)) ? e_i - epoch_post(md, sl, tl.tab, t, tb + j, k) : e_i;
        u = -ef * ie;
        const int n1 = tb + j + 1;     // the next epoch's multiplier
        amul = 0.0;
        if (!maq && n1 < md.N) {
            const bool in_tile = j + 1 < tn;
            const int k1 = in_tile ? tl.ins[j + 1] : md.ins[n1];
            const double c1 = in_tile ? tl.dt[j + 1] : md.dt[n1];
            amul = ma_mult(md, sl, k1, c1);
        }
    }
    double sa = amul, sb = u;
    double lam = 0.0;
    if (maq) {
        lam = md.ma_q == 2
                  ? lam_chunk_q<2, WPT>(md, sl, tl, valid, j, tb, tn, t, k, u, lane, wave, wsub, parity, lq_carry)
                  : lam_chunk_q<4, WPT>(md, sl, tl, valid, j, tb, tn, t, k, u, lane, wave, wsub, parity, lq_carry);
    } else if (WPT == 1) {
        wave_affine_suffix_scan(sa, sb, lane);
        lam = __builtin_fma(sa, lam_carry, sb);
        lam_carry = __shfl(lam, 0, 64);
    } else {
        wave_affine_suffix_scan(sa, sb, lane);
        if (lane == 0) sc.tot[parity][wave] = make_double2(sa, sb);
        __syncthreads();
        const int w0 = wave - wsub;
        double pa = 1.0, pb = 0.0;
        for (int w = WPT - 1; w >= 0; --w) {
            if (w == wsub) lam = __builtin_fma(sa, __builtin_fma(pa, lam_carry, pb), sb);
            const double ta = sc.tot[parity][w0 + w].x, tbv = sc.tot[parity][w0 + w].y;
            pb = __builtin_fma(ta, pb, tbv);
            pa = ta * pa;
        }
        lam_carry = __builtin_fma(pa, lam_carry, pb);
        parity ^= 1;
    }
    if (!valid) return 0.0;
    const double w = -lam;
    ia.to<EXT>(k, wacc);
    ia.off += w;
    if (md.has_jit) ia.jit = __builtin_fma(sl.jit[k], ef * ef * ie * ie - ie, ia.jit);
    if (POST && has_post(md)) post_accumulate<EXT>(md, sl, tl.tab, t, tb + j, k, -u, wacc + GradWave<EXT>::COS, 0);
    if (maq) {
        // d a_{n,c} / d phi_c = -exp(-dt / tau_c), d a_{n,c} / d tau_c = a_{n,c} dt / tau_c^2
        const int n = tb + j, set = md.ma_global ? 0 : k;
        const double* ph = sl.theta + md.off_ma + 2 * md.ma_q * set;
        for (int c = 0; c < md.ma_q; ++c) {
            const int n1 = n - 1 - c, j1 = j - 1 - c;
            if (n1 < 0) break;
            const int k1 = j1 >= 0 ? tl.ins[j1] : md.ins[n1];
            if (!(md.ma_global || k1 == k)) break;
            const double dt = __builtin_fabs(t - (j1 >= 0 ? tl.t[j1] : md.t[n1]));
            const double tau = ph[2 * c + 1];
            const double wgt = exp(-dt / tau);
            const double le = lam * eps[n1];
            atomicAdd(&wacc[GW::MAC + set * GW::QM + c], le * -wgt);
            atomicAdd(&wacc[GW::MAT + set * GW::QM + c], le * -(ph[2 * c] * wgt * dt / (tau * tau)));
        }
    } else {
        // da_i/dc = a_i / c, da_i/dtau = a_i dt / tau^2 (a_i = 0 at a segment start)
        const double col = tl.dt[j];
        const bool start = md.ma_wfixed ? col == 0.0 : col < 0.0;
        if (!start) {
            const int n = tb + j;
            const double le = lam * eps[n - 1];
            const double wgt = md.ma_wfixed ? col : exp(-col / sl.ma_tau[k]);
            if (md.ma_global) {
                atomicAdd(&wacc[GW::MAC], le * -wgt);
                if (!md.ma_wfixed) {
                    const double tau = sl.ma_tau[k];
                    atomicAdd(&wacc[GW::MAT], le * -(sl.ma_c[k] * wgt * col / (tau * tau)));
                }
            } else {
                ia.mac = __builtin_fma(le, -wgt, ia.mac);
                if (!md.ma_wfixed) {
                    const double tau = sl.ma_tau[k];
                    ia.mat = __builtin_fma(le, -(sl.ma_c[k] * wgt * col / (tau * tau)), ia.mat);
                }
            }
        }
    }
    return w;
}

// Without the MA: the lane's epoch's residual, its share of chi^2 and of the
// log-determinant, w = dlnL/dmu = r / err2 and the epoch's offset, jitter and
// post-MA terms.
template <int PREC, int EXT, class SL>
__device__ __forceinline__ double plain_w(const ModelDev& md, const SL& sl, const TileLDS& tl, double* wacc,
                                          InsAcc& ia, int j, int tb, double& chi, double& prod, int& pexp,
                                          int kmask) {
    using GW = GradWave<EXT>;
    constexpr bool POST = EXT >= 1;
    const double t = tl.t[j];
    const int k = tl.ins[j];
    double mu1[1];
    epoch_mu<PREC, 1>(md, sl, tl.tab, {t}, {k}, kmask, mu1);
    const double mu = mu1[0];
    const double err2 = tl.s2[j] + sl.jit2[k];
    const double cs = (POST && has_post(md)) ? epoch_post(md, sl, tl.tab, t, tb + j, k) : 0.0;
    const double r = tl.y[j] - mu - cs;
    const double ie = rcp_path<PREC>(err2);
    const double w = r * ie;
    chi = __builtin_fma(r * r, ie, chi);
    prod *= err2;
    pexp += __builtin_amdgcn_frexp_exp(prod);
    prod = __builtin_amdgcn_frexp_mant(prod);
    ia.to<EXT>(k, wacc);
    ia.off += w;
    if (md.has_jit) ia.jit = __builtin_fma(sl.jit[k], w * w - ie, ia.jit);
    if (POST && has_post(md)) post_accumulate<EXT>(md, sl, tl.tab, t, tb + j, k, w, wacc + GradWave<EXT>::COS, 0);
    return w;
}

// The single-pass kernel's sums over the epochs, with C = cos f, S = sin f / b,
// s = sin(f + w), q = 1 + e C = b^2 / D and tau the time the phase counts from:
//   n0 = sum w s q^2 tau, n1 = sum w s q^2, n2 = sum w s S (q + 1),
//   n3 = sum w C, n4 = sum w S,
// to the sums of w times the natural-parameter derivatives (those of
// planet_wgrad): the constants of the planet and the parts that do not depend
// on the epoch (wsum = sum w) come in once per vector instead of per epoch.
__device__ __forceinline__ void nat_basis(const PlanetC& pc, double wsum, double (&n)[5]) {
    const double kb = -pc.K * pc.ibq * pc.ibq * pc.ibq, bs = pc.bq * n[4], ew = pc.e * wsum;
    n[0] *= kb;
    n[1] *= kb;
    n[2] = pc.K * (pc.cw * wsum - pc.ibq * n[2]);
    n[4] = pc.cw * ew + (pc.cw * n[3] - pc.sw * bs);
    n[3] = -pc.K * (pc.sw * ew + (pc.sw * n[3] + pc.cw * bs));
}

// Adds the per-wave partial sums of a slot in wave order, maps the natural
// gradients to the parameterisation and writes lnL and the free gradient of
// vector b.  All threads of the workgroup call this (it holds barriers).
// BASIS: the planets' sums are those of the single-pass kernel (nat_basis).
template <int EXT, int WPT, bool BASIS = false, int NW = NWAVES, class SL>
__device__ __forceinline__ void grad_finish(const ModelDev& md, const SL& sl, GradLDS& gl,
                                            const GradWaveLDS<EXT, NW>& s_gw, bool live, int wave, int wsub, int lane,
                                            double lnl_v, int64_t b, double* __restrict__ out_lnl,
                                            double* __restrict__ out_grad, unsigned long long* nonfinite, int* stale) {
    using GW = GradWave<EXT>;
    constexpr bool POST = EXT >= 1;
    __syncthreads();
    if (live && wsub == 0) {
        const int w0 = wave;
        for (int e = lane; e < GW::N; e += 64) {
            double v = 0.0;
            for (int w = 0; w < WPT; ++w) v += s_gw.acc[w0 + w][e];
            if (POST && e >= GW::SAI) {
                if (md.sai_w && e - GW::SAI < md.sai_base[md.I]) gl.g[md.off_sai + (e - GW::SAI)] = v;
            } else if (POST && e >= GW::COS) {
                (&gl.cosg[0][0])[e - GW::COS] = v;
            } else if (e >= GW::MAC) {
                const bool tau = e >= GW::MAT;
                const int r = e - (tau ? GW::MAT : GW::MAC), set = r / GW::QM, c = r - set * GW::QM;
                if (md.ma_active && set < (md.ma_global ? 1 : md.I) && c < md.ma_q)
                    gl.g[md.off_ma + 2 * md.ma_q * set + 2 * c + (tau ? 1 : 0)] = v;
            } else if (e >= GW::JIT) {
                if (md.has_jit && e - GW::JIT < md.I) gl.g[md.off_jit + (e - GW::JIT)] = v;
            } else if (e < md.I) {
                gl.g[md.off_off + e] = v;
            }
        }
        for (int e = lane; e < WN_N; e += 64) {
            double v = 0.0;
            for (int w = 0; w < WPT; ++w) v += s_gw.nat[w0 + w][e];
            if (e < WN_ACC) {
                if (e < md.K * 5) (&gl.nat[0][0])[e] = v;
            } else if (e - WN_ACC < md.acc) {
                gl.g[md.off_acc + (e - WN_ACC)] = v;
            }
        }
    }
    __syncthreads();
    if (live && wsub == 0) {
        // Map natural gradients to the parameterisation (one lane per planet).
        if (lane < md.K) {
            const int p = lane;
            const PlanetC& pc = sl.planet[p];
            const double* th = sl.theta + md.off_kep + 5 * p;
            double* gp = gl.g + md.off_kep + 5 * p;
            double nat[5];
            for (int q = 0; q < 5; ++q) nat[q] = gl.nat[p][q];
            if (BASIS) {
                double wsum = 0.0;                   // sum of w over all epochs
                for (int k = 0; k < md.I; ++k) wsum += gl.g[md.off_off + k];
                nat_basis(pc, wsum, nat);
            }
            const double gP = nat[0] * (-pc.freq * pc.freq * INV_TWO_PI);     // dfreq/dP = -freq^2 / (2 pi)
            const double gph = nat[1];
            const double ge = nat[2], gw = nat[3], gA = nat[4];
            const int prm = md.param;
            const bool lnP = (prm == 2 || prm == 6 || prm == 7);
            const bool sc = (prm == 1 || prm == 2 || prm == 4 || prm == 7);
            gp[0] = lnP ? -nat[0] * pc.freq : gP;
            if (prm == 2) {
                const double As = th[1], Ac = th[2], A = pc.K;
                gp[1] = gA * 2.0 * As + gph * (Ac / A);
                gp[2] = gA * 2.0 * Ac - gph * (As / A);
            } else {
                gp[1] = gA;
                gp[2] = pc.tp_mode ? -pc.freq * gph : gph;
            }
            if (sc) {
                const double S = th[3], C = th[4], e = pc.e;
                const double thr = (prm == 2 || prm == 4) ? 1e-5 : 1e-6;
                const bool free_w = md.use_c || e >= thr;
                gp[3] = ge * 2.0 * S + (free_w ? gw * (C / e) : 0.0);
                gp[4] = ge * 2.0 * C - (free_w ? gw * (S / e) : 0.0);
            } else {
                gp[3] = ge;
                gp[4] = gw;
            }
        }
        if (POST && lane == 63) {
            for (int c = 0; c < md.n_cos; ++c) {
                const int m = md.off_sin >= 0 ? c - 1 : c;    // -1: the sinusoid
                const int o = m < 0 ? md.off_sin : md.off_mag;
                const double gP = gl.cosg[c][2] * -(sl.cosw[c][1] / sl.theta[o]);
                if (m < 0) {
                    gl.g[o] = gP;
                    gl.g[o + 1] = gl.cosg[c][0];
                    gl.g[o + 2] = gl.cosg[c][1];
                } else {
                    gl.g[o] += gP;
                    gl.g[o + 1 + m] = gl.cosg[c][0];
                    gl.g[o + 3 + m] = gl.cosg[c][1];
                }
            }
        }
    }
    __syncthreads();
    if (live && wsub == 0) {
        double v = lnl_v;
        bool bad = !(v == v) || v == __builtin_inf();
        for (int d = lane; d < md.D; d += 64) {
            double gv = gl.g[md.free_idx[d]];
            if (bad) gv = 0.0;
            out_grad[b * md.D + d] = gv;
        }
        if (lane == 0) {
            if (bad) { v = -__builtin_inf(); atomicAdd(nonfinite, 1ull); }
            out_lnl[b] = v;
            if (stale) stale[b] = 0;
        }
    }
}

// slot_prepare for workgroups of several vectors, whose waves all wait.
template <int WPT, class SL>
__device__ __forceinline__ void slot_prepare_wg(const ModelDev& md, SL& sl, bool live, int wsub, int lane) {
    slot_prepare<WPT>(md, sl, live, wsub, lane);
    __syncthreads();
}

// Adjoint kernel.  Per tile (forward without the MA, in reverse with it):
// stage 1 finds w = dlnL/dmu of each lane's epochs (CPT chunks of 64 WPT
// epochs, held in registers), stage 2 then takes the planets one at a time,
// adding w times each planet's derivatives over the lane's epochs and
// reducing the five sums over the wave once per planet per tile, and the
// acceleration terms likewise.  No derivative is held across planets, which
// keeps the register count near the likelihood kernel's.  With the MA a
// forward pass first computes lnL and stores eps (one scratch row per
// vector).  `stale` (optional, per vector): vectors whose flag is 0 are
// skipped; a computed vector's flag is cleared.
// EXT: 0 plain models, 1 with terms added after the MA, 2 also MA orders
// above 1.
template <int PREC, int WPT, int EXT>
__global__ __launch_bounds__(BLOCK) void k_lnl_grad(ModelDev md, const double* __restrict__ theta, int64_t B,
                                                    int64_t ld, double* __restrict__ out_lnl,
                                                    double* __restrict__ out_grad,
                                                    unsigned long long* nonfinite, double* eps_scratch, int* stale) {
    constexpr int SLOTS = NWAVES / WPT;
    constexpr int G = 64 * WPT;
    constexpr int CPT = TILE / G;             // chunks of a tile per wave
    constexpr bool POST = EXT >= 1;
    using GW = GradWave<EXT>;
    __shared__ SlotLDS<SLOTS> s_slot[SLOTS];
    __shared__ GradLDS s_grad[SLOTS];
    __shared__ GradWaveLDS<EXT> s_gw;
    __shared__ TileLDS s_tile;
    __shared__ ScanLDS s_scan;
    const int wave = wave_uniform(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int slot = wave / WPT, wsub = wave % WPT;
    const int g = wsub * 64 + lane;
    const int64_t b = (int64_t)blockIdx.x * SLOTS + slot;
    const bool live = b < B && (!stale || stale[b] != 0);
    if (!__syncthreads_or(live)) return;       // no vector of this workgroup to compute
    SlotLDS<SLOTS>& sl = s_slot[slot];
    GradLDS& gl = s_grad[slot];
    if (live) expand_theta(md, sl, theta + b * ld, g, G);
    for (int j = g; j < MAXD; j += G) gl.g[j] = 0.0;
    for (int j = g; j < KMAX * 5; j += G) (&gl.nat[0][0])[j] = 0.0;
    // From the thread's index, not the uniform wave number: with an address that is
    // the same in every lane the compiler turns each atomic sum into a loop over
    // the wave's lanes (a magnetic cycle's gradients with MA(2), 6 planets x 878
    // epochs, one vector 66 -> 102 us).
    double* wacc = s_gw.acc[threadIdx.x >> 6];
    double* wnat = s_gw.nat[wave];
    for (int j = lane; j < GW::N; j += 64) wacc[j] = 0.0;
    for (int j = lane; j < WN_N; j += 64) wnat[j] = 0.0;
    tab_load(md, s_tile.tab);
    __syncthreads();
    slot_prepare_wg<WPT>(md, sl, live, wsub, lane);
    const int kmask = kt_path<PREC>(wave_uniform(sl.ktab_mask));
    const bool tp = model_tp(md);

    const bool ma = md.ma_active;
    double* eps = ma ? eps_scratch + (live ? b : 0) * (int64_t)md.N : nullptr;
    double lnl_v = 0.0;
    if (ma) {
        // Pass 1: the likelihood, storing eps.
        lnl_v = vec_lnl<PREC, WPT, false, true, EXT>(md, sl, s_tile.tab, s_scan, live, wsub, nullptr, nullptr, eps);
        __syncthreads();   // eps rows written by every wave of the slot
    }
    double chi = 0.0, prod = 1.0;
    int pexp = 0;
    double lam_carry = 0.0;
    double lq_carry[4] = {0.0, 0.0, 0.0, 0.0};     // MA(q >= 2) adjoint state
    int parity = 0;
    InsAcc ia;
    const int ntile = (md.N + TILE - 1) / TILE;
    for (int i = 0; i < ntile; ++i) {
        const int it = ma ? ntile - 1 - i : i;
        const int tb = it * TILE, tn = min(TILE, md.N - tb);
        __syncthreads();
        tile_load(md, s_tile, tb, tn);
        __syncthreads();
        double wv[CPT];
        if (!ma) {
#pragma unroll
            for (int c = 0; c < CPT; ++c) {
                const int j = c * G + g;
                wv[c] = (live && j < tn) ? plain_w<PREC, EXT>(md, sl, s_tile, wacc, ia, j, tb, chi, prod, pexp, kmask)
                                         : 0.0;
            }
        } else {
#pragma unroll
            for (int c = CPT - 1; c >= 0; --c) {
                wv[c] = 0.0;
                if (c * G >= tn) continue;            // uniform over the workgroup
                const int j = c * G + g;
                wv[c] = ma_chunk_w<PREC, WPT, EXT>(md, sl, s_tile, s_scan, eps, wacc, ia, live && j < tn, j, tb, tn,
                                                   lane, wave, wsub, parity, lam_carry, lq_carry);
            }
        }
        if (live) {
            for (int p = 0; p < md.K; ++p) {
                double a[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
                const PlanetC& pc = sl.planet[p];
#pragma unroll
                for (int c = 0; c < CPT; ++c) {
                    const int j = c * G + g;
                    if (j < tn) planet_wgrad<PREC>(pc, s_tile.tab, sl.ktab[p], s_tile.t[j], wv[c], a, tp, kt_mode(kmask, p));
                }
                wave_reduce_add5(a, wnat + 5 * p, lane, red5_index(lane));
            }
            if (md.acc) {
                double a[AMAX] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int c = 0; c < CPT; ++c) {
                    const int j = c * G + g;
                    if (j < tn) {
                        const double x = s_tile.t[j] - md.t0;
                        double xp = wv[c] * x;
#pragma unroll
                        for (int q = AMAX - 1; q >= 0; --q) {
                            if (q < md.acc) {
                                a[q] += xp;
                                xp *= x;
                            }
                        }
                    }
                }
                wave_reduce_add4(a, md.acc, wnat + WN_ACC, red4_index(lane));
            }
        }
    }
    ia.flush<EXT>(wacc);
    if (!ma) {
        double ldet = live ? log(prod) + (double)pexp * LN2 : 0.0;
        chi = wave_sum(chi);
        ldet = wave_sum(ldet);
        if (lane == 0) { s_scan.red[wave][0] = chi; s_scan.red[wave][1] = ldet; }
        __syncthreads();
        double c2 = 0.0, l2 = 0.0;
        const int w0 = wave - wsub;
        for (int w = 0; w < WPT; ++w) { c2 += s_scan.red[w0 + w][0]; l2 += s_scan.red[w0 + w][1]; }
        lnl_v = -0.5 * (c2 + l2) + md.lnl_const;
    }
    grad_finish<EXT, WPT>(md, sl, gl, s_gw, live, wave, wsub, lane, lnl_v, b, out_lnl, out_grad, nonfinite, stale);
}

// ---------------------------------------------------------------------------
// Single-pass adjoint for models whose moving average has order 1 or is
// absent: NW waves per vector, one vector per workgroup, two consecutive epochs
// per lane per tile, loaded straight from global memory (the data of all
// vectors are the same few hundred KB, in L2).  Each planet's Kepler solve is
// done once per epoch; cos f, sin f and 1 / D stay in registers from the model
// to the derivatives, and every lane keeps its own five sums per planet over
// the whole series, reduced over the wave once per vector.
//
// The MA(1) adjoint is carried forward.  Within a tile the reverse
// recurrence lambda_i = u_i + a_{i+1} lambda_{i+1} composes (a suffix scan
// started from zero) into lambda_i = B_i + A_i Lambda, with Lambda the value
// at the next tile's first epoch, unknown while the tile is processed.  Every
// gradient sum is linear in lambda: sum_i lambda_i h_i = S_B + Lambda S_A,
// S_B = sum B_i h_i, S_A = sum A_i h_i.  With (A^n, B^n) the map of tile n as
// a whole (that of its first epoch), Lambda_{n-1} = B^n + A^n Lambda_n and
// Lambda = 0 after the last tile, so
//   sum_n (S_B^n + Lambda_n S_A^n) = sum_n (S_B^n + B^n R_n),
//   R_0 = 0, R_{n+1} = A^n R_n + S_A^n.
// Every such sum keeps a total and an R state and is complete after one pass
// over the epochs; no eps row is stored.  S_B needs no tile map, which is why
// it can stay in a lane's registers; S_A is reduced per tile, but only by the
// waves in which some A_i matters (the tile's last, unless the MA is nearly a
// random walk).  The waves take the tile's segments in turn (rotated by one
// every tile), so that this work falls on every SIMD alike.
//
// Bound by VALU issue (7 planets, MA(1): 126 instructions per planet-epoch mixed
// and 137 FP64, the epochs' share included, against the 205 and 263 of one epoch
// per lane with five sums per planet reduced in every tile; the VALU issues in
// about 70% of the cycles).  Measured before and after:
// 8192 vectors of 7 planets x 10^4 epochs, MA(1), mixed, 3.76 -> 2.36 ms; 16,384
// of 5 planets x 2000 epochs, FP64 (with its table start), 1.16 -> 0.53 ms, a
// good part of that from grouping the epochs by instrument (emp_model_host).
// ---------------------------------------------------------------------------

// The wave's sums in LDS of the terms that lanes add to as they go, in
// 2^cl copies (lane mod 2^cl): 64 lanes adding to one address take the LDS some
// 260 cycles, and the lanes of a wave often share an instrument.  `pairs` sums
// with an R state each (offsets; the MA sets' coefficients, then their
// timescales where these are free; acceleration), the totals first, then the R
// states (only with the MA), then the sums that have none: the jitters' and, in
// the order of GradWave, those of the terms after the MA.
// Measured with one copy and with this: 8192 vectors of 1500 epochs and
// 1 planet, 4 instruments, FP64, 177 -> 98 us, with MA(1) per instrument 239 -> 166;
// 3 planets x 3000 epochs with MA(1) per instrument, mixed, 509 -> 424, with a
// global one 485 -> 430; with a sinusoid, whose sums every epoch of every lane
// adds to, 1 planet x 1500 epochs 561 -> 135, 5 x 3000 1365 -> 593.
struct InsLayout {
    int sets, pairs, rows;      // MA sets; sums with an R state; all rows (of 2^cl doubles) of one wave
    int npost;                  // rows of the terms after the MA
    __host__ __device__ InsLayout(const ModelDev& md, bool has_post) {
        npost = !has_post ? 0 : 3 * CMAX + (md.sai_w ? SAIMAX : 0);
        sets = !md.ma_active ? 0 : md.ma_global ? 1 : md.I;
        pairs = md.I + (md.ma_wfixed ? 1 : 2) * sets + md.acc;
        rows = (md.ma_active ? 2 : 1) * pairs + md.I + npost;
    }
    __host__ __device__ int mac(const ModelDev& md) const { return md.I; }
    __host__ __device__ int mat(const ModelDev& md) const { return md.I + sets; }
    __host__ __device__ int acc(const ModelDev& md) const { return pairs - md.acc; }
    __host__ __device__ int post() const { return rows - npost; }
    __host__ __device__ int jit(const ModelDev& md) const { return post() - md.I; }
};

// Per-lane sums of the per-instrument terms (offset, jitter, MA(1)
// coefficient and timescale) of the lane's epochs, the offset and MA sums
// with their R states; added to the wave's sums in LDS (InsLayout) when the
// lane's instrument changes (the MA sums are keyed by instrument, or by 0 for
// a global MA).  hasR: the wave has R states that are not all zero.
struct InsAcc1 {
    int k = -1, km = -1;
    double off = 0.0, offR = 0.0, jit = 0.0, mac = 0.0, macR = 0.0, mat = 0.0, matR = 0.0;
    // copy: the lane's copy of the wave's first row
    __device__ __forceinline__ void flush_ins(const ModelDev& md, const InsLayout& il, double* copy, int cl, bool hasR) {
        if (k < 0) return;
        atomicAdd(&copy[k << cl], off);
        if (hasR) atomicAdd(&copy[(il.pairs + k) << cl], offR);
        atomicAdd(&copy[(il.jit(md) + k) << cl], jit);
        off = offR = jit = 0.0;
    }
    __device__ __forceinline__ void flush_ma(const ModelDev& md, const InsLayout& il, double* copy, int cl, bool hasR) {
        if (km < 0) return;
        atomicAdd(&copy[(il.mac(md) + km) << cl], mac);
        if (hasR) atomicAdd(&copy[(il.pairs + il.mac(md) + km) << cl], macR);
        if (!md.ma_wfixed) {
            atomicAdd(&copy[(il.mat(md) + km) << cl], mat);
            if (hasR) atomicAdd(&copy[(il.pairs + il.mat(md) + km) << cl], matR);
        }
        mac = macR = mat = matR = 0.0;
    }
    // The move to the next tile, whose map is (tA, tB).
    __device__ __forceinline__ void move(double tA, double tB) {
        off = __builtin_fma(tB, offR, off);
        mac = __builtin_fma(tB, macR, mac);
        mat = __builtin_fma(tB, matR, mat);
        offR *= tA;
        macR *= tA;
        matR *= tA;
    }
    __device__ __forceinline__ void to(const ModelDev& md, const InsLayout& il, int kk, int kkm, double* copy, int cl,
                                       bool ma, bool hasR) {
        if (kk != k) {
            flush_ins(md, il, copy, cl, hasR);
            k = kk;
        }
        if (ma && kkm != km) {
            flush_ma(md, il, copy, cl, hasR);
            km = kkm;
        }
    }
};

// The planets' constants are read from LDS where they are used: without this
// the compiler keeps those of all planets in registers over the tiles.
__device__ __forceinline__ void reload_lds() { asm volatile("" ::: "memory"); }

template <int NW>
struct Grad1LDS {
    double natR[NW][WN_ACC];             // R states of the planets' sums (per wave)
    double2 fwd[2][NW], suf[2][NW];      // per segment: its forward and suffix maps (double-buffered)
    double first[2][NW];                 // its first epoch's multiplier
};

// Single-pass adjoint (above).  EXT: 0 plain models, 1 with the terms added
// after the MA.  MA: the model may have a moving average.  NW waves per
// workgroup (one vector), tiles of 128 NW epochs.  KM: the instance holds up to
// KM planets' values and sums in registers (8 and 4 VGPRs per planet).  TP: the
// model's planets are parameterised by the time of periastron (model_tp), a
// template parameter so that no planet-epoch branches on it.  `stale` as in k_lnl_grad.
// Waves per SIMD that an instance is compiled for: as many as its registers
// allow with little spilling (KM 4 / 6 / 8: 107 / 128 / 156 VGPRs without the
// moving average; with it 128, 168 and 168, the first and the last with 22 and
// 47 spilled, which still beats two waves per SIMD at KM 8, 2.49 against 2.82 ms).
constexpr int GRAD1_FEW = 4;
constexpr int grad1_occ(bool ma, int km) { return km <= 4 || (km <= 6 && !ma) ? 4 : 3; }
template <int PREC, int EXT, bool MA, int NW, int KM, bool TP>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(grad1_occ(MA, KM)))) void k_lnl_grad1(
    ModelDev md, const double* __restrict__ theta, int64_t B, int64_t ld, double* __restrict__ out_lnl,
    double* __restrict__ out_grad, unsigned long long* nonfinite, int* stale, int cl) {
    constexpr int NT = 64 * NW, NE = 2, TILE1 = NT * NE;
    constexpr bool POST = EXT >= 1, tp = TP;
    using GW = GradWave<EXT>;
    __shared__ SlotLDSt<float4, KM> sl;
    __shared__ GradLDS gl;
    __shared__ GradWaveLDS<EXT, NW> s_gw;
    __shared__ Grad1LDS<NW> s_g1;
    extern __shared__ double s_ins[];   // [NW][rows << cl]: the sums of InsLayout
    __shared__ SinCosTab s_tab;
    __shared__ ScanLDS s_scan;
    const int wave = wave_uniform(threadIdx.x >> 6), lane = threadIdx.x & 63, g = threadIdx.x;
    const int64_t b = blockIdx.x;
    if (b >= B || (stale && stale[b] == 0)) return;     // the whole workgroup: one vector
    expand_theta(md, sl, theta + b * ld, g, NT);
    for (int j = g; j < MAXD; j += NT) gl.g[j] = 0.0;
    for (int j = g; j < KMAX * 5; j += NT) (&gl.nat[0][0])[j] = 0.0;
    double* wacc = s_gw.acc[wave];
    double* wnat = s_gw.nat[wave];
    double* wnatR = s_g1.natR[wave];
    const InsLayout il(md, POST && has_post(md));
    double* wins = s_ins + wave * (il.rows << cl);
    double* copy = wins + (lane & ((1 << cl) - 1));
    for (int j = lane; j < GW::N; j += 64) wacc[j] = 0.0;
    for (int j = lane; j < WN_N; j += 64) wnat[j] = 0.0;
    for (int j = lane; j < WN_ACC; j += 64) wnatR[j] = 0.0;
    for (int j = lane; j < il.rows << cl; j += 64) wins[j] = 0.0;
    for (int j = g; j <= SC_N; j += NT) s_tab.v[j] = md.sctab[j];
    __syncthreads();
    if (wave == 0) slot_setup(md, sl, lane);
    __syncthreads();
    for (int p = wave; p < md.K; p += NW)       // the per-vector Kepler tables, one planet per wave
        if (sl.planet[p].ktab) ktab_fill(sl.planet[p], lane, sl.ktab[p][lane]);
    __syncthreads();
    const int kmask = kt_path<PREC>(wave_uniform(sl.ktab_mask));
    const int ri5 = red5_index(lane), ri4 = red4_index(lane);    // the sums a lane holds after a reduction

    const bool ma = MA && md.ma_active;
    double mu0 = 0.0;                   // the planets' constant parts, sum of K e cos w
    for (int p = 0; p < md.K; ++p) mu0 = __builtin_fma(sl.planet[p].K * sl.planet[p].e, sl.planet[p].cw, mu0);
    // The sums of each planet (nat_basis): the first four exchanged between
    // lanes 32 and 16 apart, so that each quarter of the wave holds one of
    // them (acc4), the fifth per lane (acc1).
    double acc4[KM], acc1[KM];
#pragma unroll
    for (int p = 0; p < KM; ++p) acc4[p] = acc1[p] = 0.0;
    double chi = 0.0, prod = 1.0;
    int pexp = 0;
    double carry = 0.0;                 // eps of the last epoch so far
    int parity = 0, rot = wave;         // rot: the tile's segment this wave takes
    bool hasR = false;                  // the wave's R states are not all zero
    InsAcc1 ia;
    double tnx[NE];                     // the next tile's times, loaded a tile ahead
#pragma unroll
    for (int i = 0; i < NE; ++i) {
        const int n = NE * g + i;
        tnx[i] = n < md.N ? md.t[n] : 0.0;
    }
    for (int tb = 0; tb < md.N; tb += TILE1) {
        const int n0 = tb + NE * (rot * 64 + lane);
        const int seg = rot;
        rot = rot + 1 == NW ? 0 : rot + 1;
        // Every lane solves the planets, a lane past the series' end at t = 0:
        // its values are finite and its weights (wB, wA) exactly zero.
        double t[NE], y[NE], err2[NE], dtc[NE], mu[NE];
        int k[NE];
        bool valid[NE];
#pragma unroll
        for (int i = 0; i < NE; ++i) {
            const int n = n0 + i, nn = tb + TILE1 + NE * (rot * 64 + lane) + i;
            valid[i] = n < md.N;
            t[i] = tnx[i];
            tnx[i] = nn < md.N ? md.t[nn] : 0.0;
            mu[i] = mu0;
        }
        auto load_rest = [&]() {
#pragma unroll
            for (int i = 0; i < NE; ++i) {
                const int n = n0 + i;
                k[i] = 0;
                y[i] = 0.0;
                err2[i] = 1.0;
                dtc[i] = 0.0;
                if (valid[i]) {
                    k[i] = md.ins[n];
                    y[i] = md.y[n];
                    err2[i] = md.s2[n];
                    if (ma) dtc[i] = md.dt[n];
                }
            }
        };
        reload_lds();
        // Stage 1: every planet's C = cos f and S = sin f / b, and the model.
        double C[KM][NE], S[KM][NE];
#pragma unroll
        for (int p = 0; p < KM; ++p) {
            if (p < md.K) {
                const PlanetC& pc = sl.planet[p];
                double sE[NE], cE[NE], rD[NE];
                planet_sc<PREC, NE>(pc, s_tab, sl.ktab[p], t, sE, cE, rD, tp, kt_mode(kmask, p));
                const double e = pc.e, kc = pc.K * pc.cw, ks = pc.c2;
#pragma unroll
                for (int i = 0; i < NE; ++i) {
                    C[p][i] = (cE[i] - e) * rD[i];
                    S[p][i] = sE[i] * rD[i];
                    mu[i] = __builtin_fma(kc, C[p][i], __builtin_fma(ks, S[p][i], mu[i]));
                }
            }
        }
        if (md.acc) {
#pragma unroll
            for (int i = 0; i < NE; ++i) {
                const double x = t[i] - md.t0;
                double v = 0.0;
                for (int a = 0; a < md.acc; ++a) v = __builtin_fma(v, x, sl.acc[a]);
                mu[i] += v * x;
            }
        }
        load_rest();
        double eps[NE], em[NE], am[NE];     // eps of the epoch and of the one before; its multiplier
#pragma unroll
        for (int i = 0; i < NE; ++i) {
            eps[i] = em[i] = 0.0;
            am[i] = 1.0;
            if (valid[i]) {
                err2[i] += sl.jit2[k[i]];
                eps[i] = y[i] - (mu[i] + sl.gam[k[i]]);
            }
        }
        // The MA filter, forward: the lane's two maps composed, a scan over
        // the wave, the segments' maps composed through LDS.
        double mnext_seg = 0.0;             // multiplier of the next segment's first epoch
        if (ma) {
#pragma unroll
            for (int i = 0; i < NE; ++i)
                if (valid[i]) am[i] = ma_mult(md, sl, k[i], dtc[i]);
            const double b0 = eps[0];
            double a = am[1] * am[0], bb = __builtin_fma(am[1], b0, eps[1]);
            wave_affine_scan(a, bb, lane);
            if (lane == 63) s_g1.fwd[parity][seg] = make_double2(a, bb);
            if (lane == 0) s_g1.first[parity][seg] = am[0];
            __syncthreads();
            double e0 = carry;              // eps before this segment
            double pa = 1.0, pb = 0.0;      // the maps of segments 0 .. w composed
            double2 tot[NW];
#pragma unroll
            for (int w = 0; w < NW; ++w) tot[w] = s_g1.fwd[parity][w];
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                if (w == seg) e0 = __builtin_fma(pa, carry, pb);
                pb = w ? __builtin_fma(tot[w].x, pb, tot[w].y) : tot[w].y;
                pa = w ? tot[w].x * pa : tot[w].x;
            }
            carry = __builtin_fma(pa, carry, pb);
            if (seg + 1 < NW) mnext_seg = s_g1.first[parity][seg + 1];
            const double e1 = __builtin_fma(a, e0, bb);       // the lane's last epoch
            em[0] = wave_prev(e1, e0);
            em[1] = __builtin_fma(am[0], em[0], b0);
            eps[0] = em[1];
            eps[1] = e1;
        }
        // The likelihood's terms.
        double ef[NE], ie[NE];
#pragma unroll
        for (int i = 0; i < NE; ++i) {
            ef[i] = ie[i] = 0.0;
            if (valid[i]) {
                const double cs = (POST && has_post(md)) ? epoch_post(md, sl, s_tab, t[i], n0 + i, k[i]) : 0.0;
                ef[i] = eps[i] - cs;
                ie[i] = rcp_path<PREC>(err2[i]);
                chi = __builtin_fma(ef[i] * ef[i], ie[i], chi);
                prod *= err2[i];
                pexp += __builtin_amdgcn_frexp_exp(prod);
                prod = __builtin_amdgcn_frexp_mant(prod);
                if (POST && has_post(md))
                    post_accumulate<EXT>(md, sl, s_tab, t[i], n0 + i, k[i], ef[i] * ie[i],
                                         copy + (il.post() << cl), cl);
            }
        }
        // dlnL/dmu = wB + wA Lambda; lambda = lB + lA Lambda; (tA, tB) the tile's map.
        double wB[NE], wA[NE], tA = 0.0, tB = 0.0;
        bool needA = false;
        if (!ma) {
#pragma unroll
            for (int i = 0; i < NE; ++i) {
                wB[i] = ef[i] * ie[i];
                wA[i] = 0.0;
            }
        } else {
            // the multiplier of the epoch after the lane's last one
            double m1 = wave_next(am[0], mnext_seg);
            if (seg == NW - 1 && lane == 63 && n0 + NE < md.N) m1 = ma_mult(md, sl, md.ins[n0 + NE], md.dt[n0 + NE]);
            if (n0 + NE >= md.N) m1 = 0.0;
            const double m0 = n0 + 1 < md.N ? am[1] : 0.0;
            const double u0 = -ef[0] * ie[0], u1 = -ef[1] * ie[1];
            double sa = m0 * m1, sb = __builtin_fma(m0, u1, u0);
            wave_affine_suffix_scan(sa, sb, lane);
            if (lane == 0) s_g1.suf[parity][seg] = make_double2(sa, sb);
            __syncthreads();
            // (pa, pb): the maps of segments NW - 1 down to w composed
            double ia_ = 1.0, ib_ = 0.0;    // the map after this segment
            double pa = 1.0, pb = 0.0;
            double2 tot[NW];
#pragma unroll
            for (int w = 0; w < NW; ++w) tot[w] = s_g1.suf[parity][w];
#pragma unroll
            for (int w = NW - 1; w >= 0; --w) {
                if (w == seg) {
                    ia_ = pa;
                    ib_ = pb;
                }
                pb = __builtin_fma(tot[w].x, pb, tot[w].y);
                pa = tot[w].x * pa;
            }
            tA = pa;
            tB = pb;
            const double lB0 = __builtin_fma(sa, ib_, sb), lA0 = sa * ia_;
            const double lB1 = __builtin_fma(m1, wave_next(lB0, ib_), u1), lA1 = m1 * wave_next(lA0, ia_);
            wB[0] = valid[0] ? -lB0 : 0.0;
            wA[0] = valid[0] ? -lA0 : 0.0;
            wB[1] = valid[1] ? -lB1 : 0.0;
            wA[1] = valid[1] ? -lA1 : 0.0;
            // A wave whose every |A_i| is below 2^-100 adds nothing measurable
            // through Lambda (the terms are under 1e-17 of any gradient the
            // data can give): it reduces the B parts alone.  With |a| <= 1/3,
            // every wave of a tile but the last is such a wave.
            needA = __any(__builtin_fabs(wA[0]) > 0x1p-100 || __builtin_fabs(wA[1]) > 0x1p-100);
            // The sums this wave already holds in LDS, and the lane's own, move
            // to the next tile; a tile whose map's |A| is below 2^-100 (most
            // are) leaves no R state, by the same measure.
            if (hasR) {
                hasR = __any(__builtin_fabs(tA) > 0x1p-100);
                const double rA = hasR ? tA : 0.0;
                for (int e = lane; e < il.pairs << cl; e += 64) {
                    const double R0 = wins[(il.pairs << cl) + e];
                    wins[e] = __builtin_fma(tB, R0, wins[e]);
                    wins[(il.pairs << cl) + e] = rA * R0;
                }
                for (int e = lane; e < md.K * 5; e += 64) {
                    const double R0 = wnatR[e];
                    wnat[e] = __builtin_fma(tB, R0, wnat[e]);
                    wnatR[e] = rA * R0;
                }
                ia.move(rA, tB);
            }
            hasR = hasR || needA;
        }
        // The per-instrument sums of the lane's epochs.
#pragma unroll
        for (int i = 0; i < NE; ++i) {
            if (!valid[i]) continue;
            ia.to(md, il, k[i], md.ma_global ? 0 : k[i], copy, cl, ma, hasR);
            ia.off += wB[i];
            if (needA) ia.offR += wA[i];
            if (md.has_jit) ia.jit = __builtin_fma(sl.jit[k[i]], ef[i] * ef[i] * ie[i] * ie[i] - ie[i], ia.jit);
            if (ma) {
                // d a / d (c, tau) times the previous eps (none at a segment start)
                const bool start = md.ma_wfixed ? dtc[i] == 0.0 : dtc[i] < 0.0;
                if (!start) {
                    const double wgt = md.ma_wfixed ? dtc[i] : exp(-dtc[i] / sl.ma_tau[k[i]]);
                    const double hc = em[i] * wgt;                      // lambda = -w
                    ia.mac = __builtin_fma(wB[i], hc, ia.mac);
                    if (needA) ia.macR = __builtin_fma(wA[i], hc, ia.macR);
                    if (!md.ma_wfixed) {
                        const double tau = sl.ma_tau[k[i]];
                        const double ht = hc * (sl.ma_c[k[i]] * dtc[i] / (tau * tau));
                        ia.mat = __builtin_fma(wB[i], ht, ia.mat);
                        if (needA) ia.matR = __builtin_fma(wA[i], ht, ia.matR);
                    }
                }
            }
        }
        // Stage 2: the planets' sums, from the stage-1 values.
        reload_lds();
#pragma unroll
        for (int p = 0; p < KM; ++p) {
            if (p < md.K) {
                const PlanetC& pc = sl.planet[p];
                const double e = pc.e, sw = pc.sw, bc = pc.bq * pc.cw;
                double s[NE], q[NE];
#pragma unroll
                for (int i = 0; i < NE; ++i) {
                    s[i] = __builtin_fma(C[p][i], sw, S[p][i] * bc);            // sin(f + w)
                    q[i] = __builtin_fma(e, C[p][i], 1.0);                      // b^2 / D
                }
                auto sums = [&](const double (&w)[NE], double (&v)[5]) {
#pragma unroll
                    for (int i = 0; i < NE; ++i) {
                        const double x = w[i] * s[i], xm = x * q[i] * q[i], xs = x * S[p][i];
                        const double tau = tp ? t[i] - pc.tp : t[i];
                        v[0] = i ? __builtin_fma(xm, tau, v[0]) : xm * tau;
                        v[1] = i ? v[1] + xm : xm;
                        v[2] = i ? __builtin_fma(xs, q[i], v[2] + xs) : __builtin_fma(xs, q[i], xs);
                        v[3] = i ? __builtin_fma(w[i], C[p][i], v[3]) : w[i] * C[p][i];
                        v[4] = i ? __builtin_fma(w[i], S[p][i], v[4]) : w[i] * S[p][i];
                    }
                };
                double v[5];
                sums(wB, v);
                acc4[p] += swap_add16(swap_add32(v[0], v[1]), swap_add32(v[2], v[3]));
                acc1[p] += v[4];
                if (needA) {        // the A parts, only where some lane's A is not negligible
                    double a5[5];
                    sums(wA, a5);
                    wave_reduce_add5(a5, wnatR + 5 * p, lane, ri5);
                }
            }
        }
        if (md.acc) {
            double b4[AMAX] = {0.0, 0.0, 0.0, 0.0}, a4[AMAX] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int i = 0; i < NE; ++i) {
                const double x = t[i] - md.t0;
                double xp = x;
#pragma unroll
                for (int q = AMAX - 1; q >= 0; --q) {
                    if (q < md.acc) {
                        b4[q] = __builtin_fma(wB[i], xp, b4[q]);
                        a4[q] = __builtin_fma(wA[i], xp, a4[q]);
                        xp *= x;
                    }
                }
            }
#pragma unroll
            for (int q = 0; q < AMAX; ++q)
                if (q < md.acc) {
                    atomicAdd(&copy[(il.acc(md) + q) << cl], b4[q]);
                    if (needA) atomicAdd(&copy[(il.pairs + il.acc(md) + q) << cl], a4[q]);
                }
        }
        parity ^= 1;
    }
#pragma unroll
    for (int p = 0; p < KM; ++p)
        if (p < md.K) {
            double c = acc4[p];         // the rows of 16 lanes hold the sums 0, 2, 1, 3 (wave_reduce4)
            c += dpp_mov_f64<0x128>(c);
            c += dpp_mov_f64<0x141>(c);
            c += dpp_mov_f64<0xB1>(c);
            c += dpp_mov_f64<0x4E>(c);
            if (ri4 >= 0) wnat[5 * p + ri4] += c;
            const double v4 = wave_sum(acc1[p]);
            if (lane == 0) wnat[5 * p + 4] += v4;
        }
    // The copies of the wave's sums (R states have nothing left to meet).
    ia.flush_ins(md, il, copy, cl, false);
    ia.flush_ma(md, il, copy, cl, false);
    wave_sync();
    const int nsum = il.pairs + md.I + il.npost;
    for (int r = lane; r < nsum; r += 64) {
        const double* c = wins + ((r < il.pairs ? r : il.jit(md) + r - il.pairs) << cl);
        double v = 0.0;
        for (int q = 0; q < 1 << cl; ++q) v += c[q];
        if (POST && r >= il.pairs + md.I) wacc[GW::COS + r - il.pairs - md.I] = v;
        else if (r >= il.pairs) wacc[GW::JIT + r - il.pairs] = v;
        else if (r >= il.acc(md)) wnat[WN_ACC + r - il.acc(md)] = v;
        else if (r >= md.I + il.sets) wacc[GW::MAT + (r - il.mat(md)) * GW::QM] = v;
        else if (r >= md.I) wacc[GW::MAC + (r - md.I) * GW::QM] = v;
        else wacc[GW::OFF + r] = v;
    }
    double ldet = log(prod) + (double)pexp * LN2;
    chi = wave_sum(chi);
    ldet = wave_sum(ldet);
    if (lane == 0) { s_scan.red[wave][0] = chi; s_scan.red[wave][1] = ldet; }
    __syncthreads();
    double c2 = 0.0, l2 = 0.0;
    for (int w = 0; w < NW; ++w) { c2 += s_scan.red[w][0]; l2 += s_scan.red[w][1]; }
    const double lnl_v = -0.5 * (c2 + l2) + md.lnl_const;
    grad_finish<EXT, NW, true>(md, sl, gl, s_gw, true, wave, wave, lane, lnl_v, b, out_lnl, out_grad, nonfinite, stale);
}

// Each model runs the instance with only the features it uses: the terms
// added after the MA cost scalar registers, MA orders above 1 vector
// registers.
template <int PREC, int WPT>
static void launch_grad_t(const ModelDev& md, const double* th, int64_t B, int64_t ld, double* lnl, double* grad,
                          unsigned long long* nf, double* scratch, int* stale, hipStream_t s) {
    constexpr int SLOTS = NWAVES / WPT;
    const int64_t grid = (B + SLOTS - 1) / SLOTS;
    if (md.ma_active && md.ma_q > 1)
        hipLaunchKernelGGL((k_lnl_grad<PREC, WPT, 2>), dim3((unsigned)grid), dim3(BLOCK), 0, s, md, th, B, ld,
                           lnl, grad, nf, scratch, stale);
    else if (has_post(md))
        hipLaunchKernelGGL((k_lnl_grad<PREC, WPT, 1>), dim3((unsigned)grid), dim3(BLOCK), 0, s, md, th, B, ld,
                           lnl, grad, nf, scratch, stale);
    else
        hipLaunchKernelGGL((k_lnl_grad<PREC, WPT, 0>), dim3((unsigned)grid), dim3(BLOCK), 0, s, md, th, B, ld,
                           lnl, grad, nf, scratch, stale);
}

// The single-pass kernel runs every model whose MA order is at most 1, unless
// emp_model_set_grad_kernel asks for the two-pass one.  Two waves per vector:
// measured against 4 (whose waves wait for one another at the scans' barriers)
// and 1 (whose tiles of 128 epochs repeat the A parts' reductions most often):
// 8192 vectors of 7 planets x 10^4 epochs with MA(1), mixed, 2.49 ms against
// 2.61 and 2.79; 16,384 of 5 planets x 2000 epochs, FP64, 0.72 against 0.83 and
// 0.86.  Short series take it too: 8192 vectors of 2 planets, FP64, 64 / 73 /
// 108 / 150 us at 150 / 256 / 512 / 1000 epochs against the two-pass kernel's
// 84 / 86 / 168 / 238 (7 planets with MA(1), mixed: 135 / 139 / 223 / 361
// against 172 / 166 / 320 / 536).
constexpr int GRAD1_NW = 2;
// Four with the moving average, for series of more than one tile, while the batch
// has at most three vectors per compute unit: the launch is then one vector's chain
// of tiles long, and four waves halve the tiles.  FP64 at 2 / 4 waves per vector: 7
// planets x 1747 epochs with a global MA(1), 200 / 768 / 1024 vectors 76 / 51, 92 /
// 74 and 96 / 102 us; 2 x 10^4 with MA(1) per instrument 197 / 113, 236 / 159 and
// 243 / 189 us; 6 x 300, 26 / 18, 29 / 24 and 31 / 33 us; 7 x 256, one tile of two
// waves, 19 / 19 and 24 / 27 us (200, 768).
// One for series of at most one wave's tile, which leave a second wave without
// epochs.  FP64 at 2 waves / 1 / the two-pass kernel, 2000 and 65,536 vectors: 7 x 29
// with MA(1) 52 / 28 / 27 and 967 / 597 / 701 us, 3 x 63 without 21 / 17 / 19 and 453 /
// 299 / 446, 1 x 128 15 / 14 / 18 and 283 / 211 / 427.
constexpr int GRAD1_NW_FEW = 4, GRAD1_NW_SHORT = 1;
static int grad1_waves(const EmpModel* m, int64_t B) {
    if (m->dev.N <= 128 * GRAD1_NW_SHORT) return GRAD1_NW_SHORT;
    return m->dev.ma_active && m->dev.N > 128 * GRAD1_NW && B <= 3 * (int64_t)m->n_cu ? GRAD1_NW_FEW : GRAD1_NW;
}
// LDS for the copies of the waves' sums (InsLayout) that keeps the KM = 8
// instances' 6 workgroups per CU (160 KB, 20 KB of each without the copies).
constexpr size_t GRAD1_INS_BYTES = 5632;
// Below this many epochs the default kernel is one that a caller may still
// replace by the two-pass one after scratch was set aside for it: a batch whose
// eps rows would not fit the allocation-free entry point's scratch is refused
// there, and the gradient move holds the rows (emp_grad_scratch_reserve).
constexpr int TWO_PASS_RESERVE_N = 1024;

static bool use_grad1(const EmpModel* m) {
    const ModelDev& md = m->dev;
    if (md.ma_active && md.ma_q > 1) return false;
    return m->grad_kernel != EMP_GRAD_KERNEL_TWO_PASS;
}

extern "C" int emp_model_set_grad_kernel(EmpModel* m, int32_t which) {
    if (!m) { emp_set_error("null model"); return EMP_EINVAL; }
    if (which != EMP_GRAD_KERNEL_AUTO && which != EMP_GRAD_KERNEL_TWO_PASS && which != EMP_GRAD_KERNEL_SINGLE_PASS) {
        emp_set_error("adjoint kernel must be EMP_GRAD_KERNEL_AUTO, _TWO_PASS or _SINGLE_PASS");
        return EMP_EINVAL;
    }
    if (which == EMP_GRAD_KERNEL_SINGLE_PASS && m->dev.ma_active && m->dev.ma_q > 1) {
        emp_set_error("the single-pass adjoint handles MA orders up to 1 (this model: %d)", m->dev.ma_q);
        return EMP_EUNSUP;
    }
    m->grad_kernel = which;
    return EMP_OK;
}

// Doubles of scratch one launch over B vectors needs: with the moving
// average in the two-pass kernel, one row of eps per vector (B x N); none
// otherwise.
size_t emp_grad_scratch_doubles(const EmpModel* m, int64_t B) {
    return (m->dev.ma_active && !use_grad1(m)) ? (size_t)B * (size_t)m->dev.N : 0;
}

// Doubles to set aside where the scratch is fixed before the kernel is: what a
// launch needs now, and below TWO_PASS_RESERVE_N epochs also what it would need
// after a switch of the default to the two-pass kernel.
size_t emp_grad_scratch_reserve(const EmpModel* m, int64_t B) {
    if (m->grad_kernel == EMP_GRAD_KERNEL_AUTO && m->dev.ma_active && m->dev.N < TWO_PASS_RESERVE_N)
        return (size_t)B * (size_t)m->dev.N;
    return emp_grad_scratch_doubles(m, B);
}

// The MA adjoint's scratch, model-owned, grown (never shrunk) on demand.
static int ensure_grad_scratch(EmpModel* m, int64_t B) {
    const size_t need = emp_grad_scratch_doubles(m, B);
    if (!need) return EMP_OK;
    if (m->grad_scratch_cap >= need) return EMP_OK;
    if (m->d_grad_scratch) {
        EMP_HIP(hipDeviceSynchronize());
        (void)hipFree(m->d_grad_scratch);
        m->d_grad_scratch = nullptr;
        m->grad_scratch_cap = 0;
    }
    EMP_HIP(hipMalloc((void**)&m->d_grad_scratch, need * sizeof(double)));
    m->grad_scratch_cap = need;
    return EMP_OK;
}

// Waves per vector of the two-pass kernel for a batch of B.  Four by default:
// with one or two waves per vector a workgroup holds four or eight slots of
// LDS and the kernel's registers allow three or four waves per SIMD, with
// four both allow four to six (measured on 8192 vectors of 7 planets x 10^4
// epochs: mixed 5.1 ms at 4, 6.8 ms at 2, 6.1 ms at 8; FP64 within 4%).
// Fewer when a vector has fewer than two epochs per lane, more while the
// batch leaves SIMDs short of waves.
int emp_pick_grad_wpt(const EmpModel* m, int64_t B) {
    if (m->wpt_override) return m->wpt_override;
    const int64_t target_waves = (int64_t)m->n_cu * 4 * 6;
    int wpt = 4;
    while (wpt > 1 && 64 * wpt > m->dev.N / 2) wpt /= 2;
    while (wpt < 8 && B * wpt < target_waves && 64 * (wpt * 2) <= m->dev.N / 2) wpt *= 2;
    return wpt;
}

int emp_launch_grad_ws(const EmpModel* m, const double* th, int64_t B, int64_t ld, double* lnl, double* grad,
                       double* eps_scratch, hipStream_t s, int precision, int* stale, int wpt, int64_t shape) {
    if (B <= 0) return EMP_OK;
    if (shape <= 0) shape = B;
    unsigned long long* nf = m->d_nonfinite;
    // A grid holds fewer than 2^32 threads: larger batches in pieces (one vector
    // takes 128 threads of the single-pass kernel there, up to 512 of the other,
    // whose scratch rows a piece uses again after the one before it).
    const int64_t PIECE = (int64_t)1 << (use_grad1(m) ? 24 : 22);
    if (B > PIECE) {
        for (int64_t b = 0; b < B; b += PIECE) {
            const int rc = emp_launch_grad_ws(m, th + b * ld, std::min(PIECE, B - b), ld, lnl + b, grad + b * m->dev.D,
                                              eps_scratch, s, precision, stale ? stale + b : nullptr, wpt, shape);
            if (rc) return rc;
        }
        return EMP_OK;
    }
    if (use_grad1(m)) {
        const ModelDev& md = m->dev;
        if (precision != 0 && precision != 1) { emp_set_error("bad precision"); return EMP_EINVAL; }
        const int nw = grad1_waves(m, shape);
        // Eight copies of the wave's sums, fewer where many instruments would cost occupancy.
        const int rows = nw * InsLayout(md, has_post(md)).rows;
        int cl = 3;
        while (cl && (rows << cl) * sizeof(double) > GRAD1_INS_BYTES * nw / GRAD1_NW) --cl;
        const size_t lds = (size_t)(rows << cl) * sizeof(double);
#define EMP_CASE1(P, E, A, W, M, T) hipLaunchKernelGGL((k_lnl_grad1<P, E, A, W, M, T>), dim3((unsigned)B), dim3(64 * W), lds, s, md, th, B, ld, lnl, grad, nf, stale, cl)
#define EMP_CASE1M(P, E, A, W, T) { if (md.K <= GRAD1_FEW) EMP_CASE1(P, E, A, W, GRAD1_FEW, T); else if (W == GRAD1_NW && md.K <= 6) EMP_CASE1(P, E, A, GRAD1_NW, 6, T); else EMP_CASE1(P, E, A, W, KMAX, T); }
#define EMP_CASE1A(P, E, T) { \
    if (!md.ma_active) { if (nw == GRAD1_NW_SHORT) EMP_CASE1M(P, E, false, GRAD1_NW_SHORT, T) else EMP_CASE1M(P, E, false, GRAD1_NW, T) } \
    else if (nw == GRAD1_NW_SHORT) EMP_CASE1M(P, E, true, GRAD1_NW_SHORT, T) \
    else if (nw == GRAD1_NW_FEW) EMP_CASE1M(P, E, true, GRAD1_NW_FEW, T) \
    else EMP_CASE1M(P, E, true, GRAD1_NW, T) }
#define EMP_CASE1T(P, E) { if (model_tp(md)) EMP_CASE1A(P, E, true) else EMP_CASE1A(P, E, false) }
        if (precision == 0) { if (has_post(md)) EMP_CASE1T(0, 1) else EMP_CASE1T(0, 0) }
        else { if (has_post(md)) EMP_CASE1T(1, 1) else EMP_CASE1T(1, 0) }
#undef EMP_CASE1T
#undef EMP_CASE1A
#undef EMP_CASE1M
#undef EMP_CASE1
        EMP_HIP(hipGetLastError());
        return EMP_OK;
    }
    if (m->dev.ma_active && !eps_scratch) { emp_set_error("moving-average gradient needs a scratch buffer"); return EMP_EINVAL; }
    if (wpt <= 0) wpt = emp_pick_grad_wpt(m, shape);
#define EMP_CASE(P, W) if (precision == P && wpt == W) launch_grad_t<P, W>(m->dev, th, B, ld, lnl, grad, nf, eps_scratch, stale, s); else
    EMP_CASE(0, 1) EMP_CASE(0, 2) EMP_CASE(0, 4) EMP_CASE(0, 8)
    EMP_CASE(1, 1) EMP_CASE(1, 2) EMP_CASE(1, 4) EMP_CASE(1, 8) { emp_set_error("bad precision/wpt"); return EMP_EINVAL; }
#undef EMP_CASE
    EMP_HIP(hipGetLastError());
    return EMP_OK;
}

int emp_launch_grad(EmpModel* m, const double* th, int64_t B, int64_t ld, double* lnl, double* grad, hipStream_t s,
                    int precision) {
    int rc = ensure_grad_scratch(m, B);
    if (rc) return rc;
    return emp_launch_grad_ws(m, th, B, ld, lnl, grad, m->d_grad_scratch, s, precision);
}

extern "C" int emp_lnl_grad_batch(EmpModel* m, const double* theta, int64_t B, int64_t ld, double* lnl,
                                  double* grad, int32_t flags, void* stream) {
    if (!m) { emp_set_error("null model"); return EMP_EINVAL; }
    if (B < 0 || (B > 0 && (!theta || !lnl || !grad))) { emp_set_error("bad batch arguments"); return EMP_EINVAL; }
    if (ld < m->desc.ndim) { emp_set_error("ld < ndim"); return EMP_EINVAL; }
    if (emp_fault_injected()) return EMP_EFAULT_INJECTED;
    if (B == 0) return EMP_OK;
    hipStream_t s = (hipStream_t)stream;
    const int prec = (flags & EMP_GRAD_MIXED) ? EMP_MIXED : EMP_FP64;
    if (!(flags & EMP_HOST_POINTERS)) return emp_launch_grad(m, theta, B, ld, lnl, grad, s, prec);
    const size_t nin = (size_t)B * ld, D = (size_t)m->desc.ndim;
    double *din = nullptr, *dl = nullptr, *dg = nullptr;
    EMP_HIP(hipMalloc(&din, nin * 8));
    EMP_HIP(hipMalloc(&dl, (size_t)B * 8));
    EMP_HIP(hipMalloc(&dg, std::max<size_t>((size_t)B * D, 1) * 8));
    int rc = EMP_OK;
    if (hipMemcpyAsync(din, theta, nin * 8, hipMemcpyHostToDevice, s) != hipSuccess) rc = EMP_EHIP;
    if (!rc) rc = emp_launch_grad(m, din, B, ld, dl, dg, s, prec);
    if (!rc && hipMemcpyAsync(lnl, dl, (size_t)B * 8, hipMemcpyDeviceToHost, s) != hipSuccess) rc = EMP_EHIP;
    if (!rc && D && hipMemcpyAsync(grad, dg, (size_t)B * D * 8, hipMemcpyDeviceToHost, s) != hipSuccess) rc = EMP_EHIP;
    if (!rc && hipStreamSynchronize(s) != hipSuccess) rc = EMP_EHIP;
    if (rc == EMP_EHIP) emp_set_error("HIP error in emp_lnl_grad_batch host path");
    (void)hipFree(din);
    (void)hipFree(dl);
    (void)hipFree(dg);
    return rc;
}

// ---------------------------------------------------------------------------
// Allocation-free variant of emp_lnl_grad_batch (device pointers).  The
// moving-average scratch is `scratch`, a static device array that every
// device the library runs on holds until the process ends, instead of model
// memory grown with hipMalloc.  Host code never passes the array's name to a
// kernel: it stands for the host-side shadow, not the device address.  The
// device address comes from hipGetSymbolAddress, taken once per device with
// that device current, and is kept in scratch_dev[].
// ---------------------------------------------------------------------------
static __device__ __align__(256) double scratch[EMP_NOALLOC_SCRATCH_DOUBLES];

namespace {
constexpr int MAX_DEVICES = 64;
std::mutex scratch_mu;
double* scratch_dev[MAX_DEVICES] = {};
}  // namespace

// Device address of this device's copy of `scratch` (the current device).
static int scratch_address(int dev, double** out) {
    if (dev < 0 || dev >= MAX_DEVICES) { emp_set_error("device %d outside [0, %d)", dev, MAX_DEVICES); return EMP_EINVAL; }
    std::lock_guard<std::mutex> lock(scratch_mu);
    if (!scratch_dev[dev]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return emp_hip_fail(e, "hipGetSymbolAddress(scratch)", __FILE__, __LINE__);
        if (!p) { emp_set_error("hipGetSymbolAddress(scratch) returned a null address"); return EMP_EHIP; }
        scratch_dev[dev] = (double*)p;
    }
    *out = scratch_dev[dev];
    return EMP_OK;
}

extern "C" int emp_lnl_grad_batch_noalloc(EmpModel* m, const double* theta, int64_t B, int64_t ld, double* lnl,
                                          double* grad, int32_t flags, void* stream) {
    if (!m) { emp_set_error("null model"); return EMP_EINVAL; }
    if (B < 0 || (B > 0 && (!theta || !lnl || !grad))) { emp_set_error("bad batch arguments"); return EMP_EINVAL; }
    if (ld < m->desc.ndim) { emp_set_error("ld < ndim"); return EMP_EINVAL; }
    if (flags & EMP_HOST_POINTERS) {
        emp_set_error("the allocation-free entry point takes device pointers only (EMP_HOST_POINTERS stages through allocated memory)");
        return EMP_EINVAL;
    }
    if (flags & ~EMP_GRAD_MIXED) { emp_set_error("unknown flags 0x%x", (unsigned)flags); return EMP_EINVAL; }
    const size_t need = emp_grad_scratch_reserve(m, B);
    if (need > EMP_NOALLOC_SCRATCH_DOUBLES) {
        emp_set_error("batch of %lld vectors needs %zu doubles of scratch; the allocation-free entry point holds %zu",
                      (long long)B, need, (size_t)EMP_NOALLOC_SCRATCH_DOUBLES);
        return EMP_EINVAL;
    }
    if (emp_fault_injected()) return EMP_EFAULT_INJECTED;
    if (B == 0) return EMP_OK;
    int dev = -1;
    EMP_HIP(hipGetDevice(&dev));
    if (dev != m->device) { emp_set_error("model lives on device %d, device %d is current", m->device, dev); return EMP_EINVAL; }
    double* ws = nullptr;
    if (need) {
        const int rc = scratch_address(dev, &ws);
        if (rc) return rc;
    }
    const int prec = (flags & EMP_GRAD_MIXED) ? EMP_MIXED : EMP_FP64;
    return emp_launch_grad_ws(m, theta, B, ld, lnl, grad, ws, (hipStream_t)stream, prec);
}

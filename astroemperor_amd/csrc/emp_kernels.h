// Likelihood building blocks shared by the batched-lnL, model-eval, adjoint
// and PT kernels.
//
// Launch geometry: a parameter vector belongs to WPT waves.  With WPT > 1 the
// workgroup is those waves (in the two-pass adjoint several such vectors, which
// wait together); with one wave per vector the waves of a workgroup share the
// sin/cos table and nothing else.  The vector's waves walk the epochs
// in chunks, each lane with two consecutive epochs (one in a last chunk of at
// most 64 WPT), read straight from global memory: the data of every vector are
// the same few KB to hundreds of KB, in L1 and L2.
#pragma once
#include "emp_internal.h"

namespace emp {

constexpr double LN2 = 0.69314718055994530942;

// One prior term at x, by the reference's templates (support/priors/*.prior).
// The sums of terms run in the order of the generated my_prior
// (emp/emp.py:182-254), so that they are bit-identical to it: per block, add
// each free parameter's prior, return -inf as soon as a block leaves the sum at
// -inf, then add the block's derived eccentricity prior.
__device__ inline double prior_term(const EmpPriorTerm& p, double x) {
#pragma clang fp contract(off)
    if (!(x >= p.lo && x <= p.hi)) return -__builtin_inf();
    switch (p.kind) {
        case EMP_PRIOR_UNIFORM:
        case EMP_PRIOR_JEFFREYS:
            return p.a0;
        case EMP_PRIOR_NORMAL: {
            double z = (x - p.a0) / p.a1;
            return -0.5 * (z * z) - p.a3 - p.a2;
        }
        case EMP_PRIOR_BETA: {
            double v = -p.a2;
            if (p.a0 != 1.0) v += (p.a0 - 1.0) * log(x);
            if (p.a1 != 1.0) v += (p.a1 - 1.0) * log1p(-x);
            return v;
        }
        default:
            return 0.0;
    }
}

// Sum of a vector's prior terms by one whole wave, as if term by term: each
// block's free parameters, a return if the sum is -inf at the block's end, then
// the block's derived eccentricity prior.  The lanes evaluate the terms of that
// sequence in parallel, with their loads in flight together (term(entry, i): the
// value of sequence entry i), then the terms are added up in sequence order (a
// scalar read of each lane), with the -inf return where a ballot marks a block's
// end, so that every caller forms the same bits.
template <class F>
__device__ __forceinline__ double prior_wave(const ModelDev& md, int lane, F term) {
#pragma clang fp contract(off)
    double lp = 0.0;
    for (int i0 = 0; i0 < md.npseq; i0 += 64) {
        const int i = i0 + lane;
        double v = 0.0;
        int kind = 0;
        if (i < md.npseq) {
            const PseqEntry& pe = md.pseq_e[i];
            kind = pe.kind;
            if (kind != 2) v = term(pe, i);
        }
        const unsigned long long chk = __ballot(i < md.npseq && kind == 2);
        const int n = min(64, md.npseq - i0);
        for (int k = 0; k < n; ++k) {
            if ((chk >> k) & 1ull) {
                if (lp == -__builtin_inf()) return lp;
            } else {
                lp += readlane_f64(v, k);
            }
        }
    }
    return lp;
}

// Prior of a full parameter vector (fixed values in place).
__device__ inline double prior_vector_wave(const ModelDev& md, const double* th, int lane) {
    return prior_wave(md, lane, [&](const PseqEntry& pe, int i) {
#pragma clang fp contract(off)
        const int q = md.pseq[i];
        if (pe.kind == 0) return prior_term(pe.term, th[q]);
        const double* sc = th + md.off_kep + 5 * (PSEQ_ECC - q) + 3;
        const double x = sc[0] * sc[0] + sc[1] * sc[1];
        return prior_term(pe.term, x);
    });
}

// Planet p's constants of the full parameter vector th.  The table is for mean
// anomalies that reduce to [0, pi] and eccentricities of an orbit: its start goes
// into the sin/cos table's index unclamped.  Any other planet takes Markley's
// start, which is clamped.
__device__ __forceinline__ PlanetC planet_slot(const ModelDev& md, const double* th, int p) {
    PlanetC pc = planet_setup(th + md.off_kep + 5 * p, md.param, md.use_c);
    const double reach = __builtin_fabs(pc.freq) * (md.t[md.N] + __builtin_fabs(pc.tp)) + __builtin_fabs(pc.phase);
    const bool table = md.N >= KT_MIN_EPOCHS && !pc.bad && pc.e <= KT_EMAX && reach <= KT_MMAX;
    pc.ktab = !table ? 0 : md.N < KT_SHORT ? 2 : 1;
    return pc;
}

// Largest phase of a cosine term: reduce_2pi leaves up to 1.2e-16 of it above pi,
// here 4.2e-3 rad, within the half step (6.1e-3) that the sin/cos table takes.
constexpr double COS_MMAX = 35184372088832.0;      // 2^45

// The slot's other constants (instruments, acceleration, cosine terms) and the
// planets' Kepler path flags, kf those of planet `lane`.  Called by a whole wave.
template <class SL>
__device__ __forceinline__ void slot_rest(const ModelDev& md, SL& sl, int lane, int kf) {
    // the whole wave calls these: flag bit b of planet p to mask bit 4 p + b
    unsigned m = 0;
    for (int b = 0; b < 4; ++b) {
        const unsigned long long bits = __ballot((kf >> b) & 1);
        for (int p = 0; p < KMAX; ++p) m |= (unsigned)((bits >> p) & 1ull) << (4 * p + b);
    }
    if (lane == 0) sl.ktab_mask = (int)m;
    if (lane < md.I) {
        sl.gam[lane] = sl.theta[md.off_off + lane];
        double j = md.has_jit ? sl.theta[md.off_jit + lane] : 0.0;
        sl.jit[lane] = j;
        sl.jit2[lane] = j * j;
        if (md.ma_active) {
            int set = md.ma_global ? 0 : lane;
            sl.ma_c[lane] = sl.theta[md.off_ma + 2 * md.ma_q * set];
            sl.ma_tau[lane] = sl.theta[md.off_ma + 2 * md.ma_q * set + 1];
        }
    }
    if (lane < md.acc) sl.acc[lane] = sl.theta[md.off_acc + lane];
    if (lane < md.n_cos) {
        // Term 0 is the sinusoid when there is one (sinusoid00.model:2-5:
        // freq = 2 pi / P); the magnetic cycle's terms are (A1, pi / P, phase1)
        // and (A2, 2 pi / P, phase2) (magneticcycle00.model:2-8).
        const int c = md.off_sin >= 0 ? lane - 1 : lane;
        double A, f, ph;
        if (c < 0) {
            const double* th = sl.theta + md.off_sin;
            A = th[1]; f = (2.0 * PI_D) / th[0]; ph = th[2];
        } else {
            const double* th = sl.theta + md.off_mag;
            A = th[1 + c]; f = (c == 0 ? PI_D : 2.0 * PI_D) / th[0]; ph = th[3 + c];
        }
        // A phase beyond FP64's resolution reduces to no angle of the sin/cos
        // table: such a term is held at phase 0 (one that is not finite stays so).
        const double reach = __builtin_fabs(f) * md.t[md.N] + __builtin_fabs(ph);
        if (reach > COS_MMAX && reach < __builtin_inf()) f = ph = 0.0;
        sl.cosw[lane][0] = A;
        sl.cosw[lane][1] = f;
        sl.cosw[lane][2] = ph;
    }
}

// Per-slot constants (planets, instruments, acceleration) into LDS.
// Called by the slot's first wave; the caller synchronises afterwards.
template <class SL>
__device__ inline void slot_setup(const ModelDev& md, SL& sl, int lane) {
    int kf = 0;
    if (lane < md.K) {
        const PlanetC pc = planet_slot(md, sl.theta, lane);
        kf = kt_flags(pc.ktab, pc.e);
        sl.planet[lane] = pc;
    }
    slot_rest(md, sl, lane, kf);
}

struct TileLDS {
    double t[TILE], y[TILE], s2[TILE], dt[TILE];
    int ins[TILE];
    SinCosTab tab;
};

// The sin/cos table is read by every planet-epoch; load it once per workgroup.
__device__ __forceinline__ void tab_load(const ModelDev& md, SinCosTab& tab) {
    for (int j = threadIdx.x; j <= SC_N; j += blockDim.x) tab.v[j] = md.sctab[j];
}

__device__ __forceinline__ void tile_load(const ModelDev& md, TileLDS& tl, int tb, int tn) {
    for (int j = threadIdx.x; j < tn; j += blockDim.x) {
        tl.t[j] = md.t[tb + j];
        tl.y[j] = md.y[tb + j];
        tl.s2[j] = md.s2[tb + j];
        tl.ins[j] = md.ins[tb + j];
        if (md.ma_active) tl.dt[j] = md.dt[tb + j];
    }
}

// Per-slot constants, then the per-vector Kepler tables, one planet per wave
// of the slot.  Every wave of the vector calls this; the vector's theta must be
// in the slot and visible to them.
template <int WPT, class SL>
__device__ __forceinline__ void slot_prepare(const ModelDev& md, SL& sl, bool live, int wsub, int lane) {
    if (live && wsub == 0) slot_setup(md, sl, lane);
    vec_sync<WPT>();
    if (live) {
        for (int p = wsub; p < md.K; p += WPT)
            if (sl.planet[p].ktab) ktab_fill(sl.planet[p], lane, sl.ktab[p][lane]);
    }
    vec_sync<WPT>();
}

// A value that is the same in every lane of the wave (every kernel keeps
// one parameter vector per wave), read into a scalar register so that a
// branch on it is a scalar branch.
__device__ __forceinline__ int wave_uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Vectors per workgroup of the kernels whose vectors are independent: with one
// wave per vector four of them share the workgroup's sin/cos table.
constexpr int vecs_per_wg(int wpt) { return wpt == 1 ? 4 : 1; }

// The model's planets are parameterised by the time of periastron
// (block_repo.py:23-31, parameterisations 3 and 4).
__host__ __device__ __forceinline__ bool model_tp(const ModelDev& md) { return md.param == 3 || md.param == 4; }

// Model value (planets + offset + acceleration) of the lane's NE epochs.
// kmask: the slot's SlotLDS::ktab_mask as a wave-uniform scalar (kt_path).
template <int PREC, int NE, class SL>
__device__ __forceinline__ void epoch_mu(const ModelDev& md, const SL& sl, const SinCosTab& tb, const double (&t)[NE],
                                         const int (&k)[NE], int kmask, double (&mu)[NE]) {
#pragma unroll
    for (int i = 0; i < NE; ++i) {
        mu[i] = sl.gam[k[i]];
        if (md.acc) {
            const double x = t[i] - md.t0;
            double v = 0.0;
            for (int a = 0; a < md.acc; ++a) v = __builtin_fma(v, x, sl.acc[a]);
            mu[i] += v * x;
        }
    }
    // The planet loop twice, one copy per parameterisation (a model-wide
    // choice), so that no planet-epoch branches on it.
    if (model_tp(md)) {
        for (int p = 0; p < md.K; ++p)
            planet_mu<PREC, NE>(sl.planet[p], tb, sl.ktab[p], t, mu, true, kt_mode(kmask, p));
    } else {
        for (int p = 0; p < md.K; ++p)
            planet_mu<PREC, NE>(sl.planet[p], tb, sl.ktab[p], t, mu, false, kt_mode(kmask, p));
    }
}

// Phase freq * t + phase of cosine term c, rounded as numpy rounds
// `freq * X_ + phase` (no contraction).
template <class SL>
__device__ __forceinline__ double cos_phase(const SL& sl, int c, double t) {
#pragma clang fp contract(off)
    return sl.cosw[c][1] * t + sl.cosw[c][2];
}

// Terms added after the moving average: in the reference's block order
// StellarActivity, Sinusoid and MagneticCycle follow MOAV (emp/emp.py:
// 2628-2650), so the MA residuals do not contain them.
__host__ __device__ inline bool has_post(const ModelDev& md) { return md.n_cos > 0 || md.sai_w > 0; }

// Model features the common models do not use: 0 none of them, 1 terms added
// after the MA (activity and cosine terms), 2 also MA orders above 1.  Kernels
// come in instances that compile the others out, so that the common ones keep
// their register budget.
__host__ __device__ inline int model_ext(const ModelDev& md) {
    return md.ma_active && md.ma_q > 1 ? 2 : has_post(md) ? 1 : 0;
}

// Their sum at epoch n (device order; time t, instrument k): the activity
// columns of the epoch's instrument times their coefficients (sai00.model),
// then the cosine terms, whose angle is reduced in FP64 and whose cosine
// comes from the FP64 table on both precision paths.
template <class SL>
__device__ __forceinline__ double epoch_post(const ModelDev& md, const SL& sl, const SinCosTab& tb, double t,
                                             int n, int k) {
    double v = 0.0;
    if (md.sai_w) {
        const int b0 = md.sai_base[k], nc = md.sai_base[k + 1] - b0;
        const double* zeta = sl.theta + md.off_sai + b0;
#pragma unroll 1
        for (int c = 0; c < nc; ++c) v = __builtin_fma(zeta[c], md.sai[(size_t)c * md.N + n], v);
    }
#pragma unroll 1
    for (int c = 0; c < md.n_cos; ++c) {
        double sn, cs;
        sincos_tab(tb, __builtin_fabs(reduce_2pi(cos_phase(sl, c, t))), sn, cs);
        v = __builtin_fma(sl.cosw[c][0], cs, v);
    }
    return v;
}

// Affine map composition for the MA(1) recurrence eps_i = a_i eps_{i-1} + b_i:
// applying (a1, b1) then (a2, b2) gives (a2 a1, a2 b1 + b2).  Inclusive scan
// over the wave by DPP: within rows of 16 lanes, then across rows; lanes
// without a source compose with the identity (1, 0).  Whole wave active.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ void affine_step(double& a, double& b) {
    double pa, pb;
    if constexpr (ROW_MASK == 0xf && CTRL > 0x110 && CTRL < 0x120) {
        pa = dpp_shr_one_f64<CTRL>(a);
        pb = dpp_shr_zero_f64<CTRL>(b);
    } else {
        pa = dpp_f64<CTRL, ROW_MASK>(1.0, a);
        pb = dpp_f64<CTRL, ROW_MASK>(0.0, b);
    }
    b = __builtin_fma(a, pb, b);
    a = a * pa;
}

__device__ __forceinline__ void wave_affine_scan(double& a, double& b, int lane) {
    (void)lane;
    affine_step<0x111, 0xf>(a, b);
    affine_step<0x112, 0xf>(a, b);
    affine_step<0x114, 0xf>(a, b);
    affine_step<0x118, 0xf>(a, b);
    affine_step<0x142, 0xa>(a, b);
    affine_step<0x143, 0xc>(a, b);
}

// MA(q), q >= 2: the order-q recurrence (moav01.model:7-15)
//   eps_i = r_i + sum_{c<q} a_{i,c} eps_{i-1-c},
//   a_{i,c} = -phi_c exp(-|t_i - t_{i-1-c}| / tau_c)  (0 when epoch i-1-c is
//   not in the segment),
// as an affine map on the state (eps_i, ..., eps_{i-Q+1}): a companion matrix
// whose first row is (a_{i,0}, ..., a_{i,Q-1}) plus (r_i, 0, ...).  Maps are
// composed over the wave by DPP exactly as the order-1 scan composes its
// (a, b) pairs; lanes without a source compose with the identity.
template <int Q, int CTRL, int ROW_MASK>
__device__ __forceinline__ void affq_step(double (&m)[Q][Q], double (&v)[Q]) {
    double pm[Q][Q], pv[Q];
#pragma unroll
    for (int a = 0; a < Q; ++a) {
#pragma unroll
        for (int b = 0; b < Q; ++b) pm[a][b] = dpp_f64<CTRL, ROW_MASK>(a == b ? 1.0 : 0.0, m[a][b]);
        pv[a] = dpp_f64<CTRL, ROW_MASK>(0.0, v[a]);
    }
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

// The companion map of epoch n (time t, instrument k, residual r); the
// identity for an epoch past the series' end.
template <int Q, class SL>
__device__ __forceinline__ void maq_map(const ModelDev& md, const SL& sl, bool valid, int n, double t, int k, double r,
                                        double (&m)[Q][Q], double (&v)[Q]) {
#pragma unroll
    for (int a = 0; a < Q; ++a) {
        v[a] = 0.0;
#pragma unroll
        for (int b = 0; b < Q; ++b) m[a][b] = a == b ? 1.0 : 0.0;
    }
    if (!valid) return;
    const int q = md.ma_q;
    const double* ph = sl.theta + md.off_ma + 2 * q * (md.ma_global ? 0 : k);
#pragma unroll
    for (int c = 0; c < Q; ++c) {
        double a = 0.0;
        const int n1 = n - 1 - c;
        if (c < q && n1 >= 0 && (md.ma_global || md.ins[n1] == k))
            a = -(ph[2 * c] * exp(-__builtin_fabs(t - md.t[n1]) / ph[2 * c + 1]));
        m[0][c] = a;
    }
#pragma unroll
    for (int a = 1; a < Q; ++a)
#pragma unroll
        for (int b = 0; b < Q; ++b) m[a][b] = b == a - 1 ? 1.0 : 0.0;
    v[0] = r;
}

// One chunk of the order-q MA: the lane's NE epochs from n0 on (their times,
// instruments, residuals) and the state carried in from the previous chunk
// (`carry`, updated).  eps of the lane's epochs.  Whole wave active; with WPT > 1
// all waves of the workgroup call this together (one barrier).
template <int Q, int WPT, int NE, class SL>
__device__ __forceinline__ void ma_chunk_q(const ModelDev& md, const SL& sl, const bool (&valid)[NE], int n0,
                                           const double (&t)[NE], const int (&k)[NE], const double (&r)[NE], int lane,
                                           int wave, int wsub, int& parity, double (&carry)[4], double (&eps)[NE]) {
    __shared__ double qtot[2][MAX_WAVES][Q * Q + Q];
    double m0[Q][Q], v0[Q], m[Q][Q], v[Q];
    maq_map<Q>(md, sl, valid[0], n0, t[0], k[0], r[0], m0, v0);
    if constexpr (NE == 1) {
#pragma unroll
        for (int a = 0; a < Q; ++a) {
            v[a] = v0[a];
#pragma unroll
            for (int b = 0; b < Q; ++b) m[a][b] = m0[a][b];
        }
    } else {
        double m1[Q][Q], v1[Q];
        maq_map<Q>(md, sl, valid[1], n0 + 1, t[1], k[1], r[1], m1, v1);
#pragma unroll
        for (int a = 0; a < Q; ++a) {
            double acc = v1[a];
#pragma unroll
            for (int b = 0; b < Q; ++b) acc = __builtin_fma(m1[a][b], v0[b], acc);
            v[a] = acc;
#pragma unroll
            for (int c = 0; c < Q; ++c) {
                double e = 0.0;
#pragma unroll
                for (int b = 0; b < Q; ++b) e = __builtin_fma(m1[a][b], m0[b][c], e);
                m[a][c] = e;
            }
        }
    }
    affq_step<Q, 0x111, 0xf>(m, v);
    affq_step<Q, 0x112, 0xf>(m, v);
    affq_step<Q, 0x114, 0xf>(m, v);
    affq_step<Q, 0x118, 0xf>(m, v);
    affq_step<Q, 0x142, 0xa>(m, v);
    affq_step<Q, 0x143, 0xc>(m, v);
    double sin_[Q];
    if (WPT == 1) {
#pragma unroll
        for (int a = 0; a < Q; ++a) sin_[a] = carry[a];
    } else {
        if (lane == 63) {
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
        for (int w = 0; w < WPT; ++w) {
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
    double st[Q];                       // the state after the lane's last epoch
#pragma unroll
    for (int a = 0; a < Q; ++a) {
        double acc = v[a];
#pragma unroll
        for (int b = 0; b < Q; ++b) acc = __builtin_fma(m[a][b], sin_[b], acc);
        st[a] = acc;
    }
    if (WPT == 1) {
#pragma unroll
        for (int a = 0; a < Q; ++a) carry[a] = readlane_f64(st[a], 63);
    }
    eps[NE - 1] = st[0];
    if constexpr (NE == 2) {
        double e = v0[0];
#pragma unroll
        for (int b = 0; b < Q; ++b) e = __builtin_fma(m0[0][b], wave_prev(st[b], sin_[b]), e);
        eps[0] = e;
    }
}

// One suffix step within rows of 16 lanes: lane i composes with lane i + n
// of its row (row_shl:n), the last n lanes of a row with the identity.
template <int CTRL>
__device__ __forceinline__ void affine_suffix_step(double& a, double& b) {
    const double pa = dpp_shr_one_f64<CTRL>(a);
    const double pb = dpp_shr_zero_f64<CTRL>(b);
    b = __builtin_fma(a, pb, b);
    a = a * pa;
}

// Suffix composition for the adjoint of that recurrence, lambda_i = b_i +
// a_i lambda_{i+1}: afterwards lane i holds the map of lanes i..63, so that
// lambda_i = b + a lambda_in with lambda_in the value after lane 63.  Within
// rows by DPP, after which lane i holds the map of lanes i to the end of its
// row and the first lane of a row that of the whole row; then across rows as
// the prefix scan does it mirrored: rows 0 and 2 compose with the first lane
// of the next row, rows 0 and 1 with lane 32 (by then rows 2 and 3).  Whole
// wave active.
__device__ __forceinline__ void wave_affine_suffix_scan(double& a, double& b, int lane) {
    affine_suffix_step<0x101>(a, b);
    affine_suffix_step<0x102>(a, b);
    affine_suffix_step<0x104>(a, b);
    affine_suffix_step<0x108>(a, b);
    {
        const int src = (lane & 48) + 16;
        const double pa = __shfl(a, src, 64), pb = __shfl(b, src, 64);
        if (!(lane & 16)) {
            b = __builtin_fma(a, pb, b);
            a = a * pa;
        }
    }
    {
        const double pa = readlane_f64(a, 32), pb = readlane_f64(b, 32);
        if (lane < 32) {
            b = __builtin_fma(a, pb, b);
            a = a * pa;
        }
    }
}

struct ScanLDS {
    double2 tot[2][MAX_WAVES];     // per wave: its chunk's affine map (double-buffered)
    double red[MAX_WAVES][2];
};

// MA(1) multiplier of an epoch from its instrument and its MA column (the
// fixed-timescale weight, or dt with -1 at a segment start).
template <class SL>
__device__ __forceinline__ double ma_mult(const ModelDev& md, const SL& sl, int k, double col) {
    if (md.ma_wfixed) return -(sl.ma_c[k] * col);
    return col < 0.0 ? 0.0 : -(sl.ma_c[k] * exp(-col / sl.ma_tau[k]));
}

// Two consecutive values of a column at n in one load (aligned as one value is):
// two loads fetch every cache line twice, which bounds models without planets
// (8192 vectors of 10^4 epochs 157 -> 97 us).
template <class T>
__device__ __forceinline__ void load_pair(const T* p, int n, T (&v)[2]) {
    typedef T T2 __attribute__((ext_vector_type(2), aligned(sizeof(T))));
    const T2 q = *(const T2*)(p + n);
    v[0] = q.x;
    v[1] = q.y;
}

// One chunk of the likelihood: NE consecutive epochs per lane from cb on.
// Adds to the lane's chi^2 and log-determinant product; carries the MA state.
template <int PREC, int WPT, bool WRITE, bool WEPS, int EXT, int NE, class SL>
__device__ __forceinline__ void lnl_chunk(const ModelDev& md, const SL& sl, const SinCosTab& tab, ScanLDS& sc,
                                          bool live, int cb, int lane, int wave, int wsub, int kmask, double& chi,
                                          double& prod, int& pexp, double& carry, double (&qcarry)[4], int& parity,
                                          double* out_model, double* out_err2, double* out_eps) {
    const int n0 = cb + NE * (wsub * 64 + lane);
    const bool need_t = EXT >= 1 || md.K > 0 || md.acc > 0;
    double t[NE], y[NE], err2[NE], dtc[NE], r[NE], mu[NE];
    int k[NE];
    bool valid[NE];
#pragma unroll
    for (int i = 0; i < NE; ++i) {
        const int n = n0 + i;
        valid[i] = live && n < md.N;
        t[i] = y[i] = dtc[i] = r[i] = mu[i] = 0.0;
        err2[i] = 1.0;
        k[i] = 0;
        if (NE == 1 && valid[i]) {
            if (need_t) t[i] = md.t[n];
            k[i] = md.ins[n];
            y[i] = md.y[n];
            err2[i] = md.s2[n];
            if (md.ma_active) dtc[i] = md.dt[n];
        }
    }
    if constexpr (NE == 2) {
        if (valid[1]) {
            if (need_t) load_pair(md.t, n0, t);
            load_pair(md.ins, n0, k);
            load_pair(md.y, n0, y);
            load_pair(md.s2, n0, err2);
            if (md.ma_active) load_pair(md.dt, n0, dtc);
        } else if (valid[0]) {
            t[0] = md.t[n0];
            k[0] = md.ins[n0];
            y[0] = md.y[n0];
            err2[0] = md.s2[n0];
            if (md.ma_active) dtc[0] = md.dt[n0];
        }
    }
    // a wave past the series' end only takes part in the scan's barrier
    if (live && cb + NE * (wsub * 64) < md.N) {
        epoch_mu<PREC, NE>(md, sl, tab, t, k, kmask, mu);
#pragma unroll
        for (int i = 0; i < NE; ++i) {
            if (valid[i]) {
                err2[i] += sl.jit2[k[i]];
                r[i] = y[i] - mu[i];
            }
        }
    }
    double eps[NE];
#pragma unroll
    for (int i = 0; i < NE; ++i) eps[i] = r[i];
    if (EXT == 2 && md.ma_active && md.ma_q > 1) {
        if (md.ma_q == 2) ma_chunk_q<2, WPT, NE>(md, sl, valid, n0, t, k, r, lane, wave, wsub, parity, qcarry, eps);
        else ma_chunk_q<4, WPT, NE>(md, sl, valid, n0, t, k, r, lane, wave, wsub, parity, qcarry, eps);
    } else if (md.ma_active) {
        double am[NE];
#pragma unroll
        for (int i = 0; i < NE; ++i) am[i] = valid[i] ? ma_mult(md, sl, k[i], dtc[i]) : 1.0;
        double a = am[0], b = r[0];         // the lane's epochs composed
        if constexpr (NE == 2) {
            b = __builtin_fma(am[1], r[0], r[1]);
            a = am[1] * am[0];
        }
        wave_affine_scan(a, b, lane);
        double e0 = carry;                  // eps before this wave's epochs
        if (WPT > 1) {
            if (lane == 63) sc.tot[parity][wave] = make_double2(a, b);
            __syncthreads();
            const int w0 = wave - wsub;
            double2 tot[WPT];
#pragma unroll
            for (int w = 0; w < WPT; ++w) tot[w] = sc.tot[parity][w0 + w];
            double pa = tot[0].x, pb = tot[0].y;    // the maps of waves 0 .. w composed
#pragma unroll
            for (int w = 1; w < WPT; ++w) {
                if (w == wsub) e0 = __builtin_fma(pa, carry, pb);
                pb = __builtin_fma(tot[w].x, pb, tot[w].y);
                pa = tot[w].x * pa;
            }
            carry = __builtin_fma(pa, carry, pb);
            parity ^= 1;
        }
        eps[NE - 1] = __builtin_fma(a, e0, b);
        if (WPT == 1) carry = readlane_f64(eps[NE - 1], 63);
        if constexpr (NE == 2) eps[0] = __builtin_fma(am[0], wave_prev(eps[1], e0), r[0]);
    }
#pragma unroll
    for (int i = 0; i < NE; ++i) {
        if (valid[i]) {
            const double cs = (EXT >= 1 && has_post(md)) ? epoch_post(md, sl, tab, t[i], n0 + i, k[i]) : 0.0;
            const double res = eps[i] - cs;
            chi = __builtin_fma(res * res, rcp_path<PREC>(err2[i]), chi);
            prod *= err2[i];
            pexp += __builtin_amdgcn_frexp_exp(prod);
            prod = __builtin_amdgcn_frexp_mant(prod);
            if (WRITE) {
                out_model[n0 + i] = mu[i] + (r[i] - eps[i]) + cs;
                out_err2[n0 + i] = err2[i];
            }
            if (WEPS) out_eps[n0 + i] = eps[i];
        }
    }
}

// lnL of the parameter vector in slot sl, by its WPT waves (wave `wsub` of
// them; `wave` in the workgroup).  With WPT > 1 all threads of the workgroup
// call this together (it holds barriers); `live` == false then skips the
// arithmetic.  The slot must be prepared (slot_prepare) and the sin/cos table
// loaded.  With WRITE the per-epoch model and err2 are stored (device order);
// with WEPS the per-epoch MA-filtered residual eps (= r without MA; before the
// terms added after the MA are taken off).  EXT as model_ext.
//
// Bound by VALU issue for long series and large batches, by latency for small
// ones.  Two consecutive epochs per lane: the planet's constants, the path's
// branches and the MA scan (whose maps compose pairwise first) are paid once
// for both, and their Kepler chains interleave.  One vector per workgroup (from
// two waves on) and no tile staging: one barrier per chunk with the MA, none
// without.  Measured against one epoch per lane with LDS tiles shared by the
// vectors of a 512-thread workgroup: 8192 vectors of 7 planets x 10^4 epochs,
// MA(1), mixed, 1.10 -> 0.93 ms; 2560 of 3 x 1530 FP64 45 -> 38 us; 1283 of 4 x
// 783 with a sinusoid 43 -> 22 us (that instance also lost the MA orders above
// 1, 84 -> 74 VGPRs); stretch sweeps at 16 x 1024 x 10^4, FP64, 3.6 -> 2.5 ms.
template <int PREC, int WPT, bool WRITE, bool WEPS = false, int EXT = 2, class SL>
__device__ double vec_lnl(const ModelDev& md, const SL& sl, const SinCosTab& tab, ScanLDS& sc, bool live, int wsub,
                          double* out_model = nullptr, double* out_err2 = nullptr, double* out_eps = nullptr) {
    const int lane = threadIdx.x & 63;
    const int wave = wave_uniform(threadIdx.x >> 6);
    constexpr int G = 64 * WPT;
    const int kmask = kt_path<PREC>(wave_uniform(sl.ktab_mask));
    double chi = 0.0, prod = 1.0;
    int pexp = 0;
    double carry = 0.0;
    double qcarry[4] = {0.0, 0.0, 0.0, 0.0};   // MA(q >= 2) state carried between chunks
    int parity = 0;
    int cb = 0;
    for (; cb + G < md.N; cb += 2 * G)
        lnl_chunk<PREC, WPT, WRITE, WEPS, EXT, 2>(md, sl, tab, sc, live, cb, lane, wave, wsub, kmask, chi, prod, pexp,
                                                   carry, qcarry, parity, out_model, out_err2, out_eps);
    if (cb < md.N)
        lnl_chunk<PREC, WPT, WRITE, WEPS, EXT, 1>(md, sl, tab, sc, live, cb, lane, wave, wsub, kmask, chi, prod, pexp,
                                                   carry, qcarry, parity, out_model, out_err2, out_eps);
    double ld = live ? log(prod) + (double)pexp * LN2 : 0.0;
    chi = wave_sum(chi);
    ld = wave_sum(ld);
    if (WPT > 1) {
        if (lane == 0) { sc.red[wave][0] = chi; sc.red[wave][1] = ld; }
        __syncthreads();
        chi = 0.0; ld = 0.0;
        const int w0 = wave - wsub;
        for (int w = 0; w < WPT; ++w) { chi += sc.red[w0 + w][0]; ld += sc.red[w0 + w][1]; }
    }
    return -0.5 * (chi + ld) + md.lnl_const;
}

// Expand the free vector (global memory, row `row`) into the slot's full
// vector in LDS, re-inserting fixed values (emp/emp_model.py:709-711).
template <class SL>
__device__ __forceinline__ void expand_theta(const ModelDev& md, SL& sl, const double* row, int g, int G) {
    for (int j = g; j < md.Dfull; j += G) {
        const int f = md.inv_free[j];
        sl.theta[j] = f >= 0 ? row[f] : md.fixed_val[j];
    }
}

}  // namespace emp

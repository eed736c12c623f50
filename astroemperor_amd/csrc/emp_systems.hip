// Batched independent systems: S separate RV models, each with its own
// parallel-tempering ensemble, advanced together, a few kernel launches per
// sweep of all of them (replayed from a hipGraph).
//
// A half-step is two passes.  The prior pass, one workgroup per system, draws
// the proposals, evaluates their priors and lists those inside the support.
// The likelihood pass gives every workgroup up to `chunk` listed walkers of one
// system: their vectors, planet constants and acceptance operands are set up
// for all of them at once (one lane per walker and planet, instead of one wave
// per walker with a few lanes busy), then each wave takes walkers on its own.
// Workgroups run longest system first, so the ragged tail of small systems
// fills in behind the big ones, and the longest system's walkers spread over
// the chip.  The swap pass, one workgroup per system, ends the sweep; its last
// workgroup advances the sweep counter, so the captured launches replay
// unchanged and no workgroup ever waits for another.
//
// Randomness: the counters of the single-system engine with the system index
// mixed in (system 0 draws exactly what the single-system engine draws).
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <vector>

#include "emp_pt_common.h"

using namespace emp;

constexpr int SYS_MAX_TASKS = 512;   // T W / 2 per system
constexpr int SYS_PASS = 256;        // threads of the prior and swap passes
constexpr int SYS_SCRATCH = 24 * 1024;   // working copies of the swap pass: 12 (2 T - 1) W bytes, T W <= 1024

struct SysDev {
    int S, T, W, nsteps;
    double a;
    uint32_t key0, key1;
    int adapt_mode;
    double adapt_tau, adapt_nu;
    const ModelDev* md;        // [S]
    const int* order;          // [S] queue order
    const int64_t* xoff;       // [S] first element of system s in X
    double* X;                 // system after system: [T W slots][D_s]
    double* lnl;               // [S][T W] by slot
    double* lnp;               // [S][T W]
    int* map;                  // [S][T W] position -> slot
    double* betas;             // [S][T]
    long long* accepted;       // [S][T W] by position
    double* tsw_sum;           // [S][T-1] summed over sweeps
    double* smd_sum;           // [S][T-1]
    unsigned long long* ctl;   // (unused), swap workgroups finished, sweeps done, likelihoods evaluated
    double* tlp;               // [S][T W/2] ln prior of each task's proposal
    int* list;                 // [S][T W/2] tasks inside the prior support
    int* nlive;                // [2][S] how many, per half
    int rec_every, rec_temps;
    int64_t max_rec;
    const int64_t* rxoff;      // [S] first element of system s in one record of h_x
    int64_t rec_x;             // elements of one record of h_x
    double* h_x;               // [R][sum_s rec_temps W D_s]
    double* h_lnl;             // [R][S][rec_temps W]
    double* h_lnp;             // [R][S][rec_temps W]
};

// The model table does not change during a launch.  Reading it through the
// constant address space lets the compiler re-load a field where it is used
// instead of holding the whole ModelDev in registers across the sweep.
typedef __attribute__((address_space(4))) const ModelDev ConstModelDev;

__device__ __forceinline__ const ModelDev& sys_model(const SysDev& sd, int s) {
    const ConstModelDev* c = (const ConstModelDev*)sd.md;
    return *(const ModelDev*)&c[s];
}

__device__ __forceinline__ PTView sys_view(const SysDev& sd, int s, int D) {
    const size_t TW = (size_t)sd.T * sd.W;
    return pt_view(sd.T, sd.W, D, sd.a, sd.key0, sd.key1, (uint32_t)s, sd.adapt_mode, sd.adapt_tau, sd.adapt_nu,
                   sd.X + sd.xoff[s], sd.lnl + s * TW, sd.lnp + s * TW, sd.map + s * TW, sd.betas + (size_t)s * sd.T,
                   sd.accepted + s * TW);
}

// The prior pass: workgroup (s, c) (from system s0 on) takes the c-th SYS_PRIOR_TASKS tasks of
// system s: the proposals (one thread per task), every (task, term) pair of the
// prior's summation sequence (the system's resolved sequence in LDS, all loads
// of the walkers' rows in flight together), then the sum of each task's terms in
// sequence order with prior_wave's -inf return (one thread per task),
// bit-identical to prior_wave.  The tasks inside the support are appended to the
// system's list (in any order: the tasks of a half-step are independent); the
// other half's count is cleared for its next pass.  The term values take
// `terms` doubles of LDS, a few tasks at a time where a long sequence needs it.
// Latency-bound; measured against one workgroup per system with the sequence
// read from global memory for every term: 110 -> 24 us for 512 systems of 8 x 64
// walkers.
constexpr int SYS_PRIOR_TASKS = 64;
__host__ __device__ inline size_t sys_prior_terms(int L) {
    const size_t want = (size_t)SYS_PRIOR_TASKS * L, cap = 4096;
    return want < cap ? want : (cap > (size_t)L ? cap : (size_t)L);
}
__global__ __launch_bounds__(SYS_PASS) void k_sys_prior(SysDev sd, int s0, int half, int step, int nchunk, int terms_cap) {
#pragma clang fp contract(off)
    extern __shared__ __align__(16) char s_dyn[];
    __shared__ double s_z[SYS_PRIOR_TASKS];
    __shared__ int s_k[SYS_PRIOR_TASKS], s_j[SYS_PRIOR_TASKS];
    const int tid = threadIdx.x;
    const int sl = blockIdx.x / nchunk, s = s0 + sl, b0 = (blockIdx.x - sl * nchunk) * SYS_PRIOR_TASKS;
    const ModelDev& md = sys_model(sd, s);
    const PTView pv = sys_view(sd, s, md.D);
    const int ntask = sd.T * (sd.W / 2), nt = min(SYS_PRIOR_TASKS, ntask - b0), L = md.npseq;
    double* terms = (double*)s_dyn;
    PseqEntry* seq = (PseqEntry*)(terms + terms_cap);
    int* nlive = sd.nlive + (size_t)half * sd.S + s;
    if (b0 == 0 && tid == 0) sd.nlive[(size_t)(1 - half) * sd.S + s] = 0;
    for (int i = tid; i < L; i += SYS_PASS) seq[i] = md.pseq_e[i];
    if (tid < nt) {
        const Proposal pr = pt_propose(pv, (long long)sd.ctl[2], half, step, b0 + tid);
        s_z[tid] = pr.z;
        s_k[tid] = pr.sk;
        s_j[tid] = pr.sj;
    }
    __syncthreads();
    const int per = min(nt, terms_cap / L);
    for (int c0 = 0; c0 < nt; c0 += per) {
        const int cn = min(per, nt - c0);
        for (int e = tid; e < cn * L; e += SYS_PASS) {
            const int bl = e / L, i = e - bl * L, r = c0 + bl;
            const PseqEntry& pe = seq[i];
            if (pe.kind == 2) continue;
            const double* Xk = pv.X + (size_t)s_k[r] * pv.D;
            const double* Xj = pv.X + (size_t)s_j[r] * pv.D;
            double x;
            if (pe.kind == 0) {
                x = pt_prop_value(Xk, Xj, s_z[r], pe.fa);
            } else {
                const double s3 = pe.fa >= 0 ? pt_prop_value(Xk, Xj, s_z[r], pe.fa) : pe.va;
                const double s4 = pe.fb >= 0 ? pt_prop_value(Xk, Xj, s_z[r], pe.fb) : pe.vb;
                x = s3 * s3 + s4 * s4;
            }
            terms[e] = prior_term(pe.term, x);
        }
        __syncthreads();
        if (tid < 64) {                      // whole first wave (per <= 64)
            const bool own = tid < cn;
            double lp = 0.0;
            if (own) {
                const double* tv = terms + (size_t)tid * L;
                for (int i = 0; i < L; ++i) {
                    if (seq[i].kind == 2) {
                        if (lp == -__builtin_inf()) break;
                    } else {
                        lp += tv[i];
                    }
                }
                sd.tlp[(size_t)s * ntask + b0 + c0 + tid] = lp;
            }
            const bool live = own && lp > -__builtin_inf();
            const unsigned long long m = __ballot(live);
            int base = 0;
            if (tid == 0 && m) base = atomicAdd(nlive, __popcll(m));
            base = __builtin_amdgcn_readfirstlane(base);
            if (live) sd.list[(size_t)s * ntask + base + __popcll(m & ((1ull << tid) - 1ull))] = b0 + c0 + tid;
        }
        __syncthreads();
    }
}

// A walker's slot in the likelihood pass: its vector and planet constants are
// rows of the workgroup's, the rest belongs to the wave (or waves) at work on
// it.
template <class KTE>
struct SlotView {
    const double* theta;
    const PlanetC* planet;
    KTE (*ktab)[KT_N];
    double *gam, *jit2, *ma_c, *ma_tau, *jit, *acc;
    double (*cosw)[3];
    int ktab_mask;             // (lane 0's)
};
struct SlotRest {
    double gam[IMAX], jit2[IMAX], ma_c[IMAX], ma_tau[IMAX], jit[IMAX];
    double acc[AMAX];
    double cosw[CMAX][3];
};

constexpr int sys_vecs(int wpt) { return wpt == 1 ? 4 : 1; }       // walkers at work in a workgroup
constexpr int SYS_CHUNK = 16;                                       // most walkers per workgroup
template <int WPT>
using SysKTE = std::conditional_t<WPT == 1, float2, float4>;       // as the single-system engine's tables

// Dynamic LDS of the likelihood pass: `chunk` vectors and planet rows, and the
// Kepler tables of the walkers at work.
__host__ __device__ inline size_t sys_lds(int wpt, int chunk, int Dfull, int K) {
    const size_t kte = wpt == 1 ? sizeof(SysKTE<1>) : sizeof(SysKTE<2>);
    return (size_t)sys_vecs(wpt) * K * KT_N * kte + (size_t)chunk * (Dfull * sizeof(double) + K * sizeof(PlanetC));
}

// The likelihood pass: workgroup (it, c) takes the c-th `chunk` listed tasks of
// system it0 + it in queue order; with INIT instead every walker (the state
// loaded into slot = position order), whose prior and likelihood it stores.
// WPT waves per walker; EXT: the instance with the extended model features
// (model_ext), used when any system of the batch has them.
// Bound by VALU issue.  Measured against one persistent workgroup per compute
// unit that did a whole system's sweep at a time (16 walkers in step between
// barriers, each wave setting up its own walker, the sweep as long as the
// longest system's): per sweep of 64 / 512 / 2048 systems of 8 x 64 walkers, mixed,
// 824 -> 152, 1152 -> 701, 3820 -> 2457 us; 512 FP64 1853 -> 728 us.
template <int PREC, int WPT, bool EXT, bool INIT>
__global__ __launch_bounds__(64 * WPT * sys_vecs(WPT)) __attribute__((amdgpu_waves_per_eu(EXT ? 3 : 5))) void k_sys_lik(SysDev sd, int it0, int half, int step, int chunk,
                                                                     int nchunk) {
    constexpr int VECS = sys_vecs(WPT), NT = 64 * WPT * VECS;
    using KTE = SysKTE<WPT>;
    extern __shared__ __align__(16) char s_dyn[];
    __shared__ SinCosTab s_tab;
    __shared__ ScanLDS s_scan;
    __shared__ SlotRest s_rest[VECS];
    __shared__ TaskOps s_ops[SYS_CHUNK];
    __shared__ double s_z[SYS_CHUNK];
    __shared__ int s_k[SYS_CHUNK], s_j[SYS_CHUNK], s_acc[VECS];
    const int tid = threadIdx.x, wave = wave_uniform(tid >> 6), lane = tid & 63;
    const int it = blockIdx.x / nchunk, q0 = (blockIdx.x - it * nchunk) * chunk;
    const int s = __builtin_amdgcn_readfirstlane(sd.order[it0 + it]);
    const int ntask = INIT ? sd.T * sd.W : sd.T * (sd.W / 2);
    const int nl = INIT ? ntask : __builtin_amdgcn_readfirstlane(sd.nlive[(size_t)half * sd.S + s]);
    if (q0 >= nl) return;                    // the whole workgroup
    const int nt = min(chunk, nl - q0);
    const ModelDev& md = sys_model(sd, s);
    const PTView pv = sys_view(sd, s, md.D);
    const int Df = md.Dfull, K = md.K;
    KTE (*ktab)[KT_N] = (KTE (*)[KT_N])s_dyn;
    double* theta = (double*)(s_dyn + (size_t)VECS * K * KT_N * sizeof(KTE));
    PlanetC* planet = (PlanetC*)(theta + chunk * Df);
    tab_load(md, s_tab);
    if (tid < nt) {
        if (INIT) {
            s_z[tid] = 0.0;
            s_k[tid] = s_j[tid] = q0 + tid;
        } else {
            const int b = sd.list[(size_t)s * ntask + q0 + tid];
            const Proposal pr = pt_propose(pv, (long long)sd.ctl[2], half, step, b);
            s_z[tid] = pr.z;
            s_k[tid] = pr.sk;
            s_j[tid] = pr.sj;
            s_ops[tid] = pt_task_ops(pv, pr, sd.tlp[(size_t)s * ntask + b], md.D);
        }
    }
    __syncthreads();
    for (int e = tid; e < nt * Df; e += NT) {
        const int r = e / Df, f = md.inv_free[e - r * Df];
        double v = md.fixed_val[e - r * Df];
        if (f >= 0) {
            const double* Xk = pv.X + (size_t)s_k[r] * pv.D;
            v = INIT ? Xk[f] : pt_prop_value(Xk, pv.X + (size_t)s_j[r] * pv.D, s_z[r], f);
        }
        theta[e] = v;
    }
    __syncthreads();
    for (int e = tid; e < nt * K; e += NT) {
        const int r = e / K;
        planet[e] = planet_slot(md, theta + r * Df, e - r * K);
    }
    __syncthreads();
    const int slot = wave / WPT, wsub = wave - slot * WPT;
    SlotRest& rest = s_rest[slot];
    // one wave per walker: the waves work without waiting for one another
    // (two: one walker after the other, the workgroup together)
    for (int r = slot; r < nt; r += VECS) {
        vec_sync<WPT>();                     // the previous walker is finished with the slot
        SlotView<KTE> sl{theta + r * Df, planet + r * K, ktab + slot * K, rest.gam, rest.jit2, rest.ma_c,
                         rest.ma_tau, rest.jit, rest.acc, rest.cosw, 0};
        // every wave computes the mask (a register); the LDS values are the same
        slot_rest(md, sl, lane, lane < K ? kt_flags(sl.planet[lane].ktab, sl.planet[lane].e) : 0);
        for (int p = wsub; p < K; p += WPT)
            if (sl.planet[p].ktab) ktab_fill(sl.planet[p], lane, sl.ktab[p][lane]);
        vec_sync<WPT>();
        double ll = vec_lnl<PREC, WPT, false, false, EXT ? 2 : 0>(md, sl, s_tab, s_scan, true, wsub);
        if (INIT) {
            const double lp = prior_vector_wave(md, sl.theta, lane);
            if (wsub == 0 && lane == 0) {
                const int b = q0 + r;
                if (!(ll == ll) || ll == __builtin_inf()) ll = -__builtin_inf();
                pv.map[b] = b;
                pv.lnp[b] = lp;
                pv.lnl[b] = lp > -__builtin_inf() ? ll : -__builtin_inf();
            }
            continue;
        }
        if (wsub == 0 && lane == 0) s_acc[slot] = pt_decide(pv, s_ops[r], ll);
        vec_sync<WPT>();
        if (s_acc[slot]) {
            double* Xk = pv.X + (size_t)s_ops[r].sk * pv.D;
            for (int d = wsub * 64 + lane; d < md.D; d += 64 * WPT) Xk[d] = sl.theta[md.free_idx[d]];
        }
    }
    if (!INIT && tid == 0) atomicAdd(&sd.ctl[3], (unsigned long long)nt);
}

// The end of a sweep of one system: swap round, ladder, statistics, record.
__global__ __launch_bounds__(SYS_PASS) void k_sys_swap(SysDev sd) {
    __shared__ __align__(16) char s_scr[SYS_SCRATCH];
    __shared__ double s_bet[64], s_ld[64];
    __shared__ double s_red[64][2];
    __shared__ double s_rate[64], s_smd[64], s_sig[64];
    const int tid = threadIdx.x, s = blockIdx.x;
    const long long sweep = (long long)sd.ctl[2];
    const int T = sd.T, W = sd.W, TW = T * W;
    const ModelDev& md = sys_model(sd, s);
    const PTView pv = sys_view(sd, s, md.D);
    double* L = (double*)s_scr;
    double* LU = L + TW;
    int* Mp = (int*)(LU + (T - 1) * W);
    int* JP = Mp + TW;
    pt_swap_stage(pv, sweep, L, Mp, LU, JP, SYS_PASS);
    for (int e = tid; e < T; e += SYS_PASS) s_bet[e] = pv.betas[e];
    __syncthreads();
    pt_swap_round(pv, sweep, L, Mp, LU, JP, false, s_red, s_bet, SYS_PASS);
    for (int e = tid; e < TW; e += SYS_PASS) pv.map[e] = Mp[e];
    if (tid < T - 1) {
        const double r = s_red[tid][0] / W;
        s_rate[tid] = r;
        s_smd[tid] = s_red[tid][1] / W;
        sd.tsw_sum[(size_t)s * (T - 1) + tid] += r;
        sd.smd_sum[(size_t)s * (T - 1) + tid] += s_red[tid][1] / W;
    }
    if (sd.rec_every > 0 && (sweep + 1) % sd.rec_every == 0) {
        const long long r = (sweep + 1) / sd.rec_every - 1;
        if (r < sd.max_rec) {
            const int nw = sd.rec_temps * W, D = md.D;
            double* hx = sd.h_x + r * sd.rec_x + sd.rxoff[s];
            for (int e = tid; e < nw * D; e += SYS_PASS) {
                const int w = e / D, d = e - w * D;
                hx[e] = pv.X[(size_t)Mp[w] * D + d];
            }
            const size_t o = ((size_t)r * sd.S + s) * nw;
            for (int w = tid; w < nw; w += SYS_PASS) {
                sd.h_lnl[o + w] = pv.lnl[Mp[w]];
                sd.h_lnp[o + w] = pv.lnp[Mp[w]];
            }
        }
    }
    if (pv.adapt_mode == 2) pt_lnl_spread(pv, L, s_sig, SYS_PASS);
    __syncthreads();
    pt_ladder_update(pv, sweep, s_rate, s_smd, s_sig, s_bet, s_ld, SYS_PASS);
    if (tid == 0) {
        __threadfence();
        const unsigned long long f = atomicAdd(&sd.ctl[1], 1ull);
        if (f == (unsigned long long)gridDim.x - 1) {   // every other workgroup has read the counter
            sd.ctl[1] = 0ull;
            sd.ctl[2] = (unsigned long long)(sweep + 1);
        }
    }
}

// ---------------------------------------------------------------------------
// Host side.
// ---------------------------------------------------------------------------
struct EmpSystems {
    EmpSystemsDesc desc;
    SysDev dev;
    std::vector<void*> allocations;
    std::vector<int> D;
    std::vector<int64_t> xoff, rxoff;
    int* d_order_lpt = nullptr;
    int* d_order_input = nullptr;
    hipStream_t stream = nullptr;
    hipGraphExec_t graph_exec = nullptr;
    EmpSystemsTuning tune{};
    int n_cu = 256, device = 0;
    bool ext = false;          // some system needs the extended instance (model_ext)
    int max_d = 1, max_k = 1, max_l = 1;   // longest full vector, most planets, longest prior sequence of a system
    int64_t x_total = 0;
    double last_ms = -1.0;
    double* gather_buf = nullptr;    // device workspace of the state getters
    size_t gather_cap = 0;
};

#define EMP_SYS_CONFIGS(X) X(0, 1) X(0, 2) X(1, 1) X(1, 2)

// Walkers per likelihood workgroup: two or four for every walker at work in it
// (a workgroup's set-up serves them all), fewer while the pass has under eight
// workgroups per compute unit (512 systems of 8 x 64 walkers: 701 / 713 us per
// sweep at four / two; 64, with the mixed path's cheaper steps: 168 / 147).
static int chunk_of(const EmpSystems* p, int64_t tasks) {
    const int vecs = sys_vecs(p->tune.waves_per_theta);
    int per = p->tune.waves_per_wg == 16 ? 4 : 2;
    while (per > 1 && tasks < (int64_t)per * vecs * 8 * p->n_cu) per /= 2;
    return vecs * per;
}

// Systems per launch of `nchunk` workgroups of `nthr` threads each: a grid holds
// fewer than 2^32 threads.
static int systems_per_launch(int nchunk, int nthr) { return (int)(((int64_t)1 << 31) / ((int64_t)nchunk * nthr)); }

template <bool INIT>
static int launch_lik(EmpSystems* p, int half, int step) {
    const EmpSystemsTuning& tu = p->tune;
    const int prec = p->desc.precision, S = p->desc.n_systems;
    const int n = p->desc.ntemps * p->desc.nwalkers / (INIT ? 1 : 2), chunk = chunk_of(p, (int64_t)S * n);
    const int nchunk = (n + chunk - 1) / chunk;
    const size_t lds = sys_lds(tu.waves_per_theta, chunk, p->max_d, p->max_k);
    const int most = systems_per_launch(nchunk, 64 * tu.waves_per_theta * sys_vecs(tu.waves_per_theta));
#define EMP_CASE(P, WP)                                                                                      \
    if (prec == P && tu.waves_per_theta == WP) {                                                            \
        const dim3 nt(64 * WP * sys_vecs(WP));                                                               \
        for (int s0 = 0; s0 < S; s0 += most) {                                                              \
            const dim3 grid((unsigned)std::min(most, S - s0) * (unsigned)nchunk);                            \
            if (p->ext) hipLaunchKernelGGL((k_sys_lik<P, WP, true, INIT>), grid, nt, lds, p->stream, p->dev, s0, half, step, chunk, nchunk); \
            else hipLaunchKernelGGL((k_sys_lik<P, WP, false, INIT>), grid, nt, lds, p->stream, p->dev, s0, half, step, chunk, nchunk); \
            EMP_HIP(hipGetLastError());                                                                     \
        }                                                                                                    \
        return EMP_OK;                                                                                      \
    }
    EMP_SYS_CONFIGS(EMP_CASE)
#undef EMP_CASE
    emp_set_error("unsupported launch configuration (%d waves per walker)", tu.waves_per_theta);
    return EMP_EINVAL;
}

static int launch_sweep(EmpSystems* p) {
    const int S = p->desc.n_systems;
    p->dev.order = p->tune.order == 0 ? p->d_order_lpt : p->d_order_input;
    for (int st = 0; st < p->desc.nsteps; ++st)
        for (int half = 0; half < 2; ++half) {
            const int nc = (p->desc.ntemps * (p->desc.nwalkers / 2) + SYS_PRIOR_TASKS - 1) / SYS_PRIOR_TASKS;
            const size_t terms = sys_prior_terms(p->max_l), lds = terms * sizeof(double) + p->max_l * sizeof(PseqEntry);
            const int most = systems_per_launch(nc, SYS_PASS);
            for (int s0 = 0; s0 < S; s0 += most) {
                hipLaunchKernelGGL(k_sys_prior, dim3((unsigned)std::min(most, S - s0) * (unsigned)nc), dim3(SYS_PASS), lds,
                                   p->stream, p->dev, s0, half, st, nc, (int)terms);
                EMP_HIP(hipGetLastError());
            }
            if (int rc = launch_lik<false>(p, half, st)) return rc;
        }
    hipLaunchKernelGGL(k_sys_swap, dim3((unsigned)S), dim3(SYS_PASS), 0, p->stream, p->dev);
    EMP_HIP(hipGetLastError());
    return EMP_OK;
}

static int check_tuning(const EmpSystemsTuning& t) {
    if (!(t.waves_per_wg == 8 || t.waves_per_wg == 16) || !(t.waves_per_theta == 1 || t.waves_per_theta == 2)) {
        emp_set_error("waves_per_wg must be 8 or 16 and waves_per_theta 1 or 2");
        return EMP_EINVAL;
    }
    if (t.wgs_per_cu < 1 || t.wgs_per_cu > 4) { emp_set_error("wgs_per_cu must be in [1, 4]"); return EMP_EINVAL; }
    if (t.order != 0 && t.order != 1) { emp_set_error("order must be 0 (longest first) or 1 (input)"); return EMP_EINVAL; }
    return EMP_OK;
}

template <typename T>
static int alloc(EmpSystems* p, T** out, size_t n) {
    void* q = nullptr;
    EMP_HIP(hipMalloc(&q, std::max<size_t>(n, 1) * sizeof(T)));
    p->allocations.push_back(q);
    *out = (T*)q;
    return EMP_OK;
}

template <typename T>
static int upload(EmpSystems* p, const std::vector<T>& v, T** out) {
    int rc = alloc(p, out, v.size());
    if (rc) return rc;
    if (!v.empty()) EMP_HIP(hipMemcpy(*out, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
    return EMP_OK;
}

extern "C" void emp_systems_destroy(EmpSystems* p) {
    if (!p) return;
    if (p->graph_exec) (void)hipGraphExecDestroy(p->graph_exec);
    if (p->stream) (void)hipStreamSynchronize(p->stream);
    for (void* q : p->allocations) (void)hipFree(q);
    if (p->gather_buf) (void)hipFree(p->gather_buf);
    if (p->stream) (void)hipStreamDestroy(p->stream);
    delete p;
}

extern "C" int emp_systems_create(const EmpModelDesc* models, const EmpSystemsDesc* desc, const double* betas,
                                  const double* p0, EmpSystems** out) {
    if (!out) { emp_set_error("null output handle"); return EMP_EINVAL; }
    *out = nullptr;
    if (!models || !desc || !betas || !p0) { emp_set_error("null argument"); return EMP_EINVAL; }
    const EmpSystemsDesc& d = *desc;
    const int S = d.n_systems, T = d.ntemps, W = d.nwalkers;
    if (S < 1) { emp_set_error("n_systems must be >= 1"); return EMP_EINVAL; }
    if (T < 1 || T > 64) { emp_set_error("ntemps must be in [1, 64]"); return EMP_EINVAL; }
    if (W < 2 || W % 2 || W > 1024) { emp_set_error("nwalkers must be even and in [2, 1024]"); return EMP_EINVAL; }
    if (T * (W / 2) > SYS_MAX_TASKS) { emp_set_error("ntemps x nwalkers / 2 must be <= %d", SYS_MAX_TASKS); return EMP_EUNSUP; }
    if (d.nsteps < 1) { emp_set_error("nsteps must be >= 1"); return EMP_EINVAL; }
    if (d.precision != EMP_FP64 && d.precision != EMP_MIXED) { emp_set_error("bad precision"); return EMP_EINVAL; }
    if (!(d.a > 1.0)) { emp_set_error("stretch scale a must be > 1"); return EMP_EINVAL; }
    if (d.adapt_mode < -1 || d.adapt_mode > 2) { emp_set_error("adapt_mode must be -1 (frozen), 0, 1 or 2"); return EMP_EUNSUP; }
    if (d.adapt_mode >= 0 && !(d.adapt_tau > 0 && d.adapt_nu > 0)) { emp_set_error("adapt_tau and adapt_nu must be > 0"); return EMP_EINVAL; }
    if (d.record_every < 0 || d.max_records < 0) { emp_set_error("record_every and max_records must be >= 0"); return EMP_EINVAL; }
    if (d.record_every > 0 && (d.record_temps < 1 || d.record_temps > T)) { emp_set_error("record_temps must be in [1, ntemps]"); return EMP_EINVAL; }
    for (int i = 0; i < S * T; ++i)
        if (!(betas[i] >= 0.0 && betas[i] <= 1.0)) { emp_set_error("betas must lie in [0, 1] (entry %d)", i); return EMP_EINVAL; }

    // Host preparation and packing of every model.
    std::vector<ModelHost> hosts(S);
    size_t nep = 0, npar = 0, nfree = 0, nblk = 0, necc = 0, nseq = 0, nsai = 0, nsaib = 0;
    for (int s = 0; s < S; ++s) {
        int rc = emp_model_host(&models[s], &hosts[s]);
        if (rc) {
            char msg[1024];
            snprintf(msg, sizeof msg, "system %d: %s", s, emp_last_error());
            emp_set_error("%s", msg);
            return rc;
        }
        if (hosts[s].dev.D < 1) { emp_set_error("system %d has no free parameter", s); return EMP_EINVAL; }
        nep += hosts[s].t.size();
        npar += hosts[s].inv.size();
        nfree += hosts[s].free_idx.size();
        nblk += hosts[s].bstart.size();
        necc += hosts[s].ecc.size();
        nseq += hosts[s].pseq.size();
        nsai += hosts[s].sai.size();
        nsaib += hosts[s].sai_base.size();
    }
    EmpSystems* p = new EmpSystems();
    p->desc = d;
    {
        int dev = 0;
        hipDeviceProp_t prop;
        if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess) {
            emp_systems_destroy(p);
            emp_set_error("cannot query the HIP device");
            return EMP_EHIP;
        }
        p->n_cu = prop.multiProcessorCount;
        p->device = dev;
    }
    std::vector<double> t(nep), y(nep), s2(nep), dt(nep), fixed(npar), sai(nsai);
    std::vector<int> ins(nep), inv(npar), fidx(nfree), bst(nblk), pseq(nseq), saib(nsaib);
    std::vector<PseqEntry> pseq_e(nseq);
    std::vector<EmpPriorTerm> pri(npar), ecc(necc);
    std::vector<ModelDev> mds(S);
    std::vector<size_t> o_ep(S), o_par(S), o_free(S), o_blk(S), o_ecc(S), o_seq(S), o_sai(S), o_saib(S);
    p->D.resize(S);
    p->xoff.resize(S);
    p->rxoff.resize(S);
    {
        size_t e = 0, q = 0, f = 0, b = 0, c = 0, g = 0, a = 0, ab = 0;
        int64_t xo = 0, ro = 0;
        for (int s = 0; s < S; ++s) {
            const ModelHost& h = hosts[s];
            o_ep[s] = e; o_par[s] = q; o_free[s] = f; o_blk[s] = b; o_ecc[s] = c; o_seq[s] = g;
            o_sai[s] = a; o_saib[s] = ab;
            std::copy(h.sai.begin(), h.sai.end(), sai.begin() + a);
            std::copy(h.sai_base.begin(), h.sai_base.end(), saib.begin() + ab);
            a += h.sai.size(); ab += h.sai_base.size();
            std::copy(h.t.begin(), h.t.end(), t.begin() + e);
            std::copy(h.y.begin(), h.y.end(), y.begin() + e);
            std::copy(h.s2.begin(), h.s2.end(), s2.begin() + e);
            std::copy(h.dt.begin(), h.dt.end(), dt.begin() + e);
            std::copy(h.ins.begin(), h.ins.end(), ins.begin() + e);
            std::copy(h.inv.begin(), h.inv.end(), inv.begin() + q);
            std::copy(h.fixed.begin(), h.fixed.end(), fixed.begin() + q);
            std::copy(h.prior.begin(), h.prior.end(), pri.begin() + q);
            std::copy(h.free_idx.begin(), h.free_idx.end(), fidx.begin() + f);
            std::copy(h.bstart.begin(), h.bstart.end(), bst.begin() + b);
            std::copy(h.ecc.begin(), h.ecc.end(), ecc.begin() + c);
            std::copy(h.pseq.begin(), h.pseq.end(), pseq.begin() + g);
            std::copy(h.pseq_e.begin(), h.pseq_e.end(), pseq_e.begin() + g);
            e += h.t.size(); q += h.inv.size(); f += h.free_idx.size(); b += h.bstart.size(); c += h.ecc.size();
            g += h.pseq.size();
            p->D[s] = h.dev.D;
            p->xoff[s] = xo;
            p->rxoff[s] = ro;
            xo += (int64_t)T * W * h.dev.D;
            ro += (int64_t)(d.record_every > 0 ? d.record_temps : 0) * W * h.dev.D;
        }
        p->x_total = xo;
        p->dev.rec_x = ro;
    }
    SysDev& v = p->dev;
    v.S = S; v.T = T; v.W = W; v.nsteps = d.nsteps; v.a = d.a;
    v.key0 = (uint32_t)d.seed; v.key1 = (uint32_t)(d.seed >> 32);
    v.adapt_mode = d.adapt_mode; v.adapt_tau = d.adapt_tau; v.adapt_nu = d.adapt_nu;
    v.rec_every = d.record_every; v.rec_temps = d.record_every > 0 ? d.record_temps : 0;
    v.max_rec = d.record_every > 0 ? d.max_records : 0;
    const size_t STW = (size_t)S * T * W;
    int rc = 0;
    double *dt_, *dy, *ds2, *ddt, *dfix, *dsai;
    int *dins, *dinv, *dfidx, *dbst, *dseq, *dsaib;
    EmpPriorTerm *dpri, *decc;
    PseqEntry* dseq_e;
    double2* dtab;
    std::vector<double2> tab;
    emp_sincos_table(tab);
    if ((rc = upload(p, t, &dt_)) || (rc = upload(p, y, &dy)) || (rc = upload(p, s2, &ds2)) ||
        (rc = upload(p, dt, &ddt)) || (rc = upload(p, ins, &dins)) || (rc = upload(p, inv, &dinv)) ||
        (rc = upload(p, fixed, &dfix)) || (rc = upload(p, pri, &dpri)) || (rc = upload(p, fidx, &dfidx)) ||
        (rc = upload(p, bst, &dbst)) || (rc = upload(p, ecc, &decc)) || (rc = upload(p, tab, &dtab)) ||
        (rc = upload(p, pseq, &dseq)) || (rc = upload(p, pseq_e, &dseq_e)) || (rc = upload(p, sai, &dsai)) || (rc = upload(p, saib, &dsaib))) {
        emp_systems_destroy(p);
        return rc;
    }
    for (int s = 0; s < S; ++s) {
        ModelDev m = hosts[s].dev;
        m.t = dt_ + o_ep[s]; m.y = dy + o_ep[s]; m.s2 = ds2 + o_ep[s]; m.dt = ddt + o_ep[s]; m.ins = dins + o_ep[s];
        m.inv_free = dinv + o_par[s]; m.fixed_val = dfix + o_par[s]; m.prior = dpri + o_par[s];
        m.free_idx = dfidx + o_free[s]; m.block_start = dbst + o_blk[s]; m.ecc_prior = decc + o_ecc[s];
        m.sctab = dtab;
        m.pseq = dseq + o_seq[s];
        m.pseq_e = dseq_e + o_seq[s];
        m.sai = dsai + o_sai[s];
        m.sai_base = dsaib + o_saib[s];
        if (!emp_model_dev_complete(m)) {
            emp_systems_destroy(p);
            emp_set_error("system %d: a device array of the model is missing", s);
            return EMP_EINVAL;
        }
        p->ext = p->ext || model_ext(m) > 0;
        p->max_d = std::max(p->max_d, m.Dfull);
        p->max_k = std::max(p->max_k, m.K);
        p->max_l = std::max(p->max_l, m.npseq);
        mds[s] = m;
    }
    // Queue orders: longest first (stable), and the input order.
    std::vector<int> lpt(S), inp(S);
    std::vector<double> cost(S);
    for (int s = 0; s < S; ++s) {
        const ModelDev& m = mds[s];
        cost[s] = (double)m.N * (m.K * 51.0 + 46.0 + (m.ma_active ? 23.0 : 0.0));
        lpt[s] = inp[s] = s;
    }
    std::stable_sort(lpt.begin(), lpt.end(), [&](int a, int b) { return cost[a] > cost[b]; });
    std::vector<int64_t> xoff = p->xoff, rxoff = p->rxoff;
    ModelDev* dmd = nullptr;
    int64_t *dxoff = nullptr, *drxoff = nullptr;
    if ((rc = upload(p, mds, &dmd)) || (rc = upload(p, lpt, &p->d_order_lpt)) || (rc = upload(p, inp, &p->d_order_input)) ||
        (rc = upload(p, xoff, &dxoff)) || (rc = upload(p, rxoff, &drxoff)) ||
        (rc = alloc(p, &v.X, (size_t)p->x_total)) || (rc = alloc(p, &v.lnl, STW)) || (rc = alloc(p, &v.lnp, STW)) ||
        (rc = alloc(p, &v.map, STW)) || (rc = alloc(p, &v.betas, (size_t)S * T)) ||
        (rc = alloc(p, &v.accepted, STW)) || (rc = alloc(p, &v.tsw_sum, (size_t)S * std::max(T - 1, 1))) ||
        (rc = alloc(p, &v.smd_sum, (size_t)S * std::max(T - 1, 1))) || (rc = alloc(p, &v.ctl, 4)) ||
        (rc = alloc(p, &v.tlp, STW / 2)) || (rc = alloc(p, &v.list, STW / 2)) || (rc = alloc(p, &v.nlive, (size_t)2 * S))) {
        emp_systems_destroy(p);
        return rc;
    }
    v.md = dmd; v.xoff = dxoff; v.rxoff = drxoff; v.order = p->d_order_lpt;
    if (v.max_rec > 0) {
        const size_t nw = (size_t)v.rec_temps * W;
        if ((rc = alloc(p, &v.h_x, (size_t)v.max_rec * v.rec_x)) || (rc = alloc(p, &v.h_lnl, (size_t)v.max_rec * S * nw)) ||
            (rc = alloc(p, &v.h_lnp, (size_t)v.max_rec * S * nw))) {
            emp_systems_destroy(p);
            return rc;
        }
    }
#define EMP_TRY(x) do { hipError_t e_ = (x); if (e_ != hipSuccess) { int r_ = emp_hip_fail(e_, #x, __FILE__, __LINE__); emp_systems_destroy(p); return r_; } } while (0)
    EMP_TRY(hipStreamCreateWithFlags(&p->stream, hipStreamNonBlocking));
    EMP_TRY(hipMemcpy(v.X, p0, (size_t)p->x_total * sizeof(double), hipMemcpyHostToDevice));
    EMP_TRY(hipMemcpy(v.betas, betas, (size_t)S * T * sizeof(double), hipMemcpyHostToDevice));
    EMP_TRY(hipMemset(v.accepted, 0, STW * sizeof(long long)));
    EMP_TRY(hipMemset(v.tsw_sum, 0, (size_t)S * std::max(T - 1, 1) * sizeof(double)));
    EMP_TRY(hipMemset(v.smd_sum, 0, (size_t)S * std::max(T - 1, 1) * sizeof(double)));
    EMP_TRY(hipMemset(v.nlive, 0, 2 * (size_t)S * sizeof(int)));
    EMP_TRY(hipMemset(v.ctl, 0, 4 * sizeof(unsigned long long)));
    EMP_TRY(hipDeviceSynchronize());     // the engine stream does not wait for the null stream
#undef EMP_TRY
    // Default launch: 16 walkers per likelihood workgroup, one wave each, longest
    // system first.
    p->tune = EmpSystemsTuning{16, 1, 1, 0, -1.0};
    if ((rc = launch_lik<true>(p, 0, 0))) { emp_systems_destroy(p); return rc; }
    if (hipStreamSynchronize(p->stream) != hipSuccess) {
        rc = emp_hip_fail(hipGetLastError(), "initial evaluation", __FILE__, __LINE__);
        emp_systems_destroy(p);
        return rc;
    }
    *out = p;
    return EMP_OK;
}

static int run_sweeps(EmpSystems* p, int64_t nsweeps, bool use_graph, double* ms_out) {
    hipEvent_t e0, e1;
    EMP_HIP(hipEventCreate(&e0));
    EMP_HIP(hipEventCreate(&e1));
    EMP_HIP(hipEventRecord(e0, p->stream));
    if (use_graph) {
        if (!p->graph_exec) {
            hipGraph_t g;
            EMP_HIP(hipStreamBeginCapture(p->stream, hipStreamCaptureModeThreadLocal));
            int rc = launch_sweep(p);
            hipError_t ce = hipStreamEndCapture(p->stream, &g);
            if (rc) return rc;
            EMP_HIP(ce);
            EMP_HIP(hipGraphInstantiate(&p->graph_exec, g, nullptr, nullptr, 0));
            EMP_HIP(hipGraphDestroy(g));
        }
        for (int64_t s = 0; s < nsweeps; ++s) EMP_HIP(hipGraphLaunch(p->graph_exec, p->stream));
    } else {
        for (int64_t s = 0; s < nsweeps; ++s) {
            int rc = launch_sweep(p);
            if (rc) return rc;
        }
    }
    EMP_HIP(hipEventRecord(e1, p->stream));
    EMP_HIP(hipEventSynchronize(e1));
    float ms = 0.f;
    EMP_HIP(hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (ms_out) *ms_out = nsweeps ? ms / (double)nsweeps : 0.0;
    return EMP_OK;
}

extern "C" int emp_systems_run(EmpSystems* p, int64_t nsweeps, int32_t use_graph) {
    if (!p) { emp_set_error("null engine"); return EMP_EINVAL; }
    if (nsweeps < 0) { emp_set_error("nsweeps must be >= 0"); return EMP_EINVAL; }
    if (emp_fault_injected()) return EMP_EFAULT_INJECTED;
    if (nsweeps == 0) return EMP_OK;
    double ms = 0.0;
    int rc = run_sweeps(p, nsweeps, use_graph != 0, &ms);
    if (rc) return rc;
    p->last_ms = ms;
    return EMP_OK;
}

extern "C" int emp_systems_last_timing(EmpSystems* p, double* ms_per_sweep) {
    if (!p || !ms_per_sweep) { emp_set_error("null argument"); return EMP_EINVAL; }
    *ms_per_sweep = p->last_ms;
    return EMP_OK;
}

extern "C" int emp_systems_set_tuning(EmpSystems* p, const EmpSystemsTuning* t) {
    if (!p || !t) { emp_set_error("null argument"); return EMP_EINVAL; }
    int rc = check_tuning(*t);
    if (rc) return rc;
    EMP_HIP(hipStreamSynchronize(p->stream));
    p->tune = *t;
    if (p->graph_exec) {
        EMP_HIP(hipGraphExecDestroy(p->graph_exec));
        p->graph_exec = nullptr;
    }
    return EMP_OK;
}

extern "C" int emp_systems_get_tuning(EmpSystems* p, EmpSystemsTuning* t) {
    if (!p || !t) { emp_set_error("null argument"); return EMP_EINVAL; }
    *t = p->tune;
    return EMP_OK;
}

// Device-to-device copies of the mutable state, so that autotuning trials
// leave the chains exactly where they were.
struct SysSnapshot {
    std::vector<std::pair<void*, size_t>> items;   // (device buffer, bytes)
    std::vector<void*> copies;
};

static void snap_free(SysSnapshot& sn) {
    for (void* q : sn.copies) (void)hipFree(q);
    sn.copies.clear();
}

static int snap_take(EmpSystems* p, SysSnapshot& sn) {
    const SysDev& v = p->dev;
    const size_t STW = (size_t)v.S * v.T * v.W, ST1 = (size_t)v.S * std::max(v.T - 1, 1);
    sn.items = {{v.X, (size_t)p->x_total * 8}, {v.lnl, STW * 8}, {v.lnp, STW * 8}, {v.map, STW * 4},
                {v.betas, (size_t)v.S * v.T * 8}, {v.accepted, STW * 8}, {v.tsw_sum, ST1 * 8},
                {v.smd_sum, ST1 * 8}, {v.ctl, 4 * 8}};
    for (auto& it : sn.items) {
        void* q = nullptr;
        hipError_t e = hipMalloc(&q, it.second);
        if (e != hipSuccess) { snap_free(sn); return emp_hip_fail(e, "hipMalloc (autotune snapshot)", __FILE__, __LINE__); }
        sn.copies.push_back(q);
        EMP_HIP(hipMemcpyAsync(q, it.first, it.second, hipMemcpyDeviceToDevice, p->stream));
    }
    EMP_HIP(hipStreamSynchronize(p->stream));
    return EMP_OK;
}

static int snap_restore(EmpSystems* p, const SysSnapshot& sn) {
    for (size_t i = 0; i < sn.items.size(); ++i)
        EMP_HIP(hipMemcpyAsync(sn.items[i].first, sn.copies[i], sn.items[i].second, hipMemcpyDeviceToDevice, p->stream));
    EMP_HIP(hipStreamSynchronize(p->stream));
    return EMP_OK;
}

extern "C" int emp_systems_autotune(EmpSystems* p, int32_t trial_sweeps, EmpSystemsTuning* best_out) {
    if (!p) { emp_set_error("null engine"); return EMP_EINVAL; }
    if (trial_sweeps < 1) { emp_set_error("trial_sweeps must be >= 1"); return EMP_EINVAL; }
    SysSnapshot sn;
    int rc = snap_take(p, sn);
    if (rc) return rc;
    const EmpSystemsTuning keep = p->tune;
    EmpSystemsTuning best = keep;
    best.ms_per_sweep = -1.0;
    const int nws[2] = {16, 8}, wps[2] = {1, 2};
    for (int order = 0; order < 2 && !rc; ++order)
        for (int a = 0; a < 2 && !rc; ++a)
            for (int b = 0; b < 2 && !rc; ++b) {
                EmpSystemsTuning c{nws[a], wps[b], 1, order, -1.0};
                p->tune = c;
                double ms = 0.0;
                if ((rc = run_sweeps(p, 1, false, nullptr)) || (rc = run_sweeps(p, trial_sweeps, false, &ms)) ||
                    (rc = snap_restore(p, sn)))
                    break;
                c.ms_per_sweep = ms;
                if (best.ms_per_sweep < 0 || ms < best.ms_per_sweep) best = c;
            }
    const int rc2 = snap_restore(p, sn);
    snap_free(sn);
    if (rc) { p->tune = keep; return rc; }
    if (rc2) return rc2;
    if (best.ms_per_sweep < 0) { emp_set_error("no launch configuration fits"); p->tune = keep; return EMP_EUNSUP; }
    p->tune = best;
    if (p->graph_exec) {
        EMP_HIP(hipGraphExecDestroy(p->graph_exec));
        p->graph_exec = nullptr;
    }
    if (best_out) *best_out = best;
    return EMP_OK;
}

// The current state of systems [s0, s1) in position order (gathered through the
// maps on the device).
static int gather_systems(EmpSystems* p, int s0, int s1, int what, double* out) {
    const SysDev& v = p->dev;
    const int TW = v.T * v.W;
    if (what != EMP_PT_STATE_X)
        return emp_gather_rows(p->device, (what == EMP_PT_STATE_LNL ? v.lnl : v.lnp) + (size_t)s0 * TW, v.map + (size_t)s0 * TW,
                               (long long)(s1 - s0) * TW, TW, 1, &p->gather_buf, &p->gather_cap, p->stream, out);
    for (int s = s0; s < s1; ++s) {
        const int rc = emp_gather_rows(p->device, v.X + p->xoff[s], v.map + (size_t)s * TW, TW, TW, p->D[s], &p->gather_buf,
                                       &p->gather_cap, p->stream, out);
        if (rc) return rc;
        out += (size_t)TW * p->D[s];
    }
    return EMP_OK;
}

extern "C" int emp_systems_get(EmpSystems* p, int32_t what, int32_t system, void* host_out, int64_t cap,
                               int64_t* shape) {
    if (!p || !host_out) { emp_set_error("null argument"); return EMP_EINVAL; }
    const SysDev& v = p->dev;
    const int S = v.S, T = v.T, W = v.W;
    if (system < -1 || system >= S) { emp_set_error("system %d out of range [-1, %d)", system, S); return EMP_EINVAL; }
    EMP_HIP(hipStreamSynchronize(p->stream));
    unsigned long long ctl[4];
    EMP_HIP(hipMemcpy(ctl, v.ctl, sizeof ctl, hipMemcpyDeviceToHost));
    const long long sweeps = (long long)ctl[2];
    const long long R = v.rec_every > 0 ? std::min<long long>(sweeps / v.rec_every, v.max_rec) : 0;
    const int s0 = system < 0 ? 0 : system, s1 = system < 0 ? S : system + 1, ns = s1 - s0;
    const size_t TW = (size_t)T * W, nw = (size_t)v.rec_temps * W;
    int64_t sh[4] = {1, 1, 1, 1};
    size_t n = 0, elem = 8;
    auto need = [&](size_t count) -> bool {
        if ((int64_t)(count * elem) > cap) {
            emp_set_error("output buffer too small (%zu bytes needed)", count * elem);
            return false;
        }
        return true;
    };
    switch (what) {
        case EMP_PT_NSWEEPS: {
            sh[0] = 2; elem = 8; n = 2;
            if (!need(n)) return EMP_EINVAL;
            long long o[2] = {(long long)ctl[2], (long long)ctl[3]};
            memcpy(host_out, o, sizeof o);
            break;
        }
        case EMP_PT_STATE_X: {
            n = 0;
            for (int s = s0; s < s1; ++s) n += TW * p->D[s];
            if (system >= 0) { sh[0] = T; sh[1] = W; sh[2] = p->D[system]; } else { sh[0] = (int64_t)n; }
            if (!need(n)) return EMP_EINVAL;
            if (int rc = gather_systems(p, s0, s1, what, (double*)host_out)) return rc;
            break;
        }
        case EMP_PT_STATE_LNL:
        case EMP_PT_STATE_LNP: {
            n = (size_t)ns * TW;
            if (system >= 0) { sh[0] = T; sh[1] = W; } else { sh[0] = S; sh[1] = T; sh[2] = W; }
            if (!need(n)) return EMP_EINVAL;
            if (int rc = gather_systems(p, s0, s1, what, (double*)host_out)) return rc;
            break;
        }
        case EMP_PT_ACCEPTED:
        case EMP_PT_STATE_BETAS: {
            const bool acc = what == EMP_PT_ACCEPTED;
            const size_t per = acc ? TW : (size_t)T;
            n = (size_t)ns * per;
            if (system >= 0) { sh[0] = T; if (acc) sh[1] = W; }
            else { sh[0] = S; sh[1] = T; if (acc) sh[2] = W; }
            if (!need(n)) return EMP_EINVAL;
            const void* src = acc ? (const void*)(v.accepted + s0 * per) : (const void*)(v.betas + s0 * per);
            EMP_HIP(hipMemcpy(host_out, src, n * 8, hipMemcpyDeviceToHost));
            break;
        }
        case EMP_PT_TSW:
        case EMP_PT_SMD: {
            const size_t per = (size_t)std::max(T - 1, 0);
            n = (size_t)ns * per;
            if (system >= 0) { sh[0] = (int64_t)per; } else { sh[0] = S; sh[1] = (int64_t)per; }
            if (!need(n)) return EMP_EINVAL;
            if (n) {
                EMP_HIP(hipMemcpy(host_out, (what == EMP_PT_TSW ? v.tsw_sum : v.smd_sum) + s0 * per, n * 8,
                                  hipMemcpyDeviceToHost));
                double* o = (double*)host_out;
                for (size_t i = 0; i < n; ++i) o[i] = sweeps > 0 ? o[i] / (double)sweeps : 0.0;
            }
            break;
        }
        case EMP_PT_CHAIN: {
            if (system < 0) { emp_set_error("the recorded chain is returned one system at a time"); return EMP_EINVAL; }
            if (!v.max_rec) goto norec;
            const size_t per = nw * p->D[system];
            n = (size_t)R * per;
            sh[0] = R; sh[1] = v.rec_temps; sh[2] = W; sh[3] = p->D[system];
            if (!need(n)) return EMP_EINVAL;
            for (long long r = 0; r < R; ++r)
                EMP_HIP(hipMemcpy((double*)host_out + r * per, v.h_x + r * v.rec_x + p->rxoff[system], per * 8,
                                  hipMemcpyDeviceToHost));
            break;
        }
        case EMP_PT_LNL:
        case EMP_PT_LNP: {
            if (!v.max_rec) goto norec;
            const double* src = what == EMP_PT_LNL ? v.h_lnl : v.h_lnp;
            n = (size_t)R * ns * nw;
            if (system >= 0) { sh[0] = R; sh[1] = v.rec_temps; sh[2] = W; }
            else { sh[0] = R; sh[1] = S; sh[2] = v.rec_temps; sh[3] = W; }
            if (!need(n)) return EMP_EINVAL;
            for (long long r = 0; r < R; ++r)
                EMP_HIP(hipMemcpy((double*)host_out + (size_t)r * ns * nw, src + ((size_t)r * S + s0) * nw,
                                  (size_t)ns * nw * 8, hipMemcpyDeviceToHost));
            break;
        }
        default:
            emp_set_error("unknown quantity %d", what);
            return EMP_EINVAL;
    }
    if (shape) for (int i = 0; i < 4; ++i) shape[i] = sh[i];
    return EMP_OK;
norec:
    emp_set_error("nothing was recorded (record_every == 0 or max_records == 0)");
    return EMP_EINVAL;
}

// pict_krylov.hpp -- what the Krylov solver kernels share (pict_solve.hip, pict_cgblock.hip): the
// solver arguments and states, exchange between workgroups, FP64 reductions, the CG scalar step.
#pragma once

#include <hip/hip_runtime.h>

#include "pict_host.hpp"
#include "pict_solver.hpp"

namespace pict {

constexpr int kSolveThreads = 256;
constexpr int kSlots = 8;              // FP64 partial slots per right-hand side
constexpr unsigned kSpinLimit = 1u << 23;
constexpr int kMaxRhs = 4;

// Control block, one 128-byte line per hot word (device memory, zeroed before launch).
struct Ctl {
    unsigned count;              // top-level arrivals (one per group)
    unsigned pad0[31];
    unsigned gen;                // barrier generation
    unsigned pad1[31];
    int err;                     // a wait exceeded its spin limit
    int zero_all;                // k_cg: every right-hand side is zero; k_cg_block, k_bicg_block: not solved there
    int admit;                   // k_cg_block, k_bicg_block: kAdmit*
    unsigned pad2[29];
    unsigned group_count[32][32];  // per-group arrivals (a line per group)
};
// Resident workgroups (256 threads) per compute unit that a persistent solver grid is sized for.  Grids of seven
// and eight per unit (1792 and 2048 workgroups: the 1.77 M-row channel pressure system on the lean grid-wide CG
// and on the textbook CG) ended at the barrier's spin limit.  They sat exactly at the occupancy query's maximum,
// which SGPRs set for those kernels (102-106 per wave: 7 waves per SIMD), while grids at a VGPR-set maximum run;
// the counters and the spin budget do not depend on the grid size.  Four per unit stays below the SGPR limit of
// every solver kernel; kernels whose VGPRs allow fewer take the query's figure.
constexpr int kMaxResidentWgsPerCu = 4;
constexpr int kGroups = 8;       // arrival tree fan-in (one group per XCD when blocks are dealt round-robin)

// Loads and stores that one workgroup uses to exchange data with another: agent-scope atomic
// operations (sc1 on gfx950), coherent across the XCDs' L2 caches without L2 writeback or
// invalidation.
template <typename T>
__device__ __forceinline__ void st_coh(T *p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ T ld_coh(const T *p) {
    return __hip_atomic_load(const_cast<T *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// wait until every memory operation this thread issued has completed
__device__ __forceinline__ void ops_done() {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

struct RhsState {
    double rho, rho_prev, alpha, omega, beta;
    double best_crit, last_crit;
    int active, converged, finite, used;
    int best_it, rising, save_best, restore_best;
    double final_res;
    int on_chip;  // k_cg_block or k_bicg_block solved it (filled in with the caller's copy)
    int pad;
};

template <typename R>
struct SolveArgs {
    const int32_t *row, *col, *perm;  // perm != nullptr: use A^T (value of (j,i) for entry (i,j))
    const R *val;
    const R *b;
    R *x;
    R *r, *rhat, *p0, *p1, *v0, *v1, *s, *t, *best;  // each [nrhs*n]
    double *partials;                              // partial_doubles(nwg) (grid-wide kernels)
    Ctl *ctl;
    RhsState *st;                                  // [nrhs]
    int n, nrhs, maxit, conv, reset_steps, return_best, zero_shortcut;
    double tol;
    unsigned nwg;
    double crit_scale;                             // criterion factor: 1/sqrt(n) (NORM2_NORMALIZED), 1/n (ABS_MEAN), 1
    unsigned long long *tagged;                    // tagged partials [2][nwg][kSlots], zeroed (k_cg_local packs its
                                                   // NS values per workgroup: [2][nwg][NS])
    void *pub;                                     // k_cg_local: published rows r, w, s [3][2][n], zeroed
    int block_rpt;                                 // k_cg_block_jobs: rows per thread of a system on several workgroups
    int salt;                                      // k_cg_local, k_cg_block: stamp of this launch's foreign-read marks
    unsigned admit;                                // k_cg_block, k_bicg_block: polls of the first totals before the grid
                                                   // declines (block_admit; 0: it does); kAdmitAlways: resident by
                                                   // its launch
    unsigned spin;                                 // k_cg_block, k_bicg_block: polls of every later wait
    const int *gate;                               // non-null: the solve is left alone when *gate is 0 (a kernel queued
                                                   // behind k_cg_block or k_bicg_block for what those cannot hold)
};

// The arguments of a system from a table in memory.  A pointer read from memory has no known address space, and an
// access through it is a flat one, which waits for the LDS counter too; read as a pointer to global memory, it compiles
// to the same loads as a kernel's own pointer arguments.
template <typename T>
__device__ __forceinline__ T *load_global_ptr(T *const *p) {
    return (T *)*reinterpret_cast<__attribute__((address_space(1))) T *const *>(p);
}
template <typename R>
__device__ __forceinline__ SolveArgs<R> job_args(const SolveArgs<R> *args, unsigned job) {
    const SolveArgs<R> &in = args[job >> 16];
    SolveArgs<R> a = in;
#define PICT_GLOBAL(f) a.f = load_global_ptr(&in.f)
    PICT_GLOBAL(row), PICT_GLOBAL(col), PICT_GLOBAL(val), PICT_GLOBAL(b), PICT_GLOBAL(x);
    PICT_GLOBAL(r), PICT_GLOBAL(rhat), PICT_GLOBAL(p0), PICT_GLOBAL(p1), PICT_GLOBAL(v0), PICT_GLOBAL(v1);
    PICT_GLOBAL(s), PICT_GLOBAL(t), PICT_GLOBAL(best), PICT_GLOBAL(partials), PICT_GLOBAL(ctl), PICT_GLOBAL(st);
    PICT_GLOBAL(tagged), PICT_GLOBAL(gate);
#undef PICT_GLOBAL
    a.pub = load_global_ptr(reinterpret_cast<char *const *>(&in.pub));
    a.perm = nullptr;  // batched solves are not transposed
    return a;
}

// Admission of a block kernel's grid.  Its workgroups wait for each other, so all of them have to be resident, and an
// ordinary launch does not promise that: two such grids on concurrent streams (or in two processes) can each hold a part
// of the compute units.  Nothing is written before the first totals, whose wait therefore decides: workgroup 0 admits the
// grid once it has seen the partial sums of all workgroups, any workgroup whose wait runs out declines it, whichever
// comes first holds for all (one word), and a grid that declines leaves the system to the general kernel queued behind
// it.  A grid that is admitted is resident as a whole and always ends, so waiting for one is safe too.
// The limit, kAdmitPolls, is some 8 ms of polling: longer than most solves that hold the compute units, short against
// the general kernel's solve of a system this size.  Deciding costs one trip through memory per solve (1 us).
enum { kAdmitOpen = 0, kAdmitGo = 1, kAdmitDecline = 2 };
constexpr unsigned kAdmitPolls = 1u << 12;
constexpr unsigned kAdmitAlways = ~0u;
// between two polls of a wait that has been long
__device__ __forceinline__ void wait_long(unsigned spins) {
    if (spins > 64) __builtin_amdgcn_s_sleep(32);
}
// The grid's decision, by one wave (the same in all its lanes); all_posted: this wave has seen every partial sum.
__device__ __forceinline__ bool block_admit(Ctl *ctl, unsigned bid, bool all_posted) {
    int d = kAdmitOpen;
    if ((threadIdx.x & 63) == 0) {
        if (all_posted && bid != 0) {  // workgroup 0 is resident and decides
            for (unsigned spins = 0; spins < kSpinLimit && (d = ld_coh(&ctl->admit)) == kAdmitOpen; ++spins)
                wait_long(spins);
        }
        if (d == kAdmitOpen) {
            const int mine = all_posted && bid == 0 ? kAdmitGo : kAdmitDecline;
            if (__hip_atomic_compare_exchange_strong(&ctl->admit, &d, mine, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT)) {
                d = mine;
                if (mine == kAdmitDecline) st_coh(&ctl->zero_all, 1);
            }
        }
    }
    return __builtin_amdgcn_readfirstlane(d) == kAdmitGo;
}

// slot layout of the partial sums (per workgroup and right-hand side)
enum { S_RR = 0, S_ASUM = 1, S_AMAX = 2, S_D0 = 3, S_D1 = 4, S_BMAX = 5 };


// Wave64 reductions in DPP (quad and row rotations within 16-lane rows, then the
// four row totals in a fixed order): every lane of the wave gets the same total,
// and the result depends only on the inputs, so every workgroup reducing the same
// values gets bitwise the same result.
template <int CTRL>
__device__ __forceinline__ double dpp_d(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double lane_d(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}
template <bool MAX>
__device__ __forceinline__ double wave_reduce_dpp(double v) {
    auto op = [](double x, double y) { return MAX ? fmax(x, y) : x + y; };
    v = op(v, dpp_d<0xB1>(v));   // quad_perm [1,0,3,2]
    v = op(v, dpp_d<0x4E>(v));   // quad_perm [2,3,0,1]
    v = op(v, dpp_d<0x124>(v));  // row_ror:4
    v = op(v, dpp_d<0x128>(v));  // row_ror:8
    return op(op(lane_d(v, 0), lane_d(v, 16)), op(lane_d(v, 32), lane_d(v, 48)));
}
// first reduction of a solve: rho = (r0, r0); zero-RHS shortcut flag in omega
__device__ __forceinline__ void cg1_init(RhsState &st, double rr, int zero_all) {
    st.rho = rr;
    st.alpha = 0;
    st.beta = 0;
    st.omega = zero_all;
    st.active = zero_all ? 0 : 1;
    st.converged = zero_all;
    st.finite = 1;
    st.used = -1;
    st.final_res = 0;
    st.best_crit = 0;
    st.last_crit = 0;
    st.best_it = -1;
    st.rising = 0;
    st.save_best = 0;
    st.restore_best = 0;
}
typedef unsigned long long u64;
// A slot is rewritten every second generation, so a stale slot is exactly two generations
// old: (generation + 1) mod 4 tells them apart, and the zeroed start (tag 0) is not awaited
// before every slot has been written once.
__device__ __forceinline__ u64 tag_partial(double v, unsigned gen) {
    return (__double_as_longlong(v) & ~3ull) | (u64)((gen + 1u) & 3u);
}
__device__ __forceinline__ bool partial_ready(u64 u, unsigned gen) { return (unsigned)(u & 3u) == ((gen + 1u) & 3u); }
__device__ __forceinline__ double partial_value(u64 u) { return __longlong_as_double((long long)(u & ~3ull)); }

// Partial sums as k_cg_block and k_bicg_block post them: whole, a word that is not posted yet is 0 (+0 travels as -0,
// which adds the same).  The sets of words rotate, and a set is used again only after its owner has cleared its words.
// CG: with its post of generation g a workgroup clears its words of set g + 2 (every workgroup has posted g - 1, so all
// have read g - 2, the same set), and it waits for both stores before it polls, so before its post of g + 1, without
// which nobody reads set g + 2.  BiCGStab's other reductions lie between two of a kind, so that two sets do; the words
// are cleared behind the totals.
// That wait, for all stores of a wave before it begins to poll, is also the faster way: polls that begin while stores
// are under way slow them (CG per iteration with it and without: 256 x 256 1.8 and 2.5 us, 57 x 35 x 30 2.0 and 3.0,
// 131 x 67 x 45 3.1 and 5.1).
// A set begins on a line of its own, so that clearing one touches no line of another that is being polled.
constexpr int kCgSets = 4;
__host__ __device__ constexpr unsigned post_stride(unsigned words) { return (words + 15u) & ~15u; }
__device__ __forceinline__ u64 post_word(double v) {
    const u64 u = (u64)__double_as_longlong(v);
    return u ? u : 1ull << 63;
}
__device__ __forceinline__ double post_value(u64 u) { return __longlong_as_double((long long)u); }

// Published row values of one vector: [2][n] (parity), FP32 as (value, tag) words.
template <typename R>
struct Pub;
template <>
struct Pub<float> {
    u64 *base;
    int n;
    __device__ __forceinline__ void put(int par, int i, float v, unsigned tag) const {
        st_coh(base + (size_t)par * n + i, ((u64)tag << 32) | (u64)__float_as_uint(v));
    }
    // value of row c (parity par) once it carries `tag`; NaN after a bounded wait
    __device__ __forceinline__ float get(int par, int c, unsigned tag, int &err) const {
        if (err) return __int_as_float(0x7fc00000);
        const u64 *p = base + (size_t)par * n + c;
        u64 u = ld_coh(p);
        unsigned spins = 0;
        while ((unsigned)(u >> 32) != tag) {
            if (++spins > kSpinLimit) {
                err = 1;
                return __int_as_float(0x7fc00000);
            }
            u = ld_coh(p);
        }
        return __uint_as_float((unsigned)u);
    }
    // raw word of row c (one load, no wait), then its value and whether it carries `tag`
    using Word = u64;
    __device__ __forceinline__ u64 word(int par, int c) const { return ld_coh(base + (size_t)par * n + c); }
    static __device__ __forceinline__ float open(u64 u, unsigned tag, bool &ok) {
        ok = ok & ((unsigned)(u >> 32) == tag);
        return __uint_as_float((unsigned)u);
    }
    static constexpr bool kTagged = true;
};
template <>
struct Pub<double> {
    double *base;
    int n;
    __device__ __forceinline__ void put(int par, int i, double v, unsigned) const {
        st_coh(base + (size_t)par * n + i, v);
    }
    __device__ __forceinline__ double get(int par, int c, unsigned, int &) const {
        return ld_coh(base + (size_t)par * n + c);
    }
    using Word = double;
    __device__ __forceinline__ double word(int par, int c) const { return ld_coh(base + (size_t)par * n + c); }
    static __device__ __forceinline__ double open(double u, unsigned, bool &) { return u; }
    static constexpr bool kTagged = false;
};
// Reduction layouts of k_cg_local (slot ids and whether a slot is a maximum), as types so
// that every use folds to constants.  With a norm-2 criterion only (r,r) and (w,r) (and
// max|b| in the first pass) are needed; the sum and the maximum of |r| only for the
// absolute criteria.
struct CgFirstFull {
    static constexpr int NS = 4;
    static constexpr int ID[4] = {S_RR, S_ASUM, S_AMAX, S_BMAX};
    static constexpr bool MAX[4] = {false, false, true, true};
};
struct CgIterFull {
    static constexpr int NS = 4;
    static constexpr int ID[4] = {S_RR, S_ASUM, S_AMAX, S_D0};
    static constexpr bool MAX[4] = {false, false, true, false};
};
struct CgFirst {
    static constexpr int NS = 2;
    static constexpr int ID[2] = {S_RR, S_BMAX};
    static constexpr bool MAX[2] = {false, true};
};
struct CgIter {
    static constexpr int NS = 2;
    static constexpr int ID[2] = {S_RR, S_D0};
    static constexpr bool MAX[2] = {false, false};
};
template <bool FULL>
struct CgSlots {
    using First = CgFirstFull;
    using Iter = CgIterFull;
};
template <>
struct CgSlots<false> {
    using First = CgFirst;
    using Iter = CgIter;
};
// 1/d to about one ulp: the hardware estimate and two Newton steps
__device__ __forceinline__ double rcp64(double d) {
    double y = __builtin_amdgcn_rcp(d);
    double e = fma(-d, y, 1.0);
    y = fma(y, e, y);
    e = fma(-d, y, 1.0);
    return fma(y, e, y);
}

// a / d from y = 1 / d to about an ulp: the quotient's remainder corrects it (Markstein 1990), rounded as a division's
__device__ __forceinline__ double div64(double a, double d, double y) {
    const double q = a * y;
    return fma(fma(-d, q, a), y, q);
}

// Solver state of k_cg_local's iterations, held by every lane of wave 0 (all lanes compute the
// same values from the same totals).
struct CgRun {
    double rho, inv_rho, den, alpha, beta;  // alpha = rho / den
    double best_crit, last_crit, final_res;
    int active, converged, finite, used, best_it, rising, save_best, restore_best;
};

// cg1_update in the form k_cg_local runs it: the same tests (convergence cg_solver_kernel.cu:306-313,
// best result :330-346), and the next step from
//   beta' = gamma' / rho,  delta' - beta' gamma' / alpha = delta' - beta'^2 den,  alpha' = gamma' / that,
// equal to cg1_update's alpha' and beta' in exact arithmetic.  The candidates are formed before the
// tests, so one reciprocal (not three dependent divisions) lies on the path to the next iteration.
template <bool FULL, typename R>
__device__ __forceinline__ void cg_run_update(const SolveArgs<R> &a, CgRun &st, const double (&t)[kSlots], int it) {
    const double gam = t[S_RR];
    const double beta_n = gam * st.inv_rho;
    const double den_n = fma(-beta_n * beta_n, st.den, t[S_D0]);
    const double alpha_n = gam * rcp64(den_n);
    const double inv_rho_n = rcp64(gam);
    double crit = sqrt(gam) * a.crit_scale;
    if constexpr (FULL)
        crit = (a.conv == PICT_CONV_NORM2 || a.conv == PICT_CONV_NORM2_NORMALIZED) ? crit
               : a.conv == PICT_CONV_ABS_MAX                                      ? t[S_AMAX]
                                                                                  : t[S_ASUM] * a.crit_scale;
    st.save_best = 0;
    if (!isfinite(crit)) {
        st.converged = 0; st.used = it; st.final_res = crit; st.finite = 0; st.active = 0;
        return;
    }
    if (a.return_best) {
        if (it == 0 || crit < st.best_crit) { st.best_crit = crit; st.best_it = it; st.save_best = 1; }
        if (it > 0 && crit >= st.last_crit) ++st.rising; else st.rising = 0;
        st.last_crit = crit;
    }
    st.used = it;
    st.final_res = crit;
    if (crit < a.tol) { st.converged = 1; st.finite = 1; st.active = 0; return; }
    if (a.return_best && (it == a.maxit - 1 || st.rising >= 100)) {
        st.restore_best = st.best_it != it;
        st.converged = 0; st.used = st.best_it; st.final_res = st.best_crit; st.finite = 1;
        st.active = 0;
        return;
    }
    st.alpha = alpha_n;
    st.beta = beta_n;
    st.den = den_n;
    st.rho = gam;
    st.inv_rho = inv_rho_n;
}

// k_cg_block instances (kernel null: none): the whole system on one workgroup; `rpt` rows per thread on several.
// Rows of up to nz entries.
struct BlockKernel {
    const void *kernel;
    int threads, rpt;
};
BlockKernel cg_block_one(bool f32, int nz, long long n);
BlockKernel cg_block_many(bool f32, int nz, int rpt);
// batched launch: systems of up to kBlockJobsOne rows on one workgroup, larger ones SolveArgs::block_rpt rows per thread
// on several (those for which block_jobs_has holds)
constexpr int kBlockJobsOne = 2048;
BlockKernel cg_block_jobs(bool f32, int nz);
constexpr bool block_jobs_has(bool f32, int nz, int rpt) {
    return rpt == 2 || (rpt == 4 && (f32 || nz <= 5)) || (rpt == 8 && f32 && nz <= 5);
}
// k_bicg_block instances: `together` right-hand sides advance at once (nrhs or 1)
struct BicgBlock {
    BlockKernel k;
    int together;
};
constexpr int kBicgSums = 9;   // sums of its largest reduction
constexpr int kBicgSets = 10;  // posted: one set per group of right-hand sides, then [3 reductions][2]; each [kBicgSums][post_stride(workgroups)]
BicgBlock bicg_block(bool f32, int nz, int rpt, int nrhs);

}  // namespace pict

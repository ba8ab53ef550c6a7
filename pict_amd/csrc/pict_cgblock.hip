// pict_cgblock.hip -- single-reduction CG with a system's whole state on chip, one large workgroup per
// compute unit (one right-hand side, norm-2 criteria, rows of at most 7 entries).
//
// The recurrences of k_cg1 / k_cg_local (pict_solve.hip: Chronopoulos & Gear 1989, the iterates of
// cgSolveGPU, cg_solver_kernel.cu:114-456).  A workgroup of 512 threads owns up to 512*RPT rows; the
// matrix entries, w and s of a thread's rows stay in its registers, r in LDS (x and p in registers, in
// LDS and memory for the largest instances), so an iteration reads no matrix and no vector from memory.
//
// Other workgroups' rows ("halo").  A product needs r' of rows that another workgroup owns.  r' follows
// from r, s and w by two fmas, so a reader keeps its own copy of the halo rows' r (LDS) and s (registers),
// advances them with the owner's fma sequence (bitwise the owner's values), and only w travels: one word
// per halo row and iteration, as agent-scope atomics that need no L2 writeback or invalidation.  FP32
// words carry their iteration, so a reader waits on the data itself while the reduction is under way; FP64
// words cannot, so there a workgroup waits for its stores before it posts its partial sums.
// Halo rows are found in the first pass: every foreign column marks its tile of 8 rows in a bitmap (LDS),
// a scan numbers the marked tiles, and a row's register entry is the LDS offset of the column.
//
// Rows of a workgroup.  Rows in order for 5-entry (2-D) systems.  For 7-entry (3-D) systems a contiguous
// chunk would have most of its neighbours a plane away in other workgroups (192x96x96 on 256 workgroups:
// 14,200 halo rows for 6,912 own rows), so the grid's line length and plane are read off the matrix (the
// column offsets -d3, -d2, -1, 0, 1, d2, d3 of an interior row) and a workgroup owns a block of whole
// lines (6 x 6 lines: 4,608 halo rows).  Lines of which two are more than the halo holds (2-D: 448 to 890 cells,
// 3-D: some 300) are cut into strips first (BlockMap).  The mapping is a bijection of the rows whatever the
// matrix is: a wrong guess costs halo rows, never correctness.
//
// What bounds it: an iteration is one trip of the partial sums through memory (about 1.3 us between the XCDs for up to
// 128 workgroups, 2 for 256), three workgroup barriers, and per row 0.25 us of LDS gathers and FP64 sums on a unit that
// holds 14 of them per thread.  At 192 x 96 x 96 it takes 7.3 us where streaming the system takes 40 (184 MB at 4.6
// TB/s); figures for other sizes stand at plan_block (pict_solve.hip).
//
// A system of several workgroups that this kernel cannot hold (a longer row, too many halo rows, no block
// partition) is left alone, and so is any system while the grid does not become resident as a whole (block_admit): the
// kernel sets ctl->zero_all ("not solved") before it writes x, and the general kernel queued behind it runs; otherwise
// that kernel returns at once.
#include <hip/hip_runtime.h>

#include <cmath>

#include "pict_block.hpp"

namespace pict {

// Totals of one generation over the workgroups' posted pairs (lane l: workgroups l, l + 64, ... in that
// order, then across the lanes): the same bits in every workgroup.  At most 256 workgroups; B of a lane's in flight.
// False after `limit` polls, or once the grid has declined (admit, may be null).
template <int B>
__device__ __forceinline__ bool block_poll(const u64 *part, unsigned nwg, unsigned gen, bool max1, unsigned limit,
                                           const int *admit, double &t0, double &t1) {
    const unsigned lane = threadIdx.x & 63;
    const u64 *set = part + (size_t)((gen & (kCgSets - 1)) * post_stride(2 * nwg));
    double v0, v1;
    unsigned spins = 0;
    for (;;) {
        bool ready = true;
        v0 = v1 = 0.0;
#pragma unroll
        for (int b = 0; b < 4; b += B) {
            if (64u * b >= nwg) continue;
            u64 u[B][2];
#pragma unroll
            for (int j = 0; j < B; ++j) {
                if (64u * (b + j) >= nwg) continue;
                const unsigned w = lane + 64u * (b + j);
                const u64 *p = set + (size_t)(w < nwg ? w : 0u) * 2;
                u[j][0] = ld_coh(p);
                u[j][1] = ld_coh(p + 1);
            }
#pragma unroll
            for (int j = 0; j < B; ++j) {
                if (lane + 64u * (b + j) >= nwg) continue;
                ready = ready & (u[j][0] != 0) & (u[j][1] != 0);
                v0 += post_value(u[j][0]);
                const double q = post_value(u[j][1]);
                v1 = max1 ? fmax(v1, q) : v1 + q;
            }
        }
        if (__all(ready)) break;
        if (++spins > limit) return false;
        if (admit) {
            if (ld_coh(admit) == kAdmitDecline) return false;
            wait_long(spins);
        }
    }
    if (max1) {
        t0 = wave_reduce_dpp<false>(v0);
        t1 = wave_reduce_dpp<true>(v1);
    } else {
        const double v = wave_sum2(v0, v1);
        t0 = lane_d(v, 0);
        t1 = lane_d(v, 32);
    }
    return true;
}

// The scalar step of cg_run_update (pict_krylov.hpp) for the norm-2 criteria without best-result bookkeeping; the
// criterion's square root is taken only near the tolerance and at the end (final_res: block_run_end).
// FP64 systems take quotients as rounded as a division's (DIV); of FP32 systems the coefficients are rounded to FP32
// afterwards, and on one workgroup every wave forms them (rcp64, as in k_cg_local: 1.27 instead of 1.34 us, 75 x 54).
template <bool DIV, typename R>
__device__ __forceinline__ void block_run_update(const SolveArgs<R> &a, CgRun &st, double gam, double delta, int it) {
    const double beta_n = DIV ? div64(gam, st.rho, st.inv_rho) : gam * st.inv_rho;
    const double den_n = fma(-beta_n * beta_n, st.den, delta);
    st.used = it;
    const double near = gam * (a.crit_scale * a.crit_scale);
    if (!(near > 1.0001 * a.tol * a.tol) || !(near < 1e300)) {
        const double crit = sqrt(gam) * a.crit_scale;
        const bool finite = isfinite(crit);
        if (!finite || crit < a.tol) {
            st.converged = st.finite = finite;
            st.final_res = crit;
            st.active = 0;
            return;
        }
    }
    st.alpha = DIV ? div64(gam, den_n, rcp64(den_n)) : gam * rcp64(den_n);
    st.beta = beta_n;
    st.den = den_n;
    st.rho = gam;
    st.inv_rho = rcp64(gam);
}
template <typename R>
__device__ __forceinline__ void block_run_end(const SolveArgs<R> &a, CgRun &st) {
    if (st.active && st.used >= 0) st.final_res = sqrt(st.rho) * a.crit_scale;  // the iteration limit
}

// ONE: the system fits one workgroup: no exchange, no halo, and every thread runs the scalar step on the
// wave totals (two workgroup barriers per iteration instead of three and no trip through memory).
// HPT: halo rows per thread of waves 1..
// BIG: more rows per thread than the registers hold vectors of: p, s and the halo's s in LDS, and x in memory (4 bytes
// per row each way, while the workgroup waits for the totals).
template <typename R, int T, int RPT, int NZ, int HPT, bool BIG, bool ONE>
__device__ __forceinline__ void cg_block(const SolveArgs<R> &a, unsigned bid) {
    constexpr int kBW = T / 64;
    constexpr int kBF = T - 64;  // threads that hold halo rows: waves 1.. (wave 0 polls the reduction)
    constexpr int C = T * RPT;
    constexpr int H = ONE ? 0 : kBF * HPT;
    constexpr int LR = ONE ? C : C + (H > C / 2 ? H : C / 2);  // also the set-up's bitmap and tile numbers
    constexpr int NO = NZ - 1, NI = (NO + 1) / 2;
    constexpr bool kTagged = Pub<R>::kTagged;
    static_assert((C + H) * sizeof(R) <= 65536, "LDS offsets are 16 bits");
    __shared__ R lr[LR];  // r of the own rows, then of the halo rows
    // BIG: p, s, then s and the fetched w of the halo rows, then w of WL rows per thread
    constexpr int WL = BIG ? 4 : 0;
    __shared__ R lps[BIG ? 2 * C + 2 * H + WL * T : 1];
    __shared__ int ltile[ONE ? 1 : H / kTile + 1];  // halo tile: position of its first row / kTile
    __shared__ double wsum[2][2 * kBW];  // by generation parity: the waves' first sums, then their second
    __shared__ PlaceLds place;
    __shared__ BlockMap smap;
    __shared__ int s_over, s_err, s_declined;
    struct Step {
        double alpha, beta;
        int active;
    };
    __shared__ Step bc;
    // the wave number as a scalar: a wave takes its branch alone, without the other branch's waits
    const int t = (int)threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    if (t == 0) s_over = s_err = s_declined = 0;
    int *mark = reinterpret_cast<int *>(a.p0);  // tiles that another workgroup reads (stamped with a.salt)
    int nh = 0;                                 // halo rows (a multiple of kTile)
    if constexpr (ONE) {
        if (t == 0) smap = whole_map(a.n);
        __syncthreads();
    } else {
        nh = block_place<T, C, H, RPT, NZ>(a.row, a.col, a.n, (int)a.nwg, bid, smap, reinterpret_cast<unsigned *>(lr),
                                           ltile, place, s_over, mark, a.salt);
        if (nh < 0) return;
    }
    // (large instances leave the map in LDS: in scalar registers it spills those of the iterations, 8.5 instead of 7.4 us)
    const std::conditional_t<BIG, const BlockMap &, const BlockMap> m = pick_map<BIG>(smap);
    const unsigned nwg = (unsigned)m.nwg;
    const unsigned first = bid * (unsigned)C;  // position of the first own row
    using PubT = decltype(Pub<R>::base);
    const Pub<R> pub{reinterpret_cast<PubT>(a.pub), (int)(a.nwg * (unsigned)C)};  // w by position, two parities
    auto put_row = [&](int par, unsigned pos, R v, unsigned tag) {
        PubT base = pub.base + (size_t)par * pub.n;
        if constexpr (kTagged) st_coh(elem(base, pos), ((u64)tag << 32) | (u64)__float_as_uint(v));
        else st_coh(elem(base, pos), v);
    };

    // ---- rows into registers; r0 = b - A x0 ----
    R dv[RPT], val[RPT][NO], w[RPT], s[BIG ? 1 : RPT], x[BIG ? 1 : RPT], p[BIG ? 1 : RPT];
    unsigned idx[RPT][NI];
    unsigned longm = 0;  // bit q: row q is read from memory (ONE)
    double acc0 = 0.0, acc1 = 0.0;
    // (in two parts: in one, the largest instance's loop is more than the compiler unrolls)
    auto load_rows = [&](auto from) __attribute__((always_inline)) {
        constexpr int Q0 = decltype(from)::value, Q1 = Q0 + 7 < RPT ? Q0 + 7 : RPT;
        const BlockMap m = uniform_map(smap);
#pragma unroll
        for (int q = Q0; q < Q1; ++q) {
            const int li = t + q * T;
            const int i = block_row<C, NZ>(m, bid, (unsigned)li);
            const int ii = i < 0 ? 0 : i;
            const int rs = *elem(a.row, ii);
            int len = i < 0 ? 0 : *elem(a.row, ii + 1) - rs;
            if constexpr (ONE) {
                // a row of more entries than the registers hold is read from memory in every product
                bool diag = false;
                for (int e = 0; len >= NZ && e < NZ; ++e) diag |= a.col[rs + e] == ii;
                if (len > NO + (diag ? 1 : 0)) {
                    longm |= 1u << q;
                    len = 0;
                }
            }
            const R x0 = i < 0 ? R(0) : *elem(a.x, ii), bv = i < 0 ? R(0) : *elem(a.b, ii);
            R sum = 0;
            block_load_row<C, H, NZ, ONE, BIG>(a, m, ii, li, first, rs, len, reinterpret_cast<const unsigned *>(lr), dv[q],
                                               val[q], idx[q], [&](R v, int c) { sum += v * *elem(a.x, c); });
            if constexpr (ONE)
                if (longm >> q & 1u)
                    for (int e = rs; e < a.row[ii + 1]; ++e) sum += a.val[a.perm ? a.perm[e] : e] * a.x[a.col[e]];
            const R rv = bv - sum;
            w[q] = rv;  // until the bitmap in lr has been read
            if constexpr (BIG) {
                lps[li] = lps[C + li] = R(0);
            } else {
                x[q] = x0;
                p[q] = s[q] = R(0);
            }
            if constexpr (!ONE) put_row(1, first + li, rv, 1u);  // every row: the marks are not known yet
            acc0 += (double)rv * (double)rv;
            acc1 = fmax(acc1, fabs((double)bv));
            // a row is finished before the next one is begun (else the unrolled rows' loads and index arithmetic overlap
            // and spill)
#pragma unroll
            for (int j = 0; j < NI; ++j) asm volatile("" : "+v"(idx[q][j]));
#pragma unroll
            for (int j = 0; j < NO; ++j) asm volatile("" : "+v"(val[q][j]));
            asm volatile("" : "+v"(dv[q]), "+v"(w[q])::"memory");
            if constexpr (RPT >= 8) __builtin_amdgcn_sched_barrier(0);
        }
    };
    load_rows(std::integral_constant<int, 0>{});
    if constexpr (RPT > 7) load_rows(std::integral_constant<int, 7>{});
    if constexpr (!ONE)
        if (s_over) acc1 = INFINITY;
    __syncthreads();  // the bitmap has been read
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
        lr[t + q * T] = w[q];
        w[q] = R(0);  // (rows in LDS: written by the first product before they are read)
    }

    // the workgroup's totals from the waves' (lane l takes entry l, then across the lanes)
    auto wg_totals = [&](int par, bool max1, double &g0, double &g1) {
        double v = wsum[par][lane & (2 * kBW - 1)];
        const bool mx = max1 && (lane & kBW);
        auto op = [&](double x, double y) { return mx ? fmax(x, y) : x + y; };
        v = op(v, dpp_d<0xB1>(v));  // quad_perm [1,0,3,2]
        v = op(v, dpp_d<0x4E>(v));  // quad_perm [2,3,0,1]
        if constexpr (kBW == 8) {
            v = op(v, dpp_d<0x141>(v));  // row_half_mirror
        } else {
            static_assert(kBW == 8 || kBW == 16, "8 or 16 waves");
            v = op(v, dpp_d<0x124>(v));  // row_ror:4
            v = op(v, dpp_d<0x128>(v));  // row_ror:8
        }
        g0 = lane_d(v, 0);
        g1 = lane_d(v, kBW);
    };

    // Reduce-barrier: the totals of acc0 (sum) and acc1 (sum; of the first reduction maximum).  ONE: in every thread; else in
    // wave 0, with `mid` run by waves 1.. once the workgroup's partials are out.  False in wave 0 (else
    // ignored) when a wait ran out.
    auto reduce = [&](auto first_one, unsigned gen, double &t0, double &t1, auto mid) -> bool {
        constexpr bool max1 = decltype(first_one)::value;
        // before the partials: the halo marks, which their owners read once after the first totals, and FP64 rows (FP32
        // rows carry their iteration)
        if constexpr (!ONE)
            if (!kTagged || max1) ops_done();
        const int par = (int)(gen & 1u);
        if (max1) {
            const double w0 = wave_reduce_dpp<false>(acc0), w1 = wave_reduce_dpp<true>(acc1);
            if (lane == 0) {
                wsum[par][wave] = w0;
                wsum[par][kBW + wave] = w1;
            }
        } else {
            const double w = wave_sum2(acc0, acc1);
            if ((lane & 31) == 0) wsum[par][(lane >> 5) * kBW + wave] = w;
        }
        __syncthreads();
        bool ok = true;
        if constexpr (ONE) {
            wg_totals(par, max1, t0, t1);
        } else if (wave == 0) {
            double g0, g1;
            wg_totals(par, max1, g0, g1);
            auto slot = [&](unsigned g) {
                return a.tagged + (size_t)((g & (kCgSets - 1)) * post_stride(2 * nwg) + 2 * bid + (unsigned)lane);
            };
            if (lane < 2) st_coh(slot(gen), post_word(lane ? g1 : g0));
            if (lane < 2) st_coh(slot(gen + 2u), (u64)0);
            ops_done();
            auto poll = [&](unsigned limit, const int *admit) {
                return block_poll<BIG ? 2 : 4>(a.tagged, nwg, gen, max1, limit, admit, t0, t1);
            };
            if (max1 && a.admit != kAdmitAlways) {
                ok = a.admit > 0 && poll(a.admit, &a.ctl->admit);
                const bool go = block_admit(a.ctl, bid, ok);
                if (lane == 0) s_declined = !go;
                // admitted by workgroup 0 while this wait ran out: everything is posted
                if (go && !ok) ok = poll(a.spin, nullptr);
            } else {
                ok = poll(a.spin, nullptr);
            }
        } else {
            mid();
        }
        return ok;
    };
    // scalar state: every thread's (ONE), every lane's of wave 0, or thread 0's in LDS (large instances: registers)
    constexpr bool kRunLds = !ONE && RPT >= 8;
    __shared__ CgRun srun;
    CgRun run;
    auto fail = [&] {
        st_coh(&a.ctl->err, 1);
        s_err = 1;
    };

    double t0 = 0.0, t1 = 0.0;
    unsigned pubm = 0;  // bit q: the wave publishes its rows q (the same in all its lanes)
    // ---- first totals: (r0, r0), max|b| (infinite: some workgroup cannot hold its rows) ----
    {
        const bool ok = reduce(std::true_type{}, 0u, t0, t1, [] {});
        if constexpr (ONE) {
            if (t == 0) bc = Step{t0, t1, 1};
        } else if (t == 0) {
            if (!ok && !s_declined) fail();
            bc = Step{t0, t1, 1};
        }
        __syncthreads();
        if (s_err || s_declined) return;
        t0 = bc.alpha;
        t1 = bc.beta;
        if constexpr (!ONE) {
            if (isinf(t1)) {
                if (bid == 0 && t == 0) a.ctl->zero_all = 1;  // not solved here
                return;
            }
        }
        if (a.zero_shortcut && t1 == 0.0) {
            for (int q = 0; q < RPT; ++q) {
                const int i = block_row<C, NZ>(m, bid, (unsigned)(t + q * T));
                if (i >= 0) a.x[i] = R(0);
            }
            if (bid == 0 && t == 0) cg1_init(a.st[0], t0, 1);
            return;
        }
    }
    // halo slots of this thread
    const int h0 = t - 64;
    // BIG: x lies in memory (read and written by its thread of waves 1.. while wave 0 waits for the totals)
    R *xw = reinterpret_cast<R *>(a.pub) + (size_t)a.nwg * C * (2 * sizeof(typename Pub<R>::Word) / sizeof(R)) + first;
    if constexpr (BIG) {
        for (int k = h0; k < C && wave > 0; k += kBF) {
            const int i = block_row<C, NZ>(m, bid, (unsigned)k);
            xw[k] = i < 0 ? R(0) : a.x[i];
        }
    }
    R hv[ONE || BIG ? 1 : HPT];           // the halo rows' published values (BIG: in LDS)
    R hs[ONE || BIG ? 1 : HPT];           // their s
    // position of halo row k of this thread; rows the thread does not have repeat its first one (or position 0)
    const bool any_halo = h0 >= 0 && h0 < nh;
    auto halo_pos = [&](int k) {
        return any_halo ? (unsigned)(ltile[h0 / kTile + k * (kBF / kTile)] * kTile + h0 % kTile) : 0u;
    };
    static_assert(kBF % kTile == 0, "a thread's halo rows have the same place in their tiles");
    constexpr bool kPosReg = !ONE && RPT < 8;
    unsigned hpos[kPosReg ? HPT : 1];
    if constexpr (kPosReg) {
#pragma unroll
        for (int k = 0; k < HPT; ++k) hpos[k] = halo_pos(k);
    }
    // FP32: load until every halo word carries `tag` (bounded: the workgroup then ends at its next barrier, so that no
    // other wait is begun); FP64: one load
    auto fetch_halo = [&](int par, unsigned tag) {
        if constexpr (!ONE) {
            // BIG: half of the words at a time (registers)
            constexpr int HB = BIG ? HPT / 2 : HPT;
            static_assert(HPT % HB == 0, "whole batches");
#pragma unroll
            for (int b = 0; b < HPT; b += HB) {
                unsigned spins = 0;
                for (;;) {
                    typename Pub<R>::Word u[HB];
#pragma unroll
                    for (int k = 0; k < HB; ++k)
                        u[k] = ld_coh(elem(pub.base + (size_t)par * pub.n, kPosReg ? hpos[kPosReg ? b + k : 0] : halo_pos(b + k)));
                    unsigned stale = 0;
#pragma unroll
                    for (int k = 0; k < HB; ++k) {
                        bool mine = true;
                        const R got = Pub<R>::open(u[k], tag, mine);
                        if constexpr (BIG) lps[2 * C + H + h0 + (b + k) * kBF] = got;
                        else hv[b + k] = got;
                        stale |= mine ? 0u : 1u;
                    }
                    if (!__any(any_halo && stale)) break;
                    if (++spins > a.spin) {
                        if (lane == 0) fail();
                        break;
                    }
                }
            }
        }
    };
    auto prefetch_halo = [&](int par, unsigned tag) {
        if constexpr (kTagged) fetch_halo(par, tag);
    };
    // w = A r of the own rows (r of the halo rows in LDS), published with `tag`; (r, r) and (r, w)
    auto product = [&](int par, unsigned tag) {
        unsigned at = first + (unsigned)t;
        if constexpr (RPT >= 8) asm volatile("" : "+v"(at));
#pragma unroll
        for (int q = 0; q < RPT; ++q) {
            const int li = t + q * T;
            const R rv = lr[li];
            R wv = 0;
            // large instances: the indices stay packed (hoisted out of the iterations, their unpacked form spills)
            if constexpr (RPT >= 8) {
#pragma unroll
                for (int j = 0; j < NI; ++j) asm volatile("" : "+v"(idx[q][j]));
            }
#pragma unroll
            for (int j = 0; j < NO; ++j) {
                if (j == NO / 2) wv += dv[q] * rv;
                const unsigned off = j & 1 ? idx[q][j / 2] >> 16 : idx[q][j / 2] & 0xffffu;
                wv += val[q][j] * *reinterpret_cast<const R *>(reinterpret_cast<const char *>(lr) + off);
            }
            if constexpr (ONE)
                if (longm >> q & 1u)
                    for (int e = a.row[li]; e < a.row[li + 1]; ++e)
                        wv += a.val[a.perm ? a.perm[e] : e] * lr[a.col[e]];
            if (q < WL) lps[BIG ? 2 * C + 2 * H + li : 0] = wv;
            else w[q] = wv;
            if constexpr (!ONE)
                if (pubm >> q & 1u) {
                    R out = wv;
                    if constexpr (RPT >= 8) asm volatile("" : "+v"(out));  // a copy: w is not tied to the word's registers
                    put_row(par, at + q * T, out, tag);
                }
            acc0 += (double)rv * (double)rv;
            acc1 += (double)wv * (double)rv;
            if constexpr (RPT >= 8)
                if (q % 2 == 1) __builtin_amdgcn_sched_barrier(0);  // bounds the loads in flight (registers)
        }
    };
    if constexpr (!ONE) {
#pragma unroll
        for (int q = 0; q < RPT; ++q)
            if (__any(ld_coh(mark + (first + (unsigned)(t + q * T)) / kTile) == a.salt)) pubm |= 1u << q;
        pubm = (unsigned)__builtin_amdgcn_readfirstlane((int)pubm);
        if (wave > 0) {
            fetch_halo(1, 1u);
#pragma unroll
            for (int k = 0; k < HPT; ++k) {
                const int h = h0 + k * kBF;
                lr[C + h] = BIG ? lps[BIG ? 2 * C + H + h : 0] : hv[BIG ? 0 : k];
                if constexpr (BIG) lps[2 * C + h] = R(0);
                else hs[k] = R(0);
            }
        }
        __syncthreads();
    }
    // ---- w = A r; gamma = (r, r), delta = (w, r); alpha = gamma / delta ----
    acc0 = acc1 = 0.0;
    product(0, 2u);
    {
        double g0, g1 = 0.0;
        const bool ok = reduce(std::false_type{}, 1u, g0, g1, [&] { prefetch_halo(0, 2u); });
        auto start = [&](CgRun &r) {
            r.rho = g0;
            r.den = g1;
            r.alpha = g0 / g1;
            r.beta = 0.0;
            r.inv_rho = 1.0 / g0;
            r.final_res = 0.0;
            r.active = r.finite = 1;
            r.converged = 0;
            r.used = -1;
        };
        if constexpr (!kRunLds)
            if (ONE || wave == 0) start(run);
        if constexpr (!ONE) {
            if (t == 0) {
                if (!ok) fail();
                if constexpr (kRunLds) start(srun);
                bc = Step{g0 / g1, 0.0, 1};
            }
            __syncthreads();
            if (s_err) return;
        }
    }
    Step cs;
    if constexpr (ONE) cs = Step{run.alpha, run.beta, run.active};
    else cs = bc;
    for (int it = 0; it < a.maxit && cs.active; ++it) {
        const R alpha = (R)cs.alpha, beta = (R)cs.beta;
        acc0 = acc1 = 0.0;
        // halo rows: the owner's s and r (FP64: w is loaded once the generation that published it is complete)
        if constexpr (!ONE) {
            if (wave > 0) {
                if constexpr (!kTagged) fetch_halo(it & 1, 0u);
#pragma unroll
                for (int k = 0; k < HPT; ++k) {
                    const int h = h0 + k * kBF;
                    R sh = BIG ? lps[BIG ? 2 * C + h : 0] : hs[BIG ? 0 : k];
                    sh = fma(beta, sh, BIG ? lps[BIG ? 2 * C + H + h : 0] : hv[BIG ? 0 : k]);
                    if constexpr (BIG) lps[2 * C + h] = sh;
                    else hs[k] = sh;
                    lr[C + h] = fma(-alpha, sh, lr[C + h]);
                }
            }
        }
        // own rows: p, s, x, r
#pragma unroll
        for (int q = 0; q < RPT; ++q) {
            const int li = t + q * T;
            const R rv = lr[li];
            R sm;
            if constexpr (BIG) {
                lps[li] = fma(beta, lps[li], rv);
                sm = fma(beta, lps[C + li], q < WL ? lps[2 * C + 2 * H + li] : w[q]);
                lps[C + li] = sm;
            } else {
                const R pm = fma(beta, p[q], rv);
                p[q] = pm;
                x[q] = fma(alpha, pm, x[q]);
                sm = fma(beta, s[q], w[q]);
                s[q] = sm;
            }
            const R rm = fma(-alpha, sm, rv);
            lr[li] = rm;
            if constexpr (RPT >= 8)
                if (q % 2 == 1) __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
        product((it + 1) & 1, (unsigned)it + 3u);
        double gam = 0.0, delta = 0.0;
        const bool ok = reduce(std::false_type{}, (unsigned)it + 2u, gam, delta, [&] {
            if constexpr (BIG) {
                constexpr int XB = 4;  // rows of x in flight per thread
                static_assert(!BIG || C % (XB * kBF) == 0, "whole batches");
                for (int k = h0; k < C; k += XB * kBF) {
                    R xv[XB];
#pragma unroll
                    for (int j = 0; j < XB; ++j) xv[j] = *elem(xw, k + j * kBF);
#pragma unroll
                    for (int j = 0; j < XB; ++j) *elem(xw, k + j * kBF) = fma(alpha, lps[k + j * kBF], xv[j]);
                }
            }
            prefetch_halo((it + 1) & 1, (unsigned)it + 3u);
        });
        if constexpr (ONE) {
            block_run_update<false>(a, run, gam, delta, it);
            cs = Step{run.alpha, run.beta, run.active};
        } else {
            if (wave == 0) {
                if (!ok) {
                    if (t == 0) fail();
                } else if constexpr (kRunLds) {
                    if (t == 0) {
                        block_run_update<sizeof(R) == 8>(a, srun, gam, delta, it);
                        bc = Step{srun.alpha, srun.beta, srun.active};
                    }
                } else {
                    block_run_update<sizeof(R) == 8>(a, run, gam, delta, it);
                    if (t == 0) bc = Step{run.alpha, run.beta, run.active};
                }
            }
            __syncthreads();
            if (s_err) return;
            cs = bc;
        }
    }
    if constexpr (BIG) {
        for (int k = h0; k < C && wave > 0; k += kBF) {
            const int i = block_row<C, NZ>(m, bid, (unsigned)k);
            if (i >= 0) a.x[i] = xw[k];
        }
    }
#pragma unroll
    for (int q = 0; q < (BIG ? 0 : RPT); ++q) {
        const int li = t + q * T;
        const int i = block_row<C, NZ>(m, bid, (unsigned)li);
        if (i < 0) continue;
        a.x[i] = x[q];
    }
    if (bid == 0 && t == 0) {
        auto finish = [&](CgRun &r) {
            block_run_end(a, r);
            RhsState st;
            cg1_init(st, r.rho, 0);
            st.alpha = r.alpha;
            st.beta = r.beta;
            st.final_res = r.final_res;
            st.active = r.active;
            st.converged = r.converged;
            st.finite = r.finite;
            st.used = r.used;
            a.st[0] = st;
        };
        if constexpr (kRunLds) finish(srun);
        else finish(run);
    }
}

template <typename R, int T, int RPT, int NZ, int HPT, bool BIG, bool ONE>
__global__ __launch_bounds__(T) void k_cg_block(SolveArgs<R> a) {
    cg_block<R, T, RPT, NZ, HPT, BIG, ONE>(a, blockIdx.x);
}

// Batched launch (job lists as for k_cg_local_jobs): systems of up to 2048 rows run the one-workgroup instance that
// they would run alone, larger ones as many rows per thread as the batch's plan gave them.
template <typename R, int NZ>
__global__ __launch_bounds__(512) void k_cg_block_jobs(const SolveArgs<R> *__restrict__ args,
                                                       const unsigned *__restrict__ job_off,
                                                       const unsigned *__restrict__ jobs) {
    constexpr int H2 = NZ <= 5 ? 2 : 4, H4 = NZ <= 5 ? 3 : 6;
    constexpr bool f32 = sizeof(R) == 4;
    const unsigned j0 = job_off[blockIdx.x], j1 = job_off[blockIdx.x + 1];
    for (unsigned j = j0; j < j1; ++j) {
        const unsigned job = (unsigned)__builtin_amdgcn_readfirstlane((int)jobs[j]), bid = job & 0xffffu;
        const SolveArgs<R> a = job_args(args, job);
        if (a.n <= 512) cg_block<R, 512, 1, NZ, 1, false, true>(a, 0);
        else if (a.n <= 1024) cg_block<R, 512, 2, NZ, 1, false, true>(a, 0);
        else if (a.n <= kBlockJobsOne) cg_block<R, 512, 4, NZ, 1, false, true>(a, 0);
        else if (a.block_rpt == 2) cg_block<R, 512, 2, NZ, H2, false, false>(a, bid);
        else if (a.block_rpt == 4) {
            if constexpr (block_jobs_has(f32, NZ, 4)) cg_block<R, 512, 4, NZ, H4, false, false>(a, bid);
        } else {
            if constexpr (block_jobs_has(f32, NZ, 8)) cg_block<R, 512, 8, NZ, 4, false, false>(a, bid);
        }
        __syncthreads();
    }
}

// Instances.  One workgroup: up to 512 threads x 4 rows, FP32 1024 x 4; several: 512 threads.
template <typename R, int NZ>
static BlockKernel one_kernel(long long n) {
    constexpr bool f32 = sizeof(R) == 4;
    if (n <= 512) return {(const void *)k_cg_block<R, 512, 1, NZ, 1, false, true>, 512, 1};
    if (n <= 1024) return {(const void *)k_cg_block<R, 512, 2, NZ, 1, false, true>, 512, 2};
    if (n <= 2048) return {(const void *)k_cg_block<R, 512, 4, NZ, 1, false, true>, 512, 4};
    if constexpr (f32) {
        if (n <= 4096) return {(const void *)k_cg_block<R, 1024, 4, NZ, 1, false, true>, 1024, 4};
    }
    return {nullptr, 0, 0};
}
template <typename R, int NZ>
static BlockKernel many_kernel(int rpt) {
    if constexpr (NZ <= 5) {
        switch (rpt) {
            case 1:
                if constexpr (sizeof(R) == 4) return {(const void *)k_cg_block<R, 512, 1, 5, 2, false, false>, 512, 1};
                return {nullptr, 0, 0};
            case 2: return {(const void *)k_cg_block<R, 512, 2, 5, 2, false, false>, 512, 2};
            case 4: return {(const void *)k_cg_block<R, 512, 4, 5, 3, false, false>, 512, 4};
            case 8:
                if constexpr (sizeof(R) == 4) return {(const void *)k_cg_block<R, 512, 8, 5, 4, false, false>, 512, 8};
                return {nullptr, 0, 0};
            default: return {nullptr, 0, 0};
        }
    } else {
        switch (rpt) {
            case 1: return {(const void *)k_cg_block<R, 512, 1, 7, 3, false, false>, 512, 1};
            case 2: return {(const void *)k_cg_block<R, 512, 2, 7, 4, false, false>, 512, 2};
            case 4: return {(const void *)k_cg_block<R, 512, 4, 7, 6, false, false>, 512, 4};
            case 8:
                if constexpr (sizeof(R) == 4) return {(const void *)k_cg_block<R, 512, 8, 7, 9, false, false>, 512, 8};
                return {nullptr, 0, 0};
            case 14:
                if constexpr (sizeof(R) == 4) return {(const void *)k_cg_block<R, 512, 14, 7, 12, true, false>, 512, 14};
                return {nullptr, 0, 0};
            default: return {nullptr, 0, 0};
        }
    }
}

BlockKernel cg_block_one(bool f32, int nz, long long n) {
    return f32 ? (nz <= 5 ? one_kernel<float, 5>(n) : one_kernel<float, 7>(n))
               : (nz <= 5 ? one_kernel<double, 5>(n) : one_kernel<double, 7>(n));
}
BlockKernel cg_block_jobs(bool f32, int nz) {
    return {f32 ? (nz <= 5 ? (const void *)k_cg_block_jobs<float, 5> : (const void *)k_cg_block_jobs<float, 7>)
                : (nz <= 5 ? (const void *)k_cg_block_jobs<double, 5> : (const void *)k_cg_block_jobs<double, 7>),
            512, 0};
}
BlockKernel cg_block_many(bool f32, int nz, int rpt) {
    return f32 ? (nz <= 5 ? many_kernel<float, 5>(rpt) : many_kernel<float, 7>(rpt))
               : (nz <= 5 ? many_kernel<double, 5>(rpt) : many_kernel<double, 7>(rpt));
}

}  // namespace pict

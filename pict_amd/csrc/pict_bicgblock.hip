// pict_bicgblock.hip -- BiCGStab with a system's whole state on chip, one workgroup of 512 threads per compute unit
// (norm-2 criteria, rows of at most 7 entries).
//
// The iteration of k_bicgstab (pict_solve.hip; bicgstabSolveGPU, bicgstab_solver_kernel.cu:222-365) with the placement
// of k_cg_block (pict_block.hpp): matrix entries, v and t of a thread's rows in registers, r / s and p in LDS (x and
// the shadow residual in registers, of the largest instance in memory and v in LDS), so an iteration reads no matrix.
//
// Halo.  The products need p and s of rows that other workgroups own.  Both follow from r, p, v and t by the owner's
// fmas, so a reader keeps its own copies (r / s and p in LDS, v in registers), and only v and t travel, each once per
// iteration and row, while the workgroup waits for the reduction that follows the product which made it.  FP32 words
// carry a number of their iteration and a reader waits on the word; FP64 words cannot, so there a workgroup waits for
// its stores before it posts its partial sums and reads once the totals are there.
//
// Buffers are single: a reader has v(it) (t(it)) before it contributes to the reduction after the next product (after
// the update), and the owner writes the next one behind that reduction.  The last t of a group of right-hand sides may
// still be awaited when its owner is at the next group, whose r travels in its own region for that.
//
// Right-hand sides.  NR of them advance together (three reductions per iteration for all); where registers and LDS do
// not hold that many, NR is 1 and they follow one another on the matrix loaded once.
//
// Reductions.  Up to 3 NR sums: wave w totals, posts and polls sum w, every thread then forms the coefficients from the
// totals in LDS (the same bits in every workgroup).
//
// What bounds it: three trips of the partial sums through memory per iteration (1.3 us each between the XCDs for up to
// 128 workgroups, 2 for 256) and, with 14 rows per thread, two products of 3.5 us.  Figures stand at plan_bicg_block
// (pict_solve.hip).
//
// A system that the kernel cannot hold, or whose grid does not become resident, is left to the general kernel, as in
// k_cg_block.
#include <hip/hip_runtime.h>

#include <cmath>

#include "pict_block.hpp"

namespace pict {

// reductions: a group's first, then three per iteration
enum { kRedFirst, kRedA, kRedB, kRedC };
// set of posted partial sums of a reduction's generation (kBicgSets)
__device__ __forceinline__ unsigned bicg_set(int red, unsigned gen) {
    return red == kRedFirst ? gen : (unsigned)(kMaxRhs + 2 * (red - kRedA)) + (gen & 1u);
}
static_assert(kBicgSets == kMaxRhs + 6, "sets of posted sums");

// a wave-uniform value, held in scalar registers
__device__ __forceinline__ double uniform_d(double v) { return lane_d(v, 0); }

template <typename R, int RPT, int NZ, int HPT, int NR, bool BIG>
__global__ __launch_bounds__(512) void k_bicg_block(SolveArgs<R> a) {
    constexpr int T = 512, kBW = T / 64;
    constexpr int kBF = T - 64;  // threads that hold halo rows: waves 1..
    constexpr int C = T * RPT, H = kBF * HPT, L = C + H;
    constexpr int LR = C + (H > C / 2 ? H : C / 2);  // also the set-up's bitmap and tile numbers
    constexpr int NO = NZ - 1, NI = NO / 2;
    constexpr bool kTagged = Pub<R>::kTagged;
    constexpr int kSums = kBicgSums;
    static_assert(L * sizeof(R) <= 65536, "LDS offsets are 16 bits");
    static_assert(3 * NR <= kSums && (!BIG || NR == 1), "sums of a reduction");
    __shared__ R lr[NR][LR];           // r, then s of the iteration: own rows, halo rows
    __shared__ R lp[NR][L];            // p
    __shared__ R lv[BIG ? L : 1];      // BIG: v
    __shared__ int ltile[H / kTile];   // halo tile: position of its first row / kTile
    __shared__ double wsum[kSums][kBW], tot[kSums];
    __shared__ PlaceLds place;
    __shared__ BlockMap smap;
    __shared__ int s_over, s_err, s_late, s_go;
    const unsigned bid = blockIdx.x;
    const int t = (int)threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    if (t == 0) s_over = s_err = s_late = 0;
    int *mark = reinterpret_cast<int *>(a.p0);  // tiles that another workgroup reads (stamped with a.salt)
    const int nh = block_place<T, C, H, RPT, NZ>(a.row, a.col, a.n, (int)a.nwg, bid, smap,
                                                 reinterpret_cast<unsigned *>(&lr[0][0]), ltile, place, s_over, mark, a.salt);
    if (nh < 0) return;
    const BlockMap m = uniform_map(smap);
    const unsigned nwg = (unsigned)m.nwg;
    const unsigned first = bid * (unsigned)C;  // position of the first own row
    const size_t npos = (size_t)a.nwg * C;
    // v and t by position, [vector][right-hand side of the group]; the groups' first residuals (also the shadow
    // residuals); BIG: x of the group
    using Word = typename Pub<R>::Word;
    Word *words = reinterpret_cast<Word *>(a.pub);
    R *rh = reinterpret_cast<R *>(words + 2 * NR * npos);
    R *xw = rh + NR * npos + first;
    auto put_row = [&](int vec, int k, unsigned pos, R v, unsigned tag) {
        Word *base = words + (size_t)(vec * NR + k) * npos;
        if constexpr (kTagged) st_coh(elem(base, pos), ((u64)tag << 32) | (u64)__float_as_uint(v));
        else st_coh(elem(base, pos), v);
    };

    // ---- rows into registers ----
    R dv[RPT], val[RPT][NO];
    unsigned idx[RPT][NI];
    // (in two parts: in one, the largest instance's loop is more than the compiler unrolls)
    auto load_rows = [&](auto from) __attribute__((always_inline)) {
        constexpr int Q0 = decltype(from)::value, Q1 = Q0 + 7 < RPT ? Q0 + 7 : RPT;
#pragma unroll
        for (int q = Q0; q < Q1; ++q) {
            const int li = t + q * T;
            const int i = block_row<C, NZ>(m, bid, (unsigned)li);
            const int ii = i < 0 ? 0 : i;
            const int rs = *elem(a.row, ii);
            const int len = i < 0 ? 0 : *elem(a.row, ii + 1) - rs;
            block_load_row<C, H, NZ, false, BIG>(a, m, ii, li, first, rs, len,
                                                 reinterpret_cast<const unsigned *>(&lr[0][0]), dv[q], val[q], idx[q],
                                                 [](R, int) {});
            // a row is finished before the next one is begun (else the unrolled rows' loads overlap and spill)
#pragma unroll
            for (int j = 0; j < NI; ++j) asm volatile("" : "+v"(idx[q][j]));
#pragma unroll
            for (int j = 0; j < NO; ++j) asm volatile("" : "+v"(val[q][j]));
            asm volatile("" : "+v"(dv[q])::"memory");
            if constexpr (RPT >= 8) __builtin_amdgcn_sched_barrier(0);
        }
    };
    load_rows(std::integral_constant<int, 0>{});
    if constexpr (RPT > 7) load_rows(std::integral_constant<int, 7>{});
    __syncthreads();  // the bitmap has been read

    // A z of own row q, z in `z` (own, then halo rows)
    auto product = [&](const R *z, int q) {
        if constexpr (RPT >= 8) {
            // the indices stay packed (hoisted out of the iterations, their unpacked form spills)
#pragma unroll
            for (int j = 0; j < NI; ++j) asm volatile("" : "+v"(idx[q][j]));
        }
        R y = 0;
#pragma unroll
        for (int j = 0; j < NO; ++j) {
            if (j == NO / 2) y += dv[q] * z[t + q * T];
            const unsigned off = j & 1 ? idx[q][j / 2] >> 16 : idx[q][j / 2] & 0xffffu;
            y += val[q][j] * *reinterpret_cast<const R *>(reinterpret_cast<const char *>(z) + off);
        }
        return y;
    };
    // bounds the loads in flight (registers)
    auto fence = [](int q) {
        if constexpr (RPT >= 8)
            if (q % 2 == 1) __builtin_amdgcn_sched_barrier(0);
    };

    // Reduce-barrier: the totals of acc[0..S) over all workgroups in tot, sum S - 1 a maximum if MAXLAST.  `mid` is run
    // by waves 1.. once their partials are out.  False in every thread when a wait ran out, or the grid declined.
    auto reduce = [&](int red, unsigned gen, auto maxlast, auto &acc, auto mid) -> bool {
        constexpr int S = (int)(sizeof(acc) / sizeof(acc[0]));
        constexpr bool MAXLAST = decltype(maxlast)::value;
        if (!kTagged || red == kRedFirst) ops_done();  // published rows before the partials
        constexpr int NS = MAXLAST ? S - 1 : S;
#pragma unroll
        for (int s = 0; s + 1 < NS; s += 2) {
            const double w = wave_sum2(acc[s], acc[s + 1]);
            if ((lane & 31) == 0) wsum[s + (lane >> 5)][wave] = w;
        }
        if constexpr (NS % 2 == 1) {
            const double w = wave_reduce_dpp<false>(acc[NS - 1]);
            if (lane == 0) wsum[NS - 1][wave] = w;
        }
        if constexpr (MAXLAST) {
            const double w = wave_reduce_dpp<true>(acc[S - 1]);
            if (lane == 0) wsum[S - 1][wave] = w;
        }
        __syncthreads();
        const unsigned row = post_stride(nwg);
        u64 *post = a.tagged + (size_t)(bicg_set(red, gen) * kSums * row);
#pragma unroll
        for (int s0 = 0; s0 < S; s0 += kBW) {
            const int s = s0 + wave;
            if (s < S) {
                const bool mx = MAXLAST && s == S - 1;
                auto op = [&](double x, double y) { return mx ? fmax(x, y) : x + y; };
                static_assert(kBW == 8, "8 waves");
                double v = wsum[s][lane & 7];
                v = op(v, dpp_d<0xB1>(v));   // quad_perm [1,0,3,2]
                v = op(v, dpp_d<0x4E>(v));   // quad_perm [2,3,0,1]
                v = op(v, dpp_d<0x141>(v));  // row_half_mirror
                if (lane == 0) st_coh(post + (size_t)s * row + bid, post_word(v));
            }
        }
        if (wave > 0) mid();
        ops_done();  // before polling (kCgSets)
        // the totals: false after `limit` polls, or once the grid has declined (admit, may be null)
        auto poll = [&](unsigned limit, const int *admit) {
            bool ok = !admit || limit > 0u;
#pragma unroll
            for (int s0 = 0; s0 < S; s0 += kBW) {
                const int s = s0 + wave;
                if (s < S) {
                    const bool mx = MAXLAST && s == S - 1;
                    const u64 *set = post + (size_t)s * row;
                    double v;
                    unsigned spins = 0;
                    for (;;) {
                        u64 u[4];
                        bool ready = true;
                        v = 0.0;
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            if (64u * j >= nwg) continue;
                            const unsigned w = (unsigned)lane + 64u * j;
                            u[j] = ld_coh(set + (w < nwg ? w : 0u));
                        }
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            if ((unsigned)lane + 64u * j >= nwg) continue;
                            ready = ready & (u[j] != 0);
                            const double q = post_value(u[j]);
                            v = mx ? fmax(v, q) : v + q;
                        }
                        if (__all(ready)) break;
                        if (++spins > limit) {
                            ok = false;
                            break;
                        }
                        if (admit) {
                            if (ld_coh(admit) == kAdmitDecline) {
                                ok = false;
                                break;
                            }
                            wait_long(spins);
                        }
                    }
                    const double g = mx ? wave_reduce_dpp<true>(v) : wave_reduce_dpp<false>(v);
                    if (lane == 0) tot[s] = g;
                }
            }
            return ok;
        };
        bool ok;
        for (bool admit = red == kRedFirst && gen == 0u;; admit = false) {
            ok = poll(admit ? a.admit : a.spin, admit ? &a.ctl->admit : nullptr);
            if (!admit) break;
            if (!ok && lane == 0) s_late = 1;
            __syncthreads();
            if (wave == 0) {
                const bool go = block_admit(a.ctl, bid, !s_late);
                if (lane == 0) s_go = go;
            }
            __syncthreads();
            if (!s_go) return false;
            if (ok) break;  // else workgroup 0 admitted the grid while this wait ran out: everything is posted
        }
        if (!ok && lane == 0) {
            st_coh(&a.ctl->err, 1);
            s_err = 1;
        }
        // clear the words of the next reduction of this kind (all workgroups have read them: they have posted this one);
        // complete before this workgroup polls the next reduction of any kind, so before the post that lets others read
        // them
        if (red != kRedFirst) {
            u64 *next = a.tagged + (size_t)(bicg_set(red, gen + 1u) * kSums * row);
#pragma unroll
            for (int s0 = 0; s0 < S; s0 += kBW)
                if (lane == 0 && s0 + wave < S) st_coh(next + (size_t)(s0 + wave) * row + bid, (u64)0);
        }
        __syncthreads();
        return s_err == 0;
    };

    // halo slots of this thread
    const int h0 = t - 64;
    const bool any_halo = h0 >= 0 && h0 < nh;
    // position of halo row j of this thread; rows the thread does not have repeat its first one (or position 0)
    auto halo_pos = [&](int j) {
        return any_halo ? (unsigned)(ltile[h0 / kTile + j * (kBF / kTile)] * kTile + h0 % kTile) : 0u;
    };
    static_assert(kBF % kTile == 0, "a thread's halo rows have the same place in their tiles");
    // in registers where they fit (57 x 35 x 30, three right-hand sides: 130 us per solve, spilling, without 121; FP64 234
    // and 193)
    constexpr bool kPosReg = RPT < 4 && !(NR == 3 && RPT == 2);
    unsigned hpos[kPosReg ? HPT : 1];
    if constexpr (kPosReg) {
#pragma unroll
        for (int j = 0; j < HPT; ++j) hpos[j] = halo_pos(j);
    }
    // FP32: load until every halo word of the vector carries `tag` (bounded: the workgroup then ends with the reduction
    // under way, so that no other wait is begun); FP64: one load
    auto fetch_halo = [&](int vec, int k, unsigned tag, auto store) {
        constexpr int HB = BIG ? HPT / 2 : HPT;  // BIG: half of the words at a time (registers)
        static_assert(HPT % HB == 0, "whole batches");
        const Word *base = words + (size_t)(vec * NR + k) * npos;
#pragma unroll
        for (int b = 0; b < HPT; b += HB) {
            unsigned spins = 0;
            for (;;) {
                Word u[HB];
#pragma unroll
                for (int j = 0; j < HB; ++j)
                    u[j] = ld_coh(elem(base, kPosReg ? hpos[kPosReg ? b + j : 0] : halo_pos(b + j)));
                unsigned stale = 0;
#pragma unroll
                for (int j = 0; j < HB; ++j) {
                    bool mine = true;
                    store(b + j, Pub<R>::open(u[j], tag, mine));
                    stale |= mine ? 0u : 1u;
                }
                if (!__any(any_halo && stale)) break;
                if (++spins > a.spin) {
                    if (lane == 0) {
                        st_coh(&a.ctl->err, 1);
                        s_err = 1;
                    }
                    break;
                }
            }
        }
    };

    unsigned pubm = 0;  // bit q: the wave publishes its rows q (the same in all its lanes)
    // iterations of all groups, and those that came to their last reduction: generations; seq + 1 tags the words
    unsigned seq = 0, seq_c = 0;
    for (int k0 = 0, group = 0; k0 < (NR > 1 ? NR : a.nrhs); k0 += NR, ++group) {
        // row indices are found where they are used (kept over the iterations, they spill)
        unsigned ti = (unsigned)t;
        asm volatile("" : "+v"(ti));
        R v[NR][BIG ? 1 : RPT], x[NR][BIG ? 1 : RPT], sh[NR][BIG ? 1 : RPT], tv[NR][RPT];
        R hv[NR][BIG ? 1 : HPT], ht[NR][HPT];
        // ---- r0 = b - A x0 ----
        if (group > 0) __syncthreads();  // the last group's r and p have been read
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            const R *xk = a.x + (size_t)(k0 + k) * a.n;
#pragma unroll
            for (int q = 0; q < RPT; ++q) {
                const int li = t + q * T;
                const int i = block_row<C, NZ>(m, bid, ti + q * T);
                const R x0 = i < 0 ? R(0) : *elem(xk, (unsigned)i);
                lr[k][li] = x0;
                if constexpr (BIG) xw[li] = x0;
                else x[k][q] = x0;
                fence(q);
            }
            if (wave > 0) {
#pragma unroll
                for (int j = 0; j < HPT; ++j) {
                    const unsigned pos = halo_pos(j);
                    const int i = block_row<C, NZ>(m, pos / C, pos % C);
                    lr[k][C + h0 + j * kBF] = i < 0 ? R(0) : *elem(xk, (unsigned)i);
                    fence(j);
                }
            }
        }
        __syncthreads();
        double acc0[NR + 1];
        acc0[NR] = 0.0;  // max|b| over all right-hand sides (infinite: some workgroup cannot hold its rows)
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            acc0[k] = 0.0;
            const R *bk = a.b + (size_t)(k0 + k) * a.n;
#pragma unroll
            for (int q = 0; q < RPT; ++q) {
                const int li = t + q * T;
                const int i = block_row<C, NZ>(m, bid, ti + q * T);
                const R bv = i < 0 ? R(0) : *elem(bk, (unsigned)i);
                const R rv = bv - product(lr[k], q);
                tv[k][q] = rv;
                if constexpr (!BIG) {
                    sh[k][q] = rv;
                    v[k][q] = R(0);
                } else {
                    lv[li] = R(0);
                }
                lp[k][li] = R(0);
                st_coh(elem(rh + (size_t)k * npos, first + (unsigned)li), rv);
                acc0[k] += (double)rv * (double)rv;
                acc0[NR] = fmax(acc0[NR], fabs((double)bv));
                fence(q);
            }
        }
        if (group == 0) {
            for (int k = NR; k < a.nrhs; ++k)
                for (int q = 0; q < RPT; ++q) {
                    const int i = block_row<C, NZ>(m, bid, ti + q * T);
                    if (i >= 0) acc0[NR] = fmax(acc0[NR], fabs((double)a.b[(size_t)k * a.n + i]));
                }
            if (s_over) acc0[NR] = INFINITY;
        }
        if (!reduce(kRedFirst, (unsigned)group, std::true_type{}, acc0, [] {})) return;
#pragma unroll
        for (int k = 0; k < NR; ++k)
#pragma unroll
            for (int q = 0; q < RPT; ++q) lr[k][t + q * T] = tv[k][q];
        double rho[NR], alpha[NR], omega[NR], beta[NR], res[NR];
        int active[NR], conv[NR], finite[NR], used[NR];
        bool any = false;
        if (group == 0) {
            const double bmax = uniform_d(tot[NR]);
            if (isinf(bmax)) {
                if (bid == 0 && t == 0) a.ctl->zero_all = 1;  // not solved here
                return;
            }
            if (a.zero_shortcut && bmax == 0.0) {
                for (int k = 0; k < a.nrhs; ++k)
                    for (int q = 0; q < RPT; ++q) {
                        const int i = block_row<C, NZ>(m, bid, ti + q * T);
                        if (i >= 0) a.x[(size_t)k * a.n + i] = R(0);
                    }
                if (bid == 0 && t < a.nrhs) cg1_init(a.st[t], 0.0, 1);
                return;
            }
#pragma unroll
            for (int q = 0; q < RPT; ++q)
                if (__any(ld_coh(mark + (first + (unsigned)(t + q * T)) / kTile) == a.salt)) pubm |= 1u << q;
            pubm = (unsigned)__builtin_amdgcn_readfirstlane((int)pubm);
        }
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            rho[k] = uniform_d(tot[k]);  // (rhat, r) with rhat = r
            const double nr0 = sqrt(rho[k]) * a.crit_scale;
            alpha[k] = omega[k] = beta[k] = res[k] = 0.0;
            finite[k] = 1;
            used[k] = -1;
            conv[k] = nr0 < a.tol ? 1 : 0;  // bicgstab_solver_kernel.cu:259, :351-356
            if (conv[k]) res[k] = nr0;
            active[k] = __builtin_amdgcn_readfirstlane(conv[k] ? 0 : 1);
            any = any || active[k];
        }
        if (any && wave > 0) {
#pragma unroll
            for (int k = 0; k < NR; ++k)
#pragma unroll
                for (int j = 0; j < HPT; ++j) {
                    const int h = C + h0 + j * kBF;
                    const unsigned pos = kPosReg ? hpos[kPosReg ? j : 0] : halo_pos(j);
                    lr[k][h] = ld_coh(elem(rh + (size_t)k * npos, pos));
                    lp[k][h] = R(0);
                    if constexpr (BIG) lv[h] = R(0);
                    else hv[k][j] = R(0);
                    ht[k][j] = R(0);
                }
        }
        for (int it = 0; it < a.maxit && any; ++it, ++seq) {
            const unsigned tag = seq + 1u;
            // ---- p = r + beta (p - omega v); v = A p; (rhat, v) ----
#pragma unroll
            for (int k = 0; k < NR; ++k) {
                if (!active[k]) continue;
                const R be = (R)beta[k], mom = (R)-omega[k];
#pragma unroll
                for (int q = 0; q < RPT; ++q) {
                    const int li = t + q * T;
                    lp[k][li] = fma(be, fma(mom, BIG ? lv[BIG ? li : 0] : v[k][BIG ? 0 : q], lp[k][li]), lr[k][li]);
                    fence(q);
                }
                if (wave > 0) {
#pragma unroll
                    for (int j = 0; j < HPT; ++j) {
                        const int h = C + h0 + j * kBF;
                        lp[k][h] = fma(be, fma(mom, BIG ? lv[BIG ? h : 0] : hv[k][BIG ? 0 : j], lp[k][h]), lr[k][h]);
                    }
                }
            }
            __syncthreads();
            double acc_a[NR];
#pragma unroll
            for (int k = 0; k < NR; ++k) {
                acc_a[k] = 0.0;
                if (!active[k]) continue;
                unsigned at = first + (unsigned)t;
                if constexpr (RPT >= 8) asm volatile("" : "+v"(at));
                constexpr int B = BIG ? RPT / 2 : RPT;  // BIG: the shadow residual's loads of B rows pass the products
#pragma unroll
                for (int q0 = 0; q0 < RPT; q0 += B) {
                    R shb[B];
                    if constexpr (BIG) {
#pragma unroll
                        for (int q = 0; q < B; ++q) shb[q] = *elem(rh, at + (q0 + q) * T);
                        __builtin_amdgcn_sched_barrier(0);
                    }
#pragma unroll
                    for (int q = q0; q < q0 + B; ++q) {
                        R y = product(lp[k], q);
                        if (pubm >> q & 1u) put_row(0, k, at + q * T, y, tag);
                        if constexpr (BIG) lv[t + q * T] = y;
                        else v[k][q] = y;
                        acc_a[k] += (double)(BIG ? shb[q - q0] : sh[k][BIG ? 0 : q]) * (double)y;
                        fence(q);
                    }
                }
            }
            auto fetch_v = [&] {
#pragma unroll
                for (int k = 0; k < NR; ++k)
                    if (active[k])
                        fetch_halo(0, k, tag, [&](int j, R g) {
                            if constexpr (BIG) lv[C + h0 + j * kBF] = g;
                            else hv[k][j] = g;
                        });
            };
            auto fetch_t = [&] {
#pragma unroll
                for (int k = 0; k < NR; ++k)
                    if (active[k]) fetch_halo(1, k, tag, [&](int j, R g) { ht[k][j] = g; });
            };
            if (!reduce(kRedA, seq, std::false_type{}, acc_a, [&] {
                    if constexpr (kTagged) fetch_v();
                }))
                return;
            if constexpr (!kTagged)
                if (wave > 0) fetch_v();
            // ---- s = r - alpha v; t = A s; |s|^2, (t, s), (t, t) ----
#pragma unroll
            for (int k = 0; k < NR; ++k) {
                if (!active[k]) continue;
                alpha[k] = uniform_d(rho[k] / tot[k]);
                const R mal = (R)-alpha[k];
#pragma unroll
                for (int q = 0; q < RPT; ++q) {
                    const int li = t + q * T;
                    lr[k][li] = fma(mal, BIG ? lv[BIG ? li : 0] : v[k][BIG ? 0 : q], lr[k][li]);
                    fence(q);
                }
                if (wave > 0) {
#pragma unroll
                    for (int j = 0; j < HPT; ++j) {
                        const int h = C + h0 + j * kBF;
                        lr[k][h] = fma(mal, BIG ? lv[BIG ? h : 0] : hv[k][BIG ? 0 : j], lr[k][h]);
                    }
                }
            }
            __syncthreads();
            double acc_b[3 * NR];
#pragma unroll
            for (int k = 0; k < NR; ++k) {
                acc_b[3 * k] = acc_b[3 * k + 1] = acc_b[3 * k + 2] = 0.0;
                if (!active[k]) continue;
                unsigned at = first + (unsigned)t;
                if constexpr (RPT >= 8) asm volatile("" : "+v"(at));
#pragma unroll
                for (int q = 0; q < RPT; ++q) {
                    const R y = product(lr[k], q);
                    if (pubm >> q & 1u) {
                        R out = y;
                        if constexpr (RPT >= 8) asm volatile("" : "+v"(out));  // t is not tied to the word's registers
                        put_row(1, k, at + q * T, out, tag);
                    }
                    tv[k][q] = y;
                    const double sd = (double)lr[k][t + q * T], td = (double)y;
                    acc_b[3 * k] += sd * sd;
                    acc_b[3 * k + 1] += td * sd;
                    acc_b[3 * k + 2] += td * td;
                    fence(q);
                }
            }
            if (!reduce(kRedB, seq, std::false_type{}, acc_b, [&] {
                    if constexpr (kTagged) fetch_t();
                }))
                return;
            // ---- x += alpha p (+ omega s); r = s - omega t; |r|^2, (rhat, r) ----
            if constexpr (!kTagged)
                if (wave > 0) fetch_t();
            double acc_c[2 * NR];
            any = false;
#pragma unroll
            for (int k = 0; k < NR; ++k) {
                acc_c[2 * k] = acc_c[2 * k + 1] = 0.0;
                if (!active[k]) continue;
                const double nr = sqrt(uniform_d(tot[3 * k])) * a.crit_scale;
                used[k] = it;
                res[k] = nr;
                finite[k] = isfinite(nr) ? 1 : 0;
                conv[k] = nr < a.tol ? 1 : 0;
                omega[k] = uniform_d(tot[3 * k + 1] / tot[3 * k + 2]);
                active[k] = __builtin_amdgcn_readfirstlane(finite[k] && !conv[k] ? 1 : 0);
                any = any || active[k];
                const R al = (R)alpha[k], om = (R)omega[k];
                constexpr int B = BIG ? RPT / 2 : RPT;
                unsigned at = (unsigned)t;
                if constexpr (RPT >= 8) asm volatile("" : "+v"(at));
#pragma unroll
                for (int q0 = 0; q0 < RPT; q0 += B) {
                    R xb[B], shb[B];
#pragma unroll
                    for (int q = 0; q < B; ++q) {
                        xb[q] = BIG ? *elem(xw, at + (q0 + q) * T) : x[k][BIG ? 0 : q];
                        shb[q] = BIG ? *elem(rh, first + at + (q0 + q) * T) : sh[k][BIG ? 0 : q];
                    }
                    if constexpr (BIG) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int q = q0; q < q0 + B; ++q) {
                        const int li = t + q * T;
                        R xv = fma(al, lp[k][li], xb[q - q0]);
                        if (active[k]) {
                            const R sv = lr[k][li];
                            xv = fma(om, sv, xv);
                            const R rv = fma(-om, tv[k][q], sv);
                            lr[k][li] = rv;
                            acc_c[2 * k] += (double)rv * (double)rv;
                            acc_c[2 * k + 1] += (double)shb[q - q0] * (double)rv;
                        }
                        if constexpr (BIG) *elem(xw, at + q * T) = xv;
                        else x[k][q] = xv;
                        fence(q);
                    }
                }
                if (wave > 0 && active[k]) {
#pragma unroll
                    for (int j = 0; j < HPT; ++j) {
                        const int h = C + h0 + j * kBF;
                        lr[k][h] = fma(-om, ht[k][j], lr[k][h]);
                    }
                }
            }
            if (!any) {
                ++seq;
                break;
            }
            if (!reduce(kRedC, seq_c++, std::false_type{}, acc_c, [] {})) return;
            any = false;
#pragma unroll
            for (int k = 0; k < NR; ++k) {
                if (!active[k]) continue;
                const double nr = sqrt(uniform_d(tot[2 * k])) * a.crit_scale;
                res[k] = nr;
                if (nr < a.tol) {
                    conv[k] = 1;
                    used[k] = it + 1;
                    active[k] = 0;
                } else {
                    const double rho_n = uniform_d(tot[2 * k + 1]);
                    beta[k] = uniform_d((rho_n / rho[k]) * (alpha[k] / omega[k]));
                    rho[k] = rho_n;
                    any = true;
                }
                active[k] = __builtin_amdgcn_readfirstlane(active[k]);
            }
        }
        // ---- results of the group ----
        asm volatile("" : "+v"(ti));
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            R *xk = a.x + (size_t)(k0 + k) * a.n;
#pragma unroll
            for (int q = 0; q < RPT; ++q) {
                const int li = t + q * T;
                const int i = block_row<C, NZ>(m, bid, ti + q * T);
                if (i >= 0) *elem(xk, (unsigned)i) = BIG ? xw[li] : x[k][BIG ? 0 : q];
                fence(q);
            }
            if (bid == 0 && t == 0) {
                RhsState st;
                cg1_init(st, rho[k], 0);
                st.alpha = alpha[k];
                st.beta = beta[k];
                st.omega = omega[k];
                st.final_res = res[k];
                st.active = active[k];
                st.converged = conv[k];
                st.finite = finite[k];
                st.used = used[k];
                a.st[k0 + k] = st;
            }
        }
    }
}

// Instances: NR = nrhs right-hand sides together, or one after the other (BicgBlock::together).
template <typename R, int RPT, int NZ, int HPT, int NRM>
static BicgBlock pick(int nrhs, BicgBlock alone) {
    if (nrhs == NRM) return {{(const void *)k_bicg_block<R, RPT, NZ, HPT, NRM, false>, 512, RPT}, NRM};
    return alone;
}
template <typename R, int RPT, int NZ, int HPT, bool BIG = false>
static BicgBlock single() {
    return {{(const void *)k_bicg_block<R, RPT, NZ, HPT, 1, BIG>, 512, RPT}, 1};
}
BicgBlock bicg_block(bool f32, int nz, int rpt, int nrhs) {
    if (nz <= 5) {
        switch (rpt) {
            case 1: if (f32) return pick<float, 1, 5, 2, 2>(nrhs, single<float, 1, 5, 2>()); break;
            case 2:
                return f32 ? pick<float, 2, 5, 2, 2>(nrhs, single<float, 2, 5, 2>())
                           : pick<double, 2, 5, 2, 2>(nrhs, single<double, 2, 5, 2>());
            case 4:
                return f32 ? pick<float, 4, 5, 3, 2>(nrhs, single<float, 4, 5, 3>())
                           : pick<double, 4, 5, 3, 2>(nrhs, single<double, 4, 5, 3>());
            case 8: if (f32) return pick<float, 8, 5, 4, 2>(nrhs, single<float, 8, 5, 4>()); break;
            default: break;
        }
    } else {
        switch (rpt) {
            case 1:
                return f32 ? pick<float, 1, 7, 3, 3>(nrhs, single<float, 1, 7, 3>())
                           : pick<double, 1, 7, 3, 3>(nrhs, single<double, 1, 7, 3>());
            case 2:
                return f32 ? pick<float, 2, 7, 4, 3>(nrhs, single<float, 2, 7, 4>())
                           : pick<double, 2, 7, 4, 3>(nrhs, single<double, 2, 7, 4>());
            case 4:
                return f32 ? pick<float, 4, 7, 6, 3>(nrhs, single<float, 4, 7, 6>()) : single<double, 4, 7, 6>();
            case 8: if (f32) return single<float, 8, 7, 9>(); break;
            case 14: if (f32) return single<float, 14, 7, 12, true>(); break;
            default: break;
        }
    }
    return {{nullptr, 0, 0}, 0};
}

}  // namespace pict

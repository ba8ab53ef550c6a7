// pict_block.hpp -- the placement that k_cg_block and k_bicg_block share (pict_cgblock.hip, pict_bicgblock.hip): a
// system's rows dealt to one workgroup of 512 threads per compute unit, their entries in registers, and the rows of
// other workgroups that their products need ("halo").
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "pict_krylov.hpp"

namespace pict {

constexpr int kTile = 8;  // rows of a halo tile

// base[i] through a scalar base and a 32-bit byte offset (one address register per load, not two): every array of a
// system this kernel takes is below 4 GiB
template <typename E>
__device__ __forceinline__ E *elem(E *base, unsigned i) {
    using Byte = std::conditional_t<std::is_const_v<E>, const char, char>;
    return reinterpret_cast<E *>(reinterpret_cast<Byte *>(base) + (size_t)(i * (unsigned)sizeof(E)));
}

// Owner and local index of the rows of a system.
struct BlockMap {
    int n, nwg;                // workgroups that own rows
    int brick;                 // 0: rows in order, 1: blocks of a x b lines
    int nx, ny, nz, a, b, nby;
    float inx, iny, ia, ib, inby;  // reciprocals
};
// floor(v / d) from d's rounded reciprocal, for v < 2^21 (every position of a system this kernel takes): the exact
// (v + 1/2) / d lies at least 1 / (2 d) from an integer, the two roundings move it by less than v / d * 2^-22
__device__ __forceinline__ unsigned block_div(unsigned v, float inv) { return (unsigned)(((float)v + 0.5f) * inv); }

template <int C>
__device__ __forceinline__ int block_row(const BlockMap &m, unsigned bid, unsigned li) {
    if (!m.brick) {
        const int i = (int)(bid * (unsigned)C + li);
        return i < m.n ? i : -1;
    }
    const unsigned line = block_div(li, m.inx), x = li - line * (unsigned)m.nx;
    const unsigned lz = block_div(line, m.ia), ly = line - lz * (unsigned)m.a;
    const unsigned bz = block_div(bid, m.inby), by = bid - bz * (unsigned)m.nby;
    const unsigned y = by * (unsigned)m.a + ly, z = bz * (unsigned)m.b + lz;
    if (lz >= (unsigned)m.b || y >= (unsigned)m.ny || z >= (unsigned)m.nz) return -1;
    const int i = (int)((z * (unsigned)m.ny + y) * (unsigned)m.nx + x);
    return i < m.n ? i : -1;
}
// position of row c: owner * C + local index
template <int C>
__device__ __forceinline__ unsigned block_pos(const BlockMap &m, unsigned c) {
    if (!m.brick) return c;
    const unsigned line = block_div(c, m.inx), x = c - line * (unsigned)m.nx;
    const unsigned z = block_div(line, m.iny), y = line - z * (unsigned)m.ny;
    const unsigned by = block_div(y, m.ia), ly = y - by * (unsigned)m.a;
    const unsigned bz = block_div(z, m.ib), lz = z - bz * (unsigned)m.b;
    return (bz * (unsigned)m.nby + by) * (unsigned)C + (lz * (unsigned)m.a + ly) * (unsigned)m.nx + x;
}

// The row mapping, by all threads of a workgroup (every workgroup finds the same one); key: LDS scratch.
template <int T, int C, int NZ>
__device__ __forceinline__ void block_map(const int32_t *row, const int32_t *col, int n, int nwg, BlockMap &m,
                                          unsigned *key) {
    const int t = (int)threadIdx.x;
    if (t == 0) {
        m.n = n;
        m.brick = 0;
        m.nwg = (n + C - 1) / C;
        key[0] = key[1] = 0xffffffffu;
    }
    __syncthreads();
    if constexpr (NZ == 7) {
        // lines and planes: the first of T rows spread over the system (at varying places in their lines) with the
        // offsets of an interior row
        const int i = (int)((((long long)n * (2 * t + 1)) / (2 * T) + 37 * t) % n);
        int d2 = 0, d3 = 0;
        const int rs = row[i];
        if (row[i + 1] - rs == 7 && col[rs + 3] == i && col[rs + 4] == i + 1 && col[rs + 2] == i - 1) {
            d2 = col[rs + 5] - i;
            d3 = col[rs + 6] - i;
            const bool ok = col[rs + 1] == i - d2 && col[rs] == i - d3 && d2 >= 4 && d3 > d2 && d3 % d2 == 0;
            if (ok) atomicMin(&key[0], (unsigned)t);
        }
        __syncthreads();
        const unsigned who = key[0];
        if (who != 0xffffffffu && (unsigned)t == who) {
            m.nx = d2;
            m.ny = d3 / d2;
            m.nz = (int)(((long long)n + d3 - 1) / d3);
        }
        __syncthreads();
        if (who != 0xffffffffu) {
            // blocks of a x b lines that fit a workgroup, at most nwg of them, with the fewest halo lines
            const int nx = m.nx, ny = m.ny, nz = m.nz;
            int a = 0, b = 0, nby = 0, nbz = 0;
            if (t < ny && (long long)nx * (t + 1) <= C) {
                nby = (ny + t) / (t + 1);
                a = (ny + nby - 1) / nby;
                b = min(C / (nx * a), nz);
                nbz = (nz + b - 1) / b;
                b = (nz + nbz - 1) / nbz;
                const int halo = (nby > 1 ? b : 0) + (nbz > 1 ? a : 0);
                if ((long long)nby * nbz <= nwg) atomicMin(&key[1], ((unsigned)halo << 16) | (unsigned)t);
            }
            __syncthreads();
            if (key[1] != 0xffffffffu && (key[1] & 0xffffu) == (unsigned)t) {
                m.a = a;
                m.b = b;
                m.nby = nby;
                m.nwg = nby * nbz;
                m.inx = 1.0f / (float)nx;
                m.iny = 1.0f / (float)ny;
                m.ia = 1.0f / (float)a;
                m.ib = 1.0f / (float)b;
                m.inby = 1.0f / (float)nby;
                m.brick = 1;
            }
            __syncthreads();
        }
    }
}

// Wave totals of two sums at once: every lane of the lower half gets v0's, of the upper half v1's (the halves are
// swapped so that each carries one value, then both go through the same five steps).
__device__ __forceinline__ double wave_sum2(double v0, double v1) {
    auto swap32 = [](double &x, double &y) {
        const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(x), __double2loint(y), false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(x), __double2hiint(y), false, false);
        x = __hiloint2double((int)hi[0], (int)lo[0]);
        y = __hiloint2double((int)hi[1], (int)lo[1]);
    };
    swap32(v0, v1);
    double v = v0 + v1;
    v += dpp_d<0xB1>(v);   // quad_perm [1,0,3,2]
    v += dpp_d<0x4E>(v);   // quad_perm [2,3,0,1]
    v += dpp_d<0x124>(v);  // row_ror:4
    v += dpp_d<0x128>(v);  // row_ror:8
    const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(v), __double2loint(v), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(v), __double2hiint(v), false, false);
    return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}

// Halo tiles of workgroup bid, by all its T threads: every foreign column of its rows marks its tile of kTile rows in
// `bits` (LDS: one bit per tile of the system, then the number of marked tiles before each word, 16 bits each), a scan
// numbers the marked tiles, ltile[k] is tile k and mark[tile] = salt tells its owner.  Returns the halo rows (at most
// H); sets s_over (LDS) when there are more, or a row has more than NO entries besides its diagonal.
template <int T, int C, int H, int RPT, int NO>
__device__ __forceinline__ int block_halo(const int32_t *row, const int32_t *col, const BlockMap &m, unsigned bid,
                                          unsigned *bits, int *ltile, int *scan, int &s_over, int *mark, int salt) {
    constexpr int kBW = T / 64, kBF = T - 64;
    const int t = (int)threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const unsigned first = bid * (unsigned)C;
    const int nw = m.nwg * (C / (kTile * 32));
    unsigned short *base = reinterpret_cast<unsigned short *>(bits + nw);
    for (int k = t; k < nw; k += T) bits[k] = 0;
    __syncthreads();
    for (int q = 0; q < RPT; ++q) {
        const int i = block_row<C>(m, bid, (unsigned)(t + q * T));
        if (i < 0) continue;
        const int rs = row[i], re = row[i + 1];
        bool diag = false;
        for (int e = rs; e < re; ++e) {
            const unsigned c = (unsigned)col[e];
            diag |= (int)c == i;
            const unsigned pos = block_pos<C>(m, c);
            if (pos - first >= (unsigned)C) atomicOr(&bits[pos / (kTile * 32)], 1u << ((pos / kTile) & 31));
        }
        if (re - rs > NO + (diag ? 1 : 0)) s_over = 1;
    }
    __syncthreads();
    const int per = (nw + T - 1) / T, k0 = min(t * per, nw), k1 = min(k0 + per, nw);
    int cnt = 0;
    for (int k = k0; k < k1; ++k) cnt += __popc(bits[k]);
    int inc = cnt;
#pragma unroll
    for (int off = 1; off < 64; off *= 2) {
        const int o = __shfl_up(inc, off, 64);
        if (lane >= off) inc += o;
    }
    if (lane == 63) scan[wave] = inc;
    __syncthreads();
    int start = inc - cnt, total = 0;
    for (int w = 0; w < kBW; ++w) {
        if (w < wave) start += scan[w];
        total += scan[w];
    }
    if (total * kTile > H) {
        if (t == 0) s_over = 1;
    }
    for (int k = k0; k < k1; ++k) {
        base[k] = (unsigned short)start;
        for (unsigned b = bits[k]; b; b &= b - 1) {
            const int tile = k * 32 + __ffs((int)b) - 1;
            if (start < H / kTile) ltile[start] = tile;
            st_coh(mark + tile, salt);
            ++start;
        }
    }
    const int nh = min(total * kTile, H);
    __syncthreads();
    // a thread's unused halo slots repeat its first one
    for (int k = t; k < H / kTile; k += T)
        if (k * kTile >= nh) ltile[k] = (k % (kBF / kTile)) * kTile < nh ? ltile[k % (kBF / kTile)] : 0;
    __syncthreads();
    return nh;
}

// The entries of row ii (local index li, first entry rs, len entries, none: 0) into registers: diagonal, values and LDS
// byte offsets (16 bits, two per word) of the other columns; term(value, column) for each in the order of the products.
// The entries lie around the diagonal: up to NO / 2 before it end at slot NO / 2 - 1, those after it start at slot
// NO / 2, so that a product adds them in the row's order (rows with more on one side, such as those whose neighbours
// wrap around, fill the slots in order).  Slots without an entry hold the own column with value 0.
template <int C, int H, int NZ, bool ONE, bool PIN, typename R, typename Term>
__device__ __forceinline__ void block_load_row(const SolveArgs<R> &a, const BlockMap &m, int ii, int li, unsigned first,
                                               int rs, int len, const unsigned *bits, R &dv, R (&val)[NZ - 1],
                                               unsigned (&idx)[NZ / 2], Term term) {
    constexpr int NO = NZ - 1, NI = (NO + 1) / 2;
    static_assert(NI == NZ / 2, "odd row lengths");
    len = min(len, NZ);
    const int last = rs + max(len, 1) - 1;
    int pd = NZ;  // entry of the diagonal
#pragma unroll
    for (int e = NZ - 1; e >= 0; --e) pd = e < len && *elem(a.col, min(rs + e, last)) == ii ? e : pd;
    const bool centred = pd <= NO / 2 && len - 1 - pd <= NO / 2;
    auto value = [&](int k) { return *elem(a.val, a.perm ? *elem(a.perm, k) : k); };
    dv = pd < len ? value(rs + pd) : R(0);
#pragma unroll
    for (int j = 0; j < NI; ++j) idx[j] = 0;
#pragma unroll
    for (int j = 0; j < NO; ++j) {
        const int e = centred ? j - NO / 2 + pd + (j >= NO / 2 ? 1 : 0) : j + (j >= pd ? 1 : 0);
        const bool in = e >= 0 && e < len;
        const int k = in ? rs + e : last;
        const int cj = in ? *elem(a.col, k) : ii;
        val[j] = in ? value(k) : R(0);
        if (j == NO / 2) term(dv, ii);
        term(val[j], cj);
        const unsigned pos = block_pos<C>(m, (unsigned)cj);
        unsigned l = pos - first;
        if constexpr (!ONE) {
            const unsigned short *base =
                reinterpret_cast<const unsigned short *>(bits + (unsigned)m.nwg * (unsigned)(C / (kTile * 32)));
            const unsigned k = pos / (kTile * 32), bit = (pos / kTile) & 31;
            const unsigned slot = base[k] + (unsigned)__popc(bits[k] & ((1u << bit) - 1u));
            l = l < (unsigned)C ? l : (unsigned)C + min(slot * kTile + pos % kTile, (unsigned)(H - 1));
        }
        l = cj == ii ? (unsigned)li : l;  // (a row without entries has no position)
        idx[j / 2] |= (l * (unsigned)sizeof(R)) << (16 * (j & 1));
        if constexpr (PIN) asm volatile("" : "+v"(idx[j / 2]));  // one entry after the other (registers)
    }
}

}  // namespace pict

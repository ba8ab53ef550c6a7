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

// Owner and local index of the rows of a system: rows in order, or blocks of a x b lines of a 3-D grid.  A grid whose
// lines are too long for the halo is cut across its lines first, into strips of nx cells: strip by strip the rows get
// new numbers, line by line within it (lines that a strip does not fill leave numbers unused), and the rest sees a grid
// of `strips` times as many lines of nx cells.
struct BlockMap {
    int n, nwg;                // workgroups that own rows
    int brick;                 // 0: rows in order, 1: blocks of a x b lines
    int nx, ny, nz, a, b, nby;
    float inx, iny, ia, ib, inby;  // reciprocals
    int strips, line, lines;       // strips, cells of a line of the grid, lines of a strip
    float iline, ilines;
};
// floor(v / d) from d's rounded reciprocal, for v < 2^21 (every position of a system this kernel takes): the exact
// (v + 1/2) / d lies at least 1 / (2 d) from an integer, the two roundings move it by less than v / d * 2^-22
__host__ __device__ __forceinline__ unsigned block_div(unsigned v, float inv) { return (unsigned)(((float)v + 0.5f) * inv); }

// the row with number v (strips), or -1; of line q and cell x of the strip grid
__host__ __device__ __forceinline__ int strip_row(const BlockMap &m, unsigned q, unsigned x) {
    const unsigned s = block_div(q, m.ilines), l = q - s * (unsigned)m.lines, gx = s * (unsigned)m.nx + x;
    if (s >= (unsigned)m.strips || gx >= (unsigned)m.line) return -1;
    const int i = (int)(l * (unsigned)m.line + gx);
    return i < m.n ? i : -1;
}

// (2-D systems, NZ == 5, are always strips: rows in order are one strip of one line of n cells.  The set-up runs once and
// at the rate at which its instructions arrive; a branch around the strips in each of its unrolled copies cost 3 us.)
template <int C, int NZ>
__host__ __device__ __forceinline__ int block_row(const BlockMap &m, unsigned bid, unsigned li) {
    if (NZ == 5 || !m.brick) {
        const unsigned v = bid * (unsigned)C + li;
        if (NZ == 7) return (int)v < m.n ? (int)v : -1;
        const unsigned q = block_div(v, m.inx);
        return strip_row(m, q, v - q * (unsigned)m.nx);
    }
    const unsigned line = block_div(li, m.inx), x = li - line * (unsigned)m.nx;
    const unsigned lz = block_div(line, m.ia), ly = line - lz * (unsigned)m.a;
    const unsigned bz = block_div(bid, m.inby), by = bid - bz * (unsigned)m.nby;
    const unsigned y = by * (unsigned)m.a + ly, z = bz * (unsigned)m.b + lz;
    if (lz >= (unsigned)m.b || y >= (unsigned)m.ny || z >= (unsigned)m.nz) return -1;
    return strip_row(m, z * (unsigned)m.ny + y, x);
}
// position of row c: owner * C + local index
template <int C, int NZ>
__host__ __device__ __forceinline__ unsigned block_pos(const BlockMap &m, unsigned c) {
    if (NZ == 7 && !m.brick) return c;
    const unsigned l = block_div(c, m.iline), gx = c - l * (unsigned)m.line, s = block_div(gx, m.inx);
    const unsigned line = s * (unsigned)m.lines + l, x = gx - s * (unsigned)m.nx;
    if (NZ == 5) return line * (unsigned)m.nx + x;
    const unsigned z = block_div(line, m.iny), y = line - z * (unsigned)m.ny;
    const unsigned by = block_div(y, m.ia), ly = y - by * (unsigned)m.a;
    const unsigned bz = block_div(z, m.ib), lz = z - bz * (unsigned)m.b;
    return (bz * (unsigned)m.nby + by) * (unsigned)C + (lz * (unsigned)m.a + ly) * (unsigned)m.nx + x;
}
// the mapping in scalar registers (the same in every lane)
__device__ __forceinline__ BlockMap uniform_map(const BlockMap &in) {
    static_assert(sizeof(BlockMap) % sizeof(int) == 0, "words");
    BlockMap out;
    const int *src = reinterpret_cast<const int *>(&in);
    int *dst = reinterpret_cast<int *>(&out);
#pragma unroll
    for (int k = 0; k < (int)(sizeof(BlockMap) / sizeof(int)); ++k) dst[k] = __builtin_amdgcn_readfirstlane(src[k]);
    return out;
}

// the map as a kernel keeps it: a reference to LDS or scalar registers
template <bool REF>
__device__ __forceinline__ std::conditional_t<REF, const BlockMap &, BlockMap> pick_map(const BlockMap &map) {
    if constexpr (REF) return map;
    else return uniform_map(map);
}

// rows in order, on one workgroup unless nwg says otherwise
__host__ __device__ __forceinline__ BlockMap whole_map(int n, int nwg = 1) {
    BlockMap m{};
    m.n = m.nx = m.line = n;
    m.nwg = nwg;
    m.strips = m.lines = 1;
    m.inx = m.iline = 1.0f / (float)n;
    m.ilines = 1.0f;
    return m;
}

// whole tiles of rows
__host__ __device__ __forceinline__ int whole_tiles(int rows) { return (rows + kTile - 1) & ~(kTile - 1); }
// width of the strips when lines of nx cells are cut into k (0: no such strips)
__device__ __forceinline__ int strip_width(int nx, int k) {
    const int w = whole_tiles((nx + k - 1) / k);
    return (nx + w - 1) / w == k && w >= 2 * kTile ? w : 0;
}
// Row of sample k of K that show the lines of the grid: spread over the system, at varying places in their lines.
template <int K>
__device__ __forceinline__ int sample_row(int n, unsigned k) {
    const unsigned un = (unsigned)n;
    unsigned i = un * (2 * k + 1) / (2 * K) + 37 * k;  // below 2^32: K <= 64, systems of up to 2^21 rows
    i = i >= un ? i - un : i;
    i = i >= un ? i - un : i;
    return (int)min(i, un - 1u);
}

// 2-D: the map of a grid whose lines of nx cells do not fit the halo, by all threads of a workgroup (every workgroup
// finds the same one).  Strips need the lines above and below (of two strips, where one ends and the next begins) and a
// tile to the left and right of every line; of those that fit the fewest workgroups, then the smallest halo.
template <int T, int C, int H>
__device__ __forceinline__ void strip_map(int n, int nx, int nwg, BlockMap &m, unsigned &key) {
    const int t = (int)threadIdx.x, k = t + 2, w = strip_width(nx, k), ny = (n + nx - 1) / nx;
    if (w > 0) {
        const int wgs = (int)(((long long)k * ny * w + C - 1) / C);
        const int halo = 4 * w + 2 * kTile * ((C - 1) / w + 2);
        if (wgs <= nwg && halo <= H) atomicMin(&key, ((unsigned)wgs << 20) | ((unsigned)halo << 9) | (unsigned)t);
    }
    static_assert(T <= 512 && H < 2048, "bits of the key");
    __syncthreads();
    if (key != 0xffffffffu && (key & 0x1ffu) == (unsigned)t) {
        m.strips = k;
        m.nx = w;
        m.line = nx;
        m.lines = ny;
        m.nwg = (int)(key >> 20);
        m.inx = 1.0f / (float)w;
        m.iline = 1.0f / (float)nx;
        m.ilines = 1.0f / (float)ny;
    }
    __syncthreads();
}

// 3-D: the row mapping, by all threads of a workgroup (every workgroup finds the same one): blocks of a x b lines that
// fit a workgroup, at most nwg of them, with the fewest halo lines; a thread tries its number of lines along y.
template <int T, int C, int H>
__device__ __forceinline__ void brick_map(const int32_t *row, const int32_t *col, int n, int nwg, BlockMap &m,
                                          unsigned (&key)[2]) {
    constexpr int NZ = 7;
    const int t = (int)threadIdx.x;
    // lines and planes: the first sample with the offsets of an interior row
    int d2 = 0, d3 = 0;
    constexpr int K = 64;  // one wave's: a load touches a line of memory for each
    const int i = t < K ? sample_row<K>(n, (unsigned)t) : 0, rs = t < K ? row[i] : 0;
    if (t < K && row[i + 1] - rs == NZ) {
        int o[NZ];  // all loads before the first test
#pragma unroll
        for (int e = 0; e < NZ; ++e) o[e] = col[rs + e] - i;
        d2 = o[5];
        d3 = o[6];
        const bool ok = (o[3] == 0) & (o[4] == 1) & (o[2] == -1) & (o[1] == -d2) & (o[0] == -d3) & (d2 >= 4) & (d3 > d2);
        if (ok && d3 % d2 == 0) atomicMin(&key[0], (unsigned)t);
    }
    __syncthreads();
    const unsigned who = key[0];
    if (who == 0xffffffffu) return;
    if ((unsigned)t == who) {
        m.line = m.nx = d2;
        m.ny = d3 / d2;
        m.nz = (int)(((long long)n + d3 - 1) / d3);
    }
    __syncthreads();
    const int nx = m.nx, ny = m.ny, nz = m.nz;
    int a = 0, b = 0, nby = 0, nbz = 0;
    auto blocks = [&](int w, int k) {  // halo lines of blocks of lines cut into k strips of w cells, or -1
        if (t >= ny || (long long)w * (t + 1) > C) return -1;
        nby = (ny + t) / (t + 1);
        a = (ny + nby - 1) / nby;
        b = min(C / (w * a), nz);
        nbz = (nz + b - 1) / b;
        b = (nz + nbz - 1) / nbz;
        return (long long)k * nby * nbz <= nwg ? (nby > 1 ? b : 0) + (nbz > 1 ? a : 0) : -1;
    };
    int best_w = nx, best_k = 1;
    const int halo = blocks(nx, 1);
    if (halo >= 0) atomicMin(&key[1], ((unsigned)halo << 16) | (unsigned)t);
    __syncthreads();
    const unsigned best = key[1];
    bool mine = best != 0xffffffffu && (best & 0xffffu) == (unsigned)t;
    if (best == 0xffffffffu || 2 * (int)(best >> 16) * nx > H) {
        // lines too long for the halo: strips
        __syncthreads();
        if (t == 0) key[1] = 0xffffffffu;
        __syncthreads();
        unsigned my = 0xffffffffu;
        for (int k = 2; k <= 8; ++k) {
            const int w = strip_width(nx, k);
            const int h = w > 0 ? blocks(w, k) : -1;
            const int rows = 2 * h * w + 2 * kTile * a * b;
            if (h < 0 || rows > H || ((unsigned)rows << 16) >= my) continue;
            my = ((unsigned)rows << 16) | (unsigned)t;
            best_w = w;
            best_k = k;
        }
        if (my != 0xffffffffu) atomicMin(&key[1], my);
        __syncthreads();
        if (key[1] != 0xffffffffu) {
            mine = (key[1] & 0xffffu) == (unsigned)t;
        } else {
            best_w = nx;
            best_k = 1;
        }
        blocks(best_w, best_k);
    }
    if (mine) {
        m.a = a;
        m.b = b;
        m.nby = nby;
        m.nwg = best_k * nby * nbz;
        m.nx = best_w;
        m.strips = best_k;
        m.nz = best_k * nbz * b;  // planes that the last block of a strip does not fill are left out
        m.lines = ny * nbz * b;
        m.iline = 1.0f / (float)nx;
        m.ilines = 1.0f / (float)m.lines;
        m.inx = 1.0f / (float)best_w;
        m.iny = 1.0f / (float)ny;
        m.ia = 1.0f / (float)a;
        m.ib = 1.0f / (float)b;
        m.inby = 1.0f / (float)nby;
        m.brick = 1;
    }
    __syncthreads();
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

// Scratch of the placement in LDS.
struct PlaceLds {
    u64 line;          // first sample row that shows the lines: thread, length
    unsigned key[2];
    int scan[16];
};

// The mapping (in `map`, LDS) and the halo tiles of workgroup bid, by all its T threads: every foreign column of its rows
// marks its tile of kTile rows in `bits` (LDS: one bit per tile of the system, then the number of marked tiles before
// each word, 16 bits each), a scan numbers the marked tiles, ltile[k] is tile k and mark[tile] = salt tells its owner.
// Returns the halo rows (at most H), or -1 in a workgroup without rows; sets s_over (LDS) when there are more, or a row
// has more than NZ - 1 entries besides its diagonal.
template <int T, int C, int H, int RPT, int NZ>
__device__ __forceinline__ int block_place(const int32_t *row, const int32_t *col, int n, int nwg, unsigned bid,
                                           BlockMap &map, unsigned *bits, int *ltile, PlaceLds &lds, int &s_over,
                                           int *mark, int salt) {
    constexpr int kBW = T / 64, kBF = T - 64, NO = NZ - 1;
    static_assert(NZ == 5 || NZ == 7, "2-D and 3-D rows");
    static_assert(kBW <= (int)(sizeof(lds.scan) / sizeof(int)), "waves");
    const int t = (int)threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const unsigned first = bid * (unsigned)C;
    if (t == 0) {
        map = whole_map(n, (n + C - 1) / C);
        lds.line = ~0ull;
        lds.key[0] = lds.key[1] = 0xffffffffu;
    }
    __syncthreads();
    if constexpr (NZ == 7) brick_map<T, C, H>(row, col, n, nwg, map, lds.key);
    BlockMap m;
    int nw;
    // 2-D: rows in order first; the lengths of the lines are found with the same trips to memory
    for (bool again = false;; again = true) {
        m = uniform_map(map);
        nw = m.nwg * (C / (kTile * 32));
        for (int k = t; k < nw; k += T) bits[k] = 0;
        __syncthreads();
        // (16 samples of the last wave, on their way with its own rows' loads, cost a 2-D solve 0.3 us; 64 3 us)
        constexpr int K = 16;
        const bool sample = NZ == 5 && !again && t >= kBF && t < kBF + K;
        const int si = sample ? sample_row<K>(n, (unsigned)(t - kBF)) : 0;
        int srs = 0, slen = 0;
        if (sample) {
            const int own = row[max(block_row<C, NZ>(m, bid, (unsigned)t), 0)];  // (the loop's first trip)
            srs = row[si];
            slen = row[si + 1] - srs;
            asm volatile("" ::"v"(own));
        }
        int o[5] = {0, 0, 0, 0, 0};
        if (sample && slen == 5) {
#pragma unroll
            for (int e = 0; e < 5; ++e) o[e] = col[srs + e];
        }
        for (int q = 0; q < RPT; ++q) {
            const int i = block_row<C, NZ>(m, bid, (unsigned)(t + q * T));
            if (i < 0) continue;
            const int rs = row[i], re = row[i + 1];
            bool diag = false;
            for (int e = rs; e < re; ++e) {
                const unsigned c = (unsigned)col[e];
                diag |= (int)c == i;
                const unsigned pos = block_pos<C, NZ>(m, c);
                if (pos - first >= (unsigned)C) atomicOr(&bits[pos / (kTile * 32)], 1u << ((pos / kTile) & 31));
            }
            if (re - rs > NO + (diag ? 1 : 0)) s_over = 1;
        }
        if constexpr (NZ == 5) {
            // an interior row
            const int d2 = o[4] - si;
            if (sample && slen == 5 && (o[2] == si) & (o[3] == si + 1) & (o[1] == si - 1) & (o[0] == si - d2) & (d2 >= 4))
                atomicMin(&lds.line, ((u64)(unsigned)t << 32) | (unsigned)d2);
            __syncthreads();
            const int nx = lds.line == ~0ull ? 0 : (int)(unsigned)lds.line;
            // rows in order need the line above and the line below (and a few tiles where blocks of a domain meet)
            if (again || 2 * whole_tiles(nx) + 12 * kTile <= H) break;
            strip_map<T, C, H>(n, nx, nwg, map, lds.key[0]);
            if (map.strips == 1) break;
            if (t == 0) s_over = 0;
        } else {
            __syncthreads();
            break;
        }
    }
    if (bid >= (unsigned)m.nwg) return -1;
    unsigned short *base = reinterpret_cast<unsigned short *>(bits + nw);
    const int per = (nw + T - 1) / T, k0 = min(t * per, nw), k1 = min(k0 + per, nw);
    int cnt = 0;
    for (int k = k0; k < k1; ++k) cnt += __popc(bits[k]);
    int inc = cnt;
#pragma unroll
    for (int off = 1; off < 64; off *= 2) {
        const int o = __shfl_up(inc, off, 64);
        if (lane >= off) inc += o;
    }
    if (lane == 63) lds.scan[wave] = inc;
    __syncthreads();
    int start = inc - cnt, total = 0;
    for (int w = 0; w < kBW; ++w) {
        if (w < wave) start += lds.scan[w];
        total += lds.scan[w];
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
        const unsigned pos = block_pos<C, NZ>(m, (unsigned)cj);
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

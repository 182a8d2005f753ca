// gsofa_rows.hip -- L and U rows from the records of a reach-mode run.
//
// A mini-group of the traversal leaves, for every vertex t that its sources'
// searches reached at or above the group, one record per 64 (32) of its
// sources: (t, f, mask).  Bit j says that source f - j reaches t.  A group's
// records are sorted by t.
//
//   A pass     bit j: t is in row f - j of U.  A group's records hold those 64
//              rows whole: a 64 x 64 bit transposition gives them in order.
//   A^T pass   bit j: f - j is in row t of L.  Row t is its records, one per
//              group that reached it, in order of f.
//
// Either way one wave store writes up to 64 consecutive columns of a row, and
// no entry is sorted: records are (tens of entries each).  The column forms of
// the hand-off are the same two kernels on the other pass's records.
//
// What bounds it: the columns' own writes, and for rows of few records the
// chain offsets -> records -> store of a wave per row.
//
// Measured against what it replaces, a stream of 8 B per fill that was cleared,
// counted per row, scattered and sorted (structure pass with supernodes,
// traversal, in ms, before -> now): 48^3 grid 5.6 -> 0.9, 3.27 -> 2.78; band
// n = 659,033 5.8 -> 0.8, 5.71 -> 4.72; 128 2D grids 7.0 -> 1.8, 33.5 -> 31.2.
// 217 M fills of the 48^3 grid are 1.74 GB of stream, its records 0.1 GB.
#include <algorithm>

#include "gsofa_device.h"
#include "gsofa_internal.h"

namespace gsofa {

namespace {

using dev::WAVE;
using dev::rank_in;

constexpr int RT = 256;             // threads per block
constexpr int SITEMS = 8;           // rows per thread of a scan tile
constexpr int STILE = RT * SITEMS;
constexpr uint32_t LSLOTS = 4096;   // records of a long row held in LDS at once
constexpr uint32_t WREC = 64;       // rows of up to so many records: one wave each
constexpr int LROWS = 16;           // rows scanned per step for longer ones

// Inclusive scan over the block of one value per thread; total in *sum.
__device__ __forceinline__ int64_t block_scan(int64_t x, int64_t* sh, int64_t* sum) {
    const uint32_t lane = __lane_id(), w = threadIdx.x / WAVE;
#pragma unroll
    for (int d = 1; d < WAVE; d <<= 1) {
        const int64_t y = __shfl_up(x, d, WAVE);
        if (lane >= (uint32_t)d) x += y;
    }
    if (lane == WAVE - 1) sh[w] = x;
    __syncthreads();
    int64_t add = 0, all = 0;
#pragma unroll
    for (int k = 0; k < RT / WAVE; k++) {
        const int64_t v = sh[k];
        if ((uint32_t)k < w) add += v;
        all += v;
    }
    __syncthreads();
    *sum = all;
    return x + add;
}

// Per row: its fills (the rows' entries less A's own), and per tile of rows the
// sums of L entries, U entries and L records.
__global__ __launch_bounds__(RT) void k_row_sums(RowParams p) {
    __shared__ int64_t sh[RT / WAVE];
    const int64_t base = (int64_t)blockIdx.x * STILE + (int64_t)threadIdx.x * SITEMS;
    int64_t l = 0, u = 0, r = 0;
#pragma unroll
    for (int k = 0; k < SITEMS; k++) {
        const int64_t s = base + k;
        if (s >= p.n) break;
        const unsigned long long c = p.cntL[s];
        const int64_t cl = (int64_t)(uint32_t)c, cu = p.cntU[s];
        int64_t own = 0;  // A's entries off the diagonal
        for (int32_t e = p.rp[s]; e < p.rp[s + 1]; e++) own += p.ci[e] != (int32_t)s;
        p.row_fill[s] = cl + cu - own;
        l += cl;
        u += cu;
        r += (int64_t)(c >> 32);
    }
    if (!p.sums) return;  // counts only
    int64_t tl, tu, tr;
    block_scan(l, sh, &tl);
    block_scan(u, sh, &tu);
    block_scan(r, sh, &tr);
    if (threadIdx.x == 0) {
        p.sums[3 * blockIdx.x] = tl;
        p.sums[3 * blockIdx.x + 1] = tu;
        p.sums[3 * blockIdx.x + 2] = tr;
    }
}

// Row pointers: each block adds up the tiles before its own.
__global__ __launch_bounds__(RT) void k_row_ptrs(RowParams p) {
    __shared__ int64_t sh[RT / WAVE];
    int64_t bl = 0, bu = 0, br = 0;
    for (uint32_t t = threadIdx.x; t < blockIdx.x; t += RT) {
        bl += p.sums[3 * t];
        bu += p.sums[3 * t + 1];
        br += p.sums[3 * t + 2];
    }
    int64_t sl, su, sr;
    block_scan(bl, sh, &sl);
    block_scan(bu, sh, &su);
    block_scan(br, sh, &sr);
    const int64_t base = (int64_t)blockIdx.x * STILE + (int64_t)threadIdx.x * SITEMS;
    int64_t cl[SITEMS], cu[SITEMS], cr[SITEMS], l = 0, u = 0, r = 0;
#pragma unroll
    for (int k = 0; k < SITEMS; k++) {
        const int64_t s = base + k;
        const unsigned long long c = s < p.n ? p.cntL[s] : 0ull;
        cl[k] = l += (int64_t)(uint32_t)c;
        cu[k] = u += s < p.n ? (int64_t)p.cntU[s] : 0;
        cr[k] = r += (int64_t)(c >> 32);
    }
    int64_t tot;
    const int64_t ol = sl + block_scan(l, sh, &tot) - l;
    const int64_t ou = su + block_scan(u, sh, &tot) - u;
    const int64_t orr = sr + block_scan(r, sh, &tot) - r;
#pragma unroll
    for (int k = 0; k < SITEMS; k++) {
        const int64_t s = base + k;
        if (s >= p.n) break;
        p.L_rowptr[s + 1] = ol + cl[k];
        p.U_rowptr[s + 1] = ou + cu[k];
        p.R_ptr[s + 1] = orr + cr[k];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) p.L_rowptr[0] = p.U_rowptr[0] = p.R_ptr[0] = 0;
}

// The group of mini-group `c` (of the pass's) and its records' start.
__device__ __forceinline__ uint64_t grp_at(const RowParams& p, uint32_t ck, uint32_t* items) {
    const uint4 g = p.grp[ck];
    *items = g.z;
    return ((uint64_t)g.y << 32) | g.x;
}

// Records to their rows' lists: count[t] holds row t's records in its high
// half, counted down to zero here.
__global__ __launch_bounds__(RT) void k_rec_lists(RowParams p, uint32_t pass, unsigned long long* count,
                                                  const int64_t* ptr, uint4* list) {
    uint32_t items;
    const uint64_t o = grp_at(p, 2u * blockIdx.x + pass, &items);
    for (uint32_t i = threadIdx.x; i < items * p.words; i += RT) {
        const uint4 e = p.rec[o + i];
        if ((e.z | e.w) == 0u) continue;
        const unsigned long long c = dev::aadd64(&count[e.x], 0ull - (1ull << 32));
        const int64_t q = ptr[e.x] + (int64_t)(c >> 32) - 1;
        if (q < p.list_cap) list[q] = e;
    }
}

// Rows whose records form one group (one word of its sources): 64 x 64 bit
// transpositions.  Waves take parts of the group's records; a row's place for
// each part comes from the counts of the parts before it.
__global__ __launch_bounds__(RT) void k_rows_by_source(RowParams p, uint32_t pass, const int64_t* rowptr, int32_t* dst,
                                                       int64_t cap) {
    constexpr uint32_t NWV = RT / WAVE;
    __shared__ uint32_t cnt[NWV][WAVE];
    const uint32_t lane = __lane_id(), w = threadIdx.x / WAVE;
    const uint32_t ck = 2u * (blockIdx.x / p.words) + pass, word = blockIdx.x % p.words;
    uint32_t items;
    const uint64_t o0 = grp_at(p, ck, &items);
    const uint4* rec = p.rec + o0 + (uint64_t)word * items;
    const BlkChunk C = p.chunks[ck];
    const uint32_t f = C.first - 64u * word;  // the word's first source
    const uint32_t nsrc = C.count > 64u * word ? (C.count - 64u * word < WAVE ? C.count - 64u * word : WAVE) : 0u;
    const uint32_t tiles = (items + WAVE - 1u) / WAVE, per = (tiles + NWV - 1u) / NWV;
    const uint32_t t0 = w * per, t1 = t0 + per < tiles ? t0 + per : tiles;
    uint32_t mine = 0;  // lane j: entries of row f - j in this wave's part
    for (uint32_t t = t0; t < t1; t++) {
        const uint32_t i = t * WAVE + lane;
        const uint4 e = i < items ? rec[i] : make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
        for (int j = 0; j < 64; j++) {
            const uint32_t wd = j < 32 ? e.z : e.w;
            const uint32_t c = (uint32_t)__popcll(__ballot((wd >> (j & 31)) & 1u));
            if (lane == (uint32_t)j) mine += c;
        }
    }
    cnt[w][lane] = mine;
    __syncthreads();
    int64_t pos = lane < nsrc ? rowptr[f - lane] : 0;
    for (uint32_t k = 0; k < w; k++) pos += cnt[k][lane];
    for (uint32_t t = t0; t < t1; t++) {
        const uint32_t i = t * WAVE + lane;
        const uint4 e = i < items ? rec[i] : make_uint4(0u, 0u, 0u, 0u);
        const uint32_t plo = (uint32_t)pos, phi = (uint32_t)((uint64_t)pos >> 32);
        uint32_t add = 0;
#pragma unroll
        for (int j = 0; j < 64; j++) {
            const uint32_t wd = j < 32 ? e.z : e.w;
            const bool in = (wd >> (j & 31)) & 1u;
            const uint64_t b = __ballot(in);
            const int64_t q = (int64_t)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)phi, j) << 32) |
                                        (uint32_t)__builtin_amdgcn_readlane((int)plo, j)) + rank_in(b);
            if (in && q < cap) dst[q] = (int32_t)e.x;
            if (lane == (uint32_t)j) add = (uint32_t)__popcll(b);
        }
        pos += add;
    }
}

// Writes a record's columns in increasing order: lane l has bit S - 1 - l,
// column f - (S - 1 - l).  Every lane of the wave calls it.
__device__ __forceinline__ void store_record(uint64_t m, uint32_t f, uint32_t S, uint32_t lane, int32_t* dst, int64_t q,
                                             int64_t cap) {
    const uint32_t j = S - 1u - lane;
    const bool in = lane < S && ((m >> (j & 63u)) & 1ull);
    const uint64_t b = __ballot(in);
    const int64_t at = q + rank_in(b);
    if (in && at < cap) dst[at] = (int32_t)(f - j);
}

__device__ __forceinline__ uint64_t lane_mask(uint32_t lo, uint32_t hi, uint32_t i) {
    return ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)hi, (int)i) << 32) |
           (uint32_t)__builtin_amdgcn_readlane((int)lo, (int)i);
}

// Rows that take records from many groups, up to WREC of them: one wave per
// row sorts them by first source and stores each.
__global__ __launch_bounds__(RT) void k_rows_by_target(RowParams p, const int64_t* ptr, const uint4* list,
                                                       const int64_t* rowptr, int32_t* dst, int64_t cap) {
    const uint32_t lane = __lane_id(), S = p.slots;
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const uint32_t waves = gridDim.x * (RT / WAVE);
    for (uint32_t r = blockIdx.x * (RT / WAVE) + w; r < (uint32_t)p.n; r += waves) {
        const int64_t b = ptr[r], e = ptr[r + 1];
        if (e <= b || e - b > (int64_t)WREC || e > p.list_cap) continue;
        const uint32_t nt = (uint32_t)(e - b);
        const uint4 t = lane < nt ? list[b + lane] : make_uint4(0u, ~0u, 0u, 0u);
        uint32_t f = t.y, lo = t.z, hi = t.w;  // first sources are distinct in a row; empty lanes last
        for (uint32_t k = 2; k < 2u * nt; k <<= 1) {
            for (uint32_t j = k >> 1; j > 0; j >>= 1) {
                const uint32_t of = __shfl_xor(f, (int)j), ol = __shfl_xor(lo, (int)j), oh = __shfl_xor(hi, (int)j);
                const bool keep_min = ((lane & j) == 0u) == ((lane & k) == 0u);
                if (keep_min ? of < f : of > f) {
                    f = of;
                    lo = ol;
                    hi = oh;
                }
            }
        }
        const uint32_t c = (uint32_t)__popc(lo) + (uint32_t)__popc(hi);
        const uint32_t before = dev::wave_incl_scan(c) - c;
        const int64_t q0 = rowptr[r];
        for (uint32_t i = 0; i < nt; i++)
            store_record(lane_mask(lo, hi, i), (uint32_t)__builtin_amdgcn_readlane((int)f, (int)i), S, lane, dst,
                         q0 + (uint32_t)__builtin_amdgcn_readlane((int)before, (int)i), cap);
    }
}

// Rows of more records: one block per row puts them into LDS slots by first
// source (a row's first sources differ by multiples of the word), a window of
// LSLOTS at a time, and stores them in slot order.
__global__ __launch_bounds__(RT) void k_rows_by_target_long(RowParams p, const int64_t* ptr, const uint4* list,
                                                            const int64_t* rowptr, int32_t* dst, int64_t cap) {
    __shared__ uint64_t slot[LSLOTS];
    __shared__ uint32_t sum[LSLOTS / WAVE];
    __shared__ uint32_t red[2];
    __shared__ uint64_t longs;
    const uint32_t t = threadIdx.x, lane = __lane_id(), S = p.slots;
    const uint32_t w = __builtin_amdgcn_readfirstlane(t / WAVE);
    for (uint32_t r0 = blockIdx.x * LROWS; r0 < (uint32_t)p.n; r0 += gridDim.x * LROWS) {
        if (t < WAVE) {
            bool lng = false;
            if (t < LROWS && r0 + t < (uint32_t)p.n) {
                const int64_t b = ptr[r0 + t], e = ptr[r0 + t + 1];
                lng = e - b > (int64_t)WREC && e <= p.list_cap;
            }
            const uint64_t m = __ballot(lng);
            if (t == 0) longs = m;
        }
        __syncthreads();
        for (uint64_t m = longs; m; m &= m - 1ull) {
            const uint32_t r = r0 + (uint32_t)__builtin_ctzll(m);
            const int64_t b = ptr[r], e = ptr[r + 1];
            if (t == 0) {
                red[0] = ~0u;
                red[1] = 0u;
            }
            __syncthreads();
            uint32_t lo = ~0u, hi = 0u;
            for (int64_t i = b + t; i < e; i += RT) {
                const uint32_t f = list[i].y;
                lo = f < lo ? f : lo;
                hi = f > hi ? f : hi;
            }
            atomicMin(&red[0], lo);
            atomicMax(&red[1], hi);
            __syncthreads();
            lo = red[0];
            hi = red[1];
            int64_t q0 = rowptr[r];
            const uint32_t all = (hi - lo) / S + 1u;
            for (uint32_t s0 = 0; s0 < all; s0 += LSLOTS) {
                const uint32_t ns = all - s0 < LSLOTS ? all - s0 : LSLOTS;
                const uint32_t nt = (ns + WAVE - 1u) / WAVE;
                for (uint32_t i = t; i < nt * WAVE; i += RT) slot[i] = 0ull;
                __syncthreads();
                for (int64_t i = b + t; i < e; i += RT) {
                    const uint4 x = list[i];
                    const uint32_t k = (x.y - lo) / S - s0;
                    if (k < ns) slot[k] = ((uint64_t)x.w << 32) | x.z;
                }
                __syncthreads();
                for (uint32_t k = w; k < nt; k += RT / WAVE) {
                    const uint64_t x = dev::wave_sum64((unsigned long long)__popcll(slot[k * WAVE + lane]));
                    if (lane == 0) sum[k] = (uint32_t)x;
                }
                __syncthreads();
                if (w == 0) {  // LSLOTS / WAVE tiles: one per lane
                    static_assert(LSLOTS / WAVE == WAVE, "one tile per lane");
                    const uint32_t x = lane < nt ? sum[lane] : 0u;
                    sum[lane] = dev::wave_incl_scan(x);
                }
                __syncthreads();
                for (uint32_t k = w; k < nt; k += RT / WAVE) {
                    const uint64_t x = slot[k * WAVE + lane];
                    const uint32_t c = (uint32_t)__popcll(x);
                    const uint32_t before = (k ? sum[k - 1] : 0u) + dev::wave_incl_scan(c) - c;
                    for (uint64_t some = __ballot(c != 0u); some; some &= some - 1ull) {
                        const uint32_t i = (uint32_t)__builtin_ctzll(some);
                        store_record(lane_mask((uint32_t)x, (uint32_t)(x >> 32), i), lo + (s0 + k * WAVE + i) * S, S,
                                     lane, dst, q0 + (uint32_t)__builtin_amdgcn_readlane((int)before, (int)i), cap);
                    }
                }
                q0 += sum[nt - 1];
                __syncthreads();  // slots and sums are read
            }
            __syncthreads();  // red is read
        }
        __syncthreads();  // longs is read
    }
}

}  // namespace

// Scratch words (8 B) of launch_rows' tile sums for n rows.
size_t row_sum_words(int64_t n) { return 3 * (size_t)((n + STILE - 1) / STILE) + 3; }

// Counts only: the rows' fills.
hipError_t launch_row_fills(const RowParams& p, hipStream_t s) {
    RowParams q = p;
    q.sums = nullptr;
    hipLaunchKernelGGL(k_row_sums, dim3((uint32_t)((p.n + STILE - 1) / STILE)), dim3(RT), 0, s, q);
    return hipGetLastError();
}

// Fills, row pointers and the record lists' offsets.
hipError_t launch_row_ptrs(const RowParams& p, hipStream_t s) {
    const dim3 tiles((uint32_t)((p.n + STILE - 1) / STILE));
    hipLaunchKernelGGL(k_row_sums, tiles, dim3(RT), 0, s, p);
    hipLaunchKernelGGL(k_row_ptrs, tiles, dim3(RT), 0, s, p);
    return hipGetLastError();
}

// Sorted rows of U from the A pass's groups, of L from the A^T pass's records.
hipError_t launch_rows(const RowParams& p, hipStream_t s) {
    const uint32_t groups = p.n_chunks / 2u;
    if (groups == 0) return hipSuccess;
    hipLaunchKernelGGL(k_rows_by_source, dim3(groups * p.words), dim3(RT), 0, s, p, 0u, p.U_rowptr, p.U_col, p.U_cap);
    hipLaunchKernelGGL(k_rec_lists, dim3(groups), dim3(RT), 0, s, p, 1u, p.cntL, p.R_ptr, p.list);
    const uint32_t wb = (uint32_t)std::min<int64_t>((p.n + RT / WAVE - 1) / (RT / WAVE), 8192);
    hipLaunchKernelGGL(k_rows_by_target, dim3(wb), dim3(RT), 0, s, p, p.R_ptr, p.list, p.L_rowptr, p.L_col, p.L_cap);
    const uint32_t lb = (uint32_t)std::min<int64_t>((p.n + LROWS - 1) / LROWS, 8192);
    hipLaunchKernelGGL(k_rows_by_target_long, dim3(lb), dim3(RT), 0, s, p, p.R_ptr, p.list, p.L_rowptr, p.L_col,
                       p.L_cap);
    return hipGetLastError();
}

}  // namespace gsofa

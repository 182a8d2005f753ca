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
// traversal, in ms, before -> now): 48^3 grid 5.6 -> 0.73, 3.27 -> 2.78; band
// n = 659,033 5.8 -> 0.65, 5.71 -> 4.72; 128 2D grids 7.0 -> 1.1, 33.5 -> 31.2.
// Rows of L with four rows a wave, and those of over 64 records from a list: 0.48
// -> 0.32 ms at 48^3, 0.90 -> 0.46 at the 128 grids (a workgroup's barriers per
// long row and a wave for every short one before).
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
constexpr uint32_t LSLOTS = 2048;   // record slots of a wave, for rows of over 64 records
constexpr uint32_t LGRID = 512;     // workgroups of k_rows_long: two per CU by their slots
constexpr uint32_t SUB = 16;        // lanes of a row of up to so many records

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

// Per row: its fills (the rows' entries less A's own; not for columns), and per
// tile of rows the sums of L entries, U entries and L records.  Whether A holds a row's diagonal
// comes from a binary search, all of a thread's rows in step.
__global__ __launch_bounds__(RT) void k_row_sums(RowParams p) {
    __shared__ unsigned long long sh[3];
    if (threadIdx.x < 3) sh[threadIdx.x] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * STILE + threadIdx.x;
    int32_t lo[SITEMS], len[SITEMS], end[SITEMS];
#pragma unroll
    for (int k = 0; k < SITEMS; k++) {
        const int64_t s = base + (int64_t)k * RT;
        lo[k] = s < p.n ? p.rp[s] : 0;
        end[k] = s < p.n ? p.rp[s + 1] : 0;
        len[k] = end[k] - lo[k];
    }
    for (bool more = p.row_fill != nullptr; more;) {
        more = false;
#pragma unroll
        for (int k = 0; k < SITEMS; k++) {
            if (len[k] <= 0) continue;
            const int32_t half = len[k] >> 1;
            if (p.ci[lo[k] + half] < (int32_t)(base + (int64_t)k * RT)) {
                lo[k] += half + 1;
                len[k] -= half + 1;
            } else {
                len[k] = half;
            }
            more |= len[k] > 0;
        }
    }
    unsigned long long l = 0, u = 0, r = 0;
#pragma unroll
    for (int k = 0; k < SITEMS; k++) {
        const int64_t s = base + (int64_t)k * RT;
        if (s >= p.n) continue;
        const unsigned long long c = p.cntL[s];
        const int64_t cl = (int64_t)(uint32_t)c, cu = p.cntU[s];
        if (p.row_fill) {
            const int64_t diag = lo[k] < end[k] && p.ci[lo[k]] == (int32_t)s;
            p.row_fill[s] = cl + cu - ((int64_t)(end[k] - p.rp[s]) - diag);
        }
        l += (unsigned long long)cl;
        u += (unsigned long long)cu;
        r += c >> 32;
    }
    if (!p.sums) return;  // counts only
    l = dev::wave_sum64(l);
    u = dev::wave_sum64(u);
    r = dev::wave_sum64(r);
    if (__lane_id() == 0) {
        atomicAdd(&sh[0], l);
        atomicAdd(&sh[1], u);
        atomicAdd(&sh[2], r);
    }
    __syncthreads();
    if (threadIdx.x < 3) p.sums[3 * blockIdx.x + threadIdx.x] = (int64_t)sh[threadIdx.x];
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
        if (p.ctrl && s + 1 == p.n) {
            p.ctrl->nnz_L = ol + cl[k];
            p.ctrl->nnz_U = ou + cu[k];
        }
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

// Counts for the column forms: L columns' entries from the A^T pass's groups
// (the first blocks, p.cntU), U columns' entries and records from the A pass's
// records (p.cntL, zero on entry).
__global__ __launch_bounds__(RT) void k_col_counts(RowParams p, uint32_t* cnt_l, uint32_t by_source) {
    constexpr uint32_t NWV = RT / WAVE;
    __shared__ uint32_t cnt[NWV][WAVE];
    const uint32_t lane = __lane_id(), w = threadIdx.x / WAVE;
    uint32_t items;
    if (blockIdx.x >= by_source) {
        const uint64_t o = grp_at(p, 2u * (blockIdx.x - by_source), &items);
        for (uint32_t i = threadIdx.x; i < items * p.words; i += RT) {
            const uint4 e = p.rec[o + i];
            const uint32_t c = (uint32_t)__popc(e.z) + (uint32_t)__popc(e.w);
            if (c) dev::aadd64(&p.cntL[e.x], (1ull << 32) | c);
        }
        return;
    }
    const uint32_t ck = 2u * (blockIdx.x / p.words) + 1u, word = blockIdx.x % p.words;
    const uint64_t o0 = grp_at(p, ck, &items);
    const uint4* rec = p.rec + o0 + (uint64_t)word * items;
    const BlkChunk C = p.chunks[ck];
    const uint32_t nsrc = C.count > 64u * word ? (C.count - 64u * word < WAVE ? C.count - 64u * word : WAVE) : 0u;
    uint32_t mine = 0;  // lane j: entries of column f - j in this wave's records
    for (uint32_t i0 = w * WAVE; i0 < items; i0 += RT) {
        const uint4 e = i0 + lane < items ? rec[i0 + lane] : make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
        for (int j = 0; j < 64; j++) {
            const uint32_t c = (uint32_t)__popcll(__ballot(((j < 32 ? e.z : e.w) >> (j & 31)) & 1u));
            if (lane == (uint32_t)j) mine += c;
        }
    }
    cnt[w][lane] = mine;
    __syncthreads();
    if (w == 0 && lane < nsrc) {
        for (uint32_t k = 1; k < NWV; k++) mine += cnt[k][lane];
        cnt_l[C.first - 64u * word - lane] = mine;
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

// A wave's row of nt <= 64 records, sorted by first source in registers.
__device__ void row_in_registers(uint32_t S, const uint4* list, int64_t b, uint32_t nt, int32_t* dst, int64_t q0,
                                 int64_t cap) {
    const uint32_t lane = __lane_id();
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
    for (uint32_t i = 0; i < nt; i++)
        store_record(lane_mask(lo, hi, i), (uint32_t)__builtin_amdgcn_readlane((int)f, (int)i), S, lane, dst,
                     q0 + (uint32_t)__builtin_amdgcn_readlane((int)before, (int)i), cap);
}

// A wave's row of any number of records: they go to LDS slots by first source
// (a row's first sources differ by multiples of the word), a window of LSLOTS
// at a time, and are stored in slot order.
__device__ void row_by_slots(uint32_t S, const uint4* list, int64_t b, int64_t e, int32_t* dst, int64_t q0,
                             int64_t cap, uint64_t* slot) {
    const uint32_t lane = __lane_id();
    uint32_t lo = ~0u, hi = 0u;
    for (int64_t i = b + lane; i < e; i += WAVE) {
        const uint32_t f = list[i].y;
        lo = f < lo ? f : lo;
        hi = f > hi ? f : hi;
    }
#pragma unroll
    for (int d = 1; d < WAVE; d <<= 1) {
        const uint32_t ol = __shfl_xor(lo, d), oh = __shfl_xor(hi, d);
        lo = ol < lo ? ol : lo;
        hi = oh > hi ? oh : hi;
    }
    const uint32_t all = (hi - lo) / S + 1u;
    for (uint32_t s0 = 0; s0 < all; s0 += LSLOTS) {
        const uint32_t ns = all - s0 < LSLOTS ? all - s0 : LSLOTS;
        const uint32_t tiles = (ns + WAVE - 1u) / WAVE;
        for (uint32_t k = 0; k < tiles; k++) slot[k * WAVE + lane] = 0ull;
        dev::wave_sync();
        for (int64_t i = b + lane; i < e; i += WAVE) {
            const uint4 x = list[i];
            const uint32_t k = (x.y - lo) / S - s0;
            if (k < ns) slot[k] = ((uint64_t)x.w << 32) | x.z;
        }
        dev::wave_sync();
        for (uint32_t k = 0; k < tiles; k++) {
            const uint64_t x = slot[k * WAVE + lane];
            const uint32_t c = (uint32_t)__popcll(x);
            const uint32_t incl = dev::wave_incl_scan(c);
            for (uint64_t some = __ballot(c != 0u); some; some &= some - 1ull) {
                const uint32_t i = (uint32_t)__builtin_ctzll(some);
                store_record(lane_mask((uint32_t)x, (uint32_t)(x >> 32), i), lo + (s0 + k * WAVE + i) * S, S, lane, dst,
                             q0 + (uint32_t)__builtin_amdgcn_readlane((int)(incl - c), (int)i), cap);
            }
            q0 += (uint32_t)__builtin_amdgcn_readlane((int)incl, WAVE - 1);
        }
        dev::wave_sync();  // slots are read before the next window clears them
    }
}

// Rows that take records from many groups.  A wave takes four rows at a time:
// SUB lanes each while none has over SUB records (most rows of banded and 2D
// matrices), else one after the other; rows of over 64 records go to the list
// of k_rows_long, whose LDS slots would leave this kernel few waves.
__global__ __launch_bounds__(RT) void k_rows_by_target(RowParams p, const int64_t* ptr, const uint4* list,
                                                       const int64_t* rowptr, int32_t* dst, int64_t cap) {
    constexpr uint32_t PER = WAVE / SUB;
    const uint32_t lane = __lane_id(), S = p.slots, sub = lane / SUB, l = lane % SUB;
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const uint32_t step = gridDim.x * (RT / WAVE) * PER;
    for (uint32_t r0 = (blockIdx.x * (RT / WAVE) + w) * PER; r0 < (uint32_t)p.n; r0 += step) {
        const uint32_t r = r0 + sub;
        int64_t b = 0, e = 0, q = 0;
        if (r < (uint32_t)p.n) {
            b = ptr[r];
            e = ptr[r + 1];
            q = rowptr[r];
        }
        if (e > p.list_cap) e = b;
        const uint32_t nt = e - b > 0xFFFF ? 0xFFFFu : (uint32_t)(e - b);
        uint32_t most = nt;
#pragma unroll
        for (uint32_t d = SUB; d < WAVE; d <<= 1) {
            const uint32_t o = __shfl_xor(most, (int)d);
            most = o > most ? o : most;
        }
        most = __builtin_amdgcn_readfirstlane(most);
        if (most == 0u) continue;
        if (most > SUB) {
            for (uint32_t k = 0; k < PER; k++) {
                const int src = (int)(k * SUB);
                const int64_t bk = (int64_t)dev::bcast_64((uint64_t)b, src), ek = (int64_t)dev::bcast_64((uint64_t)e, src);
                const int64_t qk = (int64_t)dev::bcast_64((uint64_t)q, src);
                if (ek <= bk) continue;
                if (ek - bk <= WAVE) row_in_registers(S, list, bk, (uint32_t)(ek - bk), dst, qk, cap);
                else if (lane == 0) p.long_rows[atomicAdd(p.long_count, 1u)] = r0 + k;
            }
            continue;
        }
        const uint4 t = l < nt ? list[b + l] : make_uint4(0u, ~0u, 0u, 0u);
        uint32_t f = t.y, lo = t.z, hi = t.w;
        for (uint32_t k = 2; k < 2u * most; k <<= 1) {
            for (uint32_t j = k >> 1; j > 0; j >>= 1) {
                const uint32_t of = __shfl_xor(f, (int)j), ol = __shfl_xor(lo, (int)j), oh = __shfl_xor(hi, (int)j);
                const bool keep_min = ((l & j) == 0u) == ((l & k) == 0u);
                if (keep_min ? of < f : of > f) {
                    f = of;
                    lo = ol;
                    hi = oh;
                }
            }
        }
        // a record's columns in increasing order: lane l of the row has its bits
        // S - 1 - 4 l down to S - 4 - 4 l
        for (uint32_t i = 0; i < most; i++) {
            const uint64_t m = ((uint64_t)__shfl(hi, (int)i, SUB) << 32) | __shfl(lo, (int)i, SUB);
            const uint32_t fi = __shfl(f, (int)i, SUB);
            const uint32_t top = S - 1u - 4u * l;  // wraps past the word's bits
            const uint32_t nib = i < nt && top < S ? (uint32_t)(m >> (top - 3u)) & 15u : 0u;
            const uint32_t c = (uint32_t)__popc(nib);
            uint32_t incl = c;
#pragma unroll
            for (uint32_t d = 1; d < SUB; d <<= 1) {
                const uint32_t y = __shfl_up(incl, d, SUB);
                if (l >= d) incl += y;
            }
            int64_t at = q + (incl - c);
#pragma unroll
            for (uint32_t j = 0; j < 4u; j++) {
                if ((nib >> (3u - j)) & 1u) {
                    if (at < cap) dst[at] = (int32_t)(fi - (top - j));
                    at++;
                }
            }
            q += __shfl(incl, (int)SUB - 1, SUB);
        }
    }
}

// The listed rows, one wave each.
__global__ __launch_bounds__(RT) void k_rows_long(RowParams p, const int64_t* ptr, const uint4* list,
                                                  const int64_t* rowptr, int32_t* dst, int64_t cap) {
    __shared__ uint64_t slots[RT / WAVE][LSLOTS];
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const uint32_t count = *p.long_count, step = gridDim.x * (RT / WAVE);
    for (uint32_t i = blockIdx.x * (RT / WAVE) + w; i < count; i += step) {
        const uint32_t r = p.long_rows[i];
        row_by_slots(p.slots, list, ptr[r], ptr[r + 1], dst, rowptr[r], cap, slots[w]);
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

// Sorted rows of U from the A pass's groups, of L from the A^T pass's records;
// with `columns` the passes change places (rows_by_source: columns of L).
static hipError_t write_rows(const RowParams& p, bool columns, hipStream_t s) {
    const uint32_t groups = p.n_chunks / 2u, by_source = columns ? 1u : 0u;
    if (groups == 0) return hipSuccess;
    hipLaunchKernelGGL(k_rows_by_source, dim3(groups * p.words), dim3(RT), 0, s, p, by_source, p.U_rowptr, p.U_col,
                       p.U_cap);
    hipLaunchKernelGGL(k_rec_lists, dim3(groups), dim3(RT), 0, s, p, 1u - by_source, p.cntL, p.R_ptr, p.list);
    const int64_t per = (int64_t)(RT / WAVE) * (WAVE / SUB);
    const uint32_t wb = (uint32_t)std::min<int64_t>((p.n + per - 1) / per, 8192);
    hipLaunchKernelGGL(k_rows_by_target, dim3(wb), dim3(RT), 0, s, p, p.R_ptr, p.list, p.L_rowptr, p.L_col, p.L_cap);
    hipLaunchKernelGGL(k_rows_long, dim3(LGRID), dim3(RT), 0, s, p, p.R_ptr, p.list, p.L_rowptr, p.L_col, p.L_cap);
    return hipGetLastError();
}

hipError_t launch_rows(const RowParams& p, hipStream_t s) { return write_rows(p, false, s); }

// Columns of L and U from the records: what a row of p means for U is a column
// of L here and the other way round.  p.cntL, p.long_count zero on entry.
// Against transposing the finished rows (counts and places by global atomics,
// then a sort of every column): 27^3 grid 1.29 -> 0.14 ms.
hipError_t launch_columns(const RowParams& p, uint32_t* cnt_l, hipStream_t s) {
    const uint32_t groups = p.n_chunks / 2u;
    if (groups == 0) return hipSuccess;
    hipLaunchKernelGGL(k_col_counts, dim3(groups * (p.words + 1u)), dim3(RT), 0, s, p, cnt_l, groups * p.words);
    const hipError_t e = launch_row_ptrs(p, s);
    return e != hipSuccess ? e : write_rows(p, true, s);
}

}  // namespace gsofa

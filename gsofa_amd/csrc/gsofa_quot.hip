// gsofa_quot.hip -- strongly connected classes of vertex ranges, which the
// reach-mode traversal walks instead of their vertices.
//
// A source s is searched for through vertices below s.  If a set of vertices
// below s is strongly connected within the vertices below s, the search
// reaches all of it or none of it, so one node stands for the set: its edges
// are those that leave the set, its weight the set's size and row lengths
// (|R| and TE count every vertex).  Reachability, and with it L, U, |R| and
// TE, is exactly what the walk over single vertices gives.
//
// Each matrix's vertices are cut into blocks of 128 (or 64, see quot_shift).
// Level h holds the complete, aligned ranges of 2^h blocks; a range's classes are found in the
// subgraph of its own vertices, from its two halves' classes (level 0: from
// single vertices).  A source in block j uses the ranges of j's binary
// decomposition: the vertices below block j are covered by one range per set
// bit of j, so a vertex of block b < j belongs to its level-h class, h the
// highest bit in which b and j differ.  No level depends on another range of
// the same level, so log2(blocks) launches build them all, and a class set is
// kept once per level however many sources use it.
//
// Classes need not be maximal for the results to be right (any strongly
// connected set will do), so the search for them is bounded: a range with too
// many nodes keeps its halves' classes, and label rounds stop at a fixed count.
//
// What bounds it: latency.  A level is one launch; a range is a chain of
// dependent gathers (row, column, class, class of the class) and barriers,
// 15-20 us of one workgroup whatever its nodes, up to 50 us with rows of
// thousands of targets.  So a range's nodes are closed as a bit matrix
// (2.4 us for 64 nodes, 8 us for 128, 22 us for 240), lanes that share a row
// step its cursor once, rows of a level lie where the matrix's rows lie (no
// allocation), and the vertices' classes of one level are written behind the
// ranges of the next.
//
// Measured, traversal of one execute walking vertices -> classes (the
// classes' construction included): band n = 659,033 780 -> 3.1 ms, band
// n = 100,003 32.3 -> 0.59, 48^3 grid 64.9 -> 1.56, 181^2 grid 16.4 -> 0.45,
// n = 11,948 1.13 -> 0.22.  The construction with label rounds for every range
// and two launches a level took 0.73 ms at 48^3, now 0.36.
#include <algorithm>

#include "gsofa_device.h"
#include "gsofa_internal.h"

namespace gsofa {

namespace {

using dev::WAVE;

constexpr uint32_t NOIDX = 0xFFFFFFFFu;
constexpr uint16_t INERT = 0xFFFFu;
constexpr uint32_t SHORT_ROW = 64;   // rows up to here: 8 lanes each
constexpr uint32_t MID_ROW = 256;    // rows up to here: one wave each; longer ones: the workgroup
constexpr int QN = 256;              // live nodes whose reachability is closed as a bit matrix
constexpr int QM = 4096;             // nodes of a range, at most, if its halves' classes are to be merged
// Ranges with more live nodes are rare where classes pay at all: sparse bands
// near the bottom, before their main class forms.  Up to 2^QBIG_SHIFT vertices
// they go to a few large workgroups that take up to QCAP by label rounds.
constexpr int QCAP = 2048;
constexpr uint32_t QBIG_SHIFT = 11, QBIG_GRID = 256;
// Up to one range per CU, a range gets 1,024 threads: 181^2 grid 0.564 -> 0.549
// ms, 48^3 2.28 -> 2.24, 33^3 0.780 -> 0.769.  More ranges share the CUs, which
// hold two workgroups of 512 threads for one of 1,024: 128 2D grids at 1,024
// threads 6.90 -> 7.36, band n = 659,033 4.09 -> 4.29.
constexpr uint32_t QFEW = 256;
constexpr uint32_t QSEEN = 4096;     // a power of two, at least two rows for every node
// Where merged classes' rows have so many entries, and 16 for every node, their
// members share targets (a band's class of 1,024 vertices has 2,000 entries and
// 256 targets): each goes in once.  Execute ms without -> with: band n = 659,033
// 4.61 -> 3.97, n = 100,003 0.71 -> 0.67, n = 11,948 0.30 -> 0.28; sifting every
// row cost 64^2 and 181^2 grids and the 128 2D grids 2 to 5 percent.
constexpr uint32_t QSIFT = 2048;
static_assert(QSEEN >= 2u * QCAP, "a place and a target name the row");
constexpr int ROUNDS = 4, ITERS = 96;  // label rounds of a range and iterations of a round, at most
constexpr int QB = 1 << kQuotShift;  // vertices of a block, at most
constexpr int QNT = 512, QNT_LEVEL = 512, QNT_BIG = 1024;
static_assert(QB <= QN && QB == 2 * WAVE && 2 << kQuotShiftChain == QB,
              "a block's vertices are the nodes of one bit matrix");

template <int N>
struct QLds {
    uint32_t rb[2 * N], re[2 * N];       // the live nodes' rows over A, then over A^T
    uint32_t cnt[N], deg[2 * N];         // their vertices, their vertices' row lengths
    uint16_t node[N];                    // live node k's number in the range
    uint16_t root[N];                    // class of a live node, named by one of its nodes
    union {
        struct {                         // classes by closure
            uint64_t adj[QN][QN / 64];   // reachability
            uint64_t tr[QN][QN / 64];    // its transpose
        } c;
        struct {                         // classes by label rounds
            uint32_t fw[N], bw[N];
        } l;
        struct {                         // then, of class c:
            uint32_t id[N], size[N];         // its number, its members
            uint32_t sumA[N], sumT[N];       // their row lengths (later row cursors)
            uint32_t vcnt[N], degA[N], degT[N];
            uint32_t seen[QSEEN];            // targets written to rows lately, by row and target
        } s;
    } u;
    uint32_t ne, nlive, nnew, offA, offT, left, got;
    uint32_t chg[3];
    uint16_t live[QM];                   // more than QN nodes: place among the live ones, or INERT
};

// f(i, k, end, step, W) covers edges k, k + step, .. k + 3 step (below end) of
// row i = [rb(i), re(i)); every edge of every row is covered once by the
// workgroup.  W lanes of a wave (8 or 64) work on the row together and call f
// together.
template <int NT, class Row, class F>
__device__ __forceinline__ void each_row(uint32_t m, Row row, F f) {
    const uint32_t tid = threadIdx.x, lane = __lane_id(), w = tid / WAVE;
    for (uint32_t i = tid / 8u; i < m; i += NT / 8) {
        const uint2 r = row(i);
        if (r.y - r.x > SHORT_ROW) continue;
        for (uint32_t k = r.x; k < r.y; k += 32u) f(i, k + (tid & 7u), r.y, 8u, 8);
    }
    uint32_t turn = 0;
    for (uint32_t t0 = 0; t0 < m; t0 += WAVE) {
        const uint32_t i0 = t0 + lane;
        const uint2 r0 = i0 < m ? row(i0) : make_uint2(0u, 0u);
        const uint32_t len = r0.y - r0.x;
        for (uint64_t b = __ballot(len > SHORT_ROW && len <= MID_ROW); b; b &= b - 1ull) {
            if (turn++ % (uint32_t)(NT / WAVE) != w) continue;
            const uint32_t i = t0 + (uint32_t)__builtin_ctzll(b);
            const uint2 r = row(i);
            for (uint32_t k = r.x; k < r.y; k += 4u * WAVE) f(i, k + lane, r.y, (uint32_t)WAVE, WAVE);
        }
        for (uint64_t b = __ballot(len > MID_ROW); b; b &= b - 1ull) {
            const uint32_t i = t0 + (uint32_t)__builtin_ctzll(b);
            const uint2 r = row(i);
            for (uint32_t k = r.x + w * WAVE; k < r.y; k += 4u * NT) f(i, k + lane, r.y, (uint32_t)NT, WAVE);
        }
    }
}

// Strongly connected classes of m <= 64 NW nodes from their adjacency bits
// S.u.c.adj (rows of nodes at or above m empty): Warshall's closure, 64 pivots
// at a time.  Wave w of the first NW holds columns 64 w .. of every row, row
// 64 g + lane as r[g].  The pivots' wave closes its columns by lane broadcasts
// (two and-ors per pivot and row), publishes them, and the others add the
// pivots' rows to the rows that the closed bits name.  root[i]: the smallest
// node that i reaches and that reaches i.  Called by the whole workgroup.
//
// Bound by instruction issue of the few waves that work, and by fetching code
// that a workgroup runs once: a lane per row with every pivot unrolled (NW * 64
// pivots of 17 instructions at NW = 4) took 35 us for 256 nodes, and its code
// evicted the other phases'.  Loops over the pivots below m and columns split
// over the waves take 22; 9.4 -> 7.5 us at 128 nodes.  Pivots taken in pairs
// need fewer steps in sequence and more instructions: 10.4.  With the base
// blocks at 512 threads in place of 128, execute ms before -> after: 181^2 grid
// 0.64 -> 0.57, 128 2D grids 7.25 -> 6.90, n = 11,948 0.278 -> 0.253, 64^2
// 0.345 -> 0.326, 16^2 0.159 -> 0.146, band n = 659,033 4.30 -> 4.09.
template <int NW, int N, int NT>
__device__ __forceinline__ void closure_classes(QLds<N>& S, uint32_t m) {
    constexpr int QD = QN / 32;
    constexpr uint32_t CW = 64u * NW / (NT / WAVE);  // columns that a wave transposes
    static_assert(CW >= 1u && CW <= 32u && 32u % CW == 0u && NT / WAVE >= NW, "a wave's columns are in one dword");
    const uint32_t tid = threadIdx.x, lane = __lane_id(), w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid / WAVE));
    uint32_t(*adj)[QD] = reinterpret_cast<uint32_t(*)[QD]>(S.u.c.adj);
    uint32_t r[NW][2];
    // r |= the rows of block b's pivots, in o, that the bits c name
    auto pivots = [&](int b, const uint32_t (&o)[2], const uint32_t (&c)[NW][2]) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t k0 = 64u * (uint32_t)b + 32u * (uint32_t)h;
            const uint32_t n = m <= k0 ? 0u : m - k0 < 32u ? m - k0 : 32u;
#pragma unroll 4
            for (uint32_t k = 0; k < n; k++) {
                const uint32_t p0 = (uint32_t)__builtin_amdgcn_readlane((int)o[0], (int)(32u * h + k));
                const uint32_t p1 = (uint32_t)__builtin_amdgcn_readlane((int)o[1], (int)(32u * h + k));
#pragma unroll
                for (int g = 0; g < NW; g++) {
                    const uint32_t has = (uint32_t)__builtin_amdgcn_sbfe((int)c[g][h], k, 1u);
                    r[g][0] |= p0 & has;
                    r[g][1] |= p1 & has;
                }
            }
        }
    };
    if (w < (uint32_t)NW) {
#pragma unroll
        for (int g = 0; g < NW; g++) {
            r[g][0] = adj[64 * g + (int)lane][2u * w];
            r[g][1] = adj[64 * g + (int)lane][2u * w + 1u];
        }
    }
#pragma unroll
    for (int b = 0; b < NW; b++) {
        if (w == (uint32_t)b) {
            pivots(b, r[b], r);
#pragma unroll
            for (int g = 0; g < NW; g++) {
                adj[64 * g + (int)lane][2 * b] = r[g][0];
                adj[64 * g + (int)lane][2 * b + 1] = r[g][1];
            }
        }
        if (NW == 1) break;
        __syncthreads();
        if (w < (uint32_t)NW && w != (uint32_t)b) {
            uint32_t c[NW][2];
#pragma unroll
            for (int g = 0; g < NW; g++) {
                c[g][0] = adj[64 * g + (int)lane][2 * b];
                c[g][1] = adj[64 * g + (int)lane][2 * b + 1];
            }
            const uint32_t o[2] = {r[b][0], r[b][1]};
            pivots(b, o, c);
        }
        // the next block's wave writes its own columns only
    }
    if (NW > 1 && w + 1u < (uint32_t)NW) {  // the last wave's columns are complete
#pragma unroll
        for (int g = 0; g < NW; g++) {
            adj[64 * g + (int)lane][2u * w] = r[g][0];
            adj[64 * g + (int)lane][2u * w + 1u] = r[g][1];
        }
    }
    __syncthreads();
    // transpose, by all waves: the ballot of bit c over rows 64 g .. is word g of row c
    {
        const uint32_t c0 = w * CW;
        uint32_t x[NW];
        uint64_t mine[NW];
#pragma unroll
        for (int g = 0; g < NW; g++) {
            x[g] = adj[64 * g + (int)lane][c0 >> 5];
            mine[g] = 0;
        }
#pragma unroll 2
        for (uint32_t k = 0; k < CW; k++) {
#pragma unroll
            for (int g = 0; g < NW; g++) {
                const uint64_t bal = __ballot((x[g] >> ((c0 & 31u) + k)) & 1u);
                if (lane == k) mine[g] = bal;
            }
        }
        if (lane < CW) {
#pragma unroll
            for (int g = 0; g < NW; g++) S.u.c.tr[c0 + lane][g] = mine[g];
        }
    }
    __syncthreads();
    if (tid < m) {
        uint32_t c = tid;
#pragma unroll
        for (int q = NW - 1; q >= 0; q--) {
            const uint64_t both = S.u.c.adj[tid][q] & S.u.c.tr[tid][q];
            if (both) {
                const uint32_t j = 64u * (uint32_t)q + (uint32_t)__builtin_ctzll(both);
                c = j < c ? j : c;
            }
        }
        S.root[tid] = (uint16_t)c;
    }
}

// Classes of m <= N nodes by label rounds over the edge list eb (node pairs):
// every node carries the largest label that reaches it and the largest that it
// reaches; where both are the same node c, the node is strongly connected with
// c.  Labels of heavy nodes are larger, so the range's main class is found in
// the first round and is not hidden behind single vertices that only lead into
// or out of it.  Assigned nodes leave the graph; the next round looks at the
// rest.  Nodes left after ROUNDS stay classes of their own.
template <int N, int NT>
__device__ __forceinline__ void label_classes(QLds<N>& S, uint32_t m, uint32_t ne, const uint32_t* eb) {
    const uint32_t tid = threadIdx.x;
    constexpr uint32_t PM = 2531u;  // odd: a bijection modulo N
    uint32_t inv = PM;              // PM * inv = 1 modulo 2^32, by Newton's iteration
    for (int k = 0; k < 4; k++) inv *= 2u - PM * inv;
    uint32_t* fw = S.u.l.fw;
    uint32_t* bw = S.u.l.bw;
    auto label = [&](uint32_t i) {
        return ((31u - (uint32_t)__builtin_clz(S.cnt[i] | 1u)) << 16) | ((i * PM) & (uint32_t)(N - 1));
    };
    auto named = [&](uint32_t l) { return (l * inv) & (uint32_t)(N - 1); };
    for (uint32_t i = tid; i < m; i += NT) S.root[i] = INERT;
    if (tid < 3) S.chg[tid] = 0;
    for (int rd = 0; rd < ROUNDS; rd++) {
        __syncthreads();
        for (uint32_t i = tid; i < m; i += NT)
            if (S.root[i] == INERT) fw[i] = bw[i] = label(i);
        if (tid == 0) S.left = S.got = 0;
        __syncthreads();
        for (int it = 0; it < ITERS; it++) {
            if (tid == 0) S.chg[(it + 1) % 3] = 0;  // last read two barriers ago
            bool ch = false;
            for (uint32_t e0 = tid; e0 < ne; e0 += 4u * NT) {
                uint32_t ed[4];
#pragma unroll
                for (int q = 0; q < 4; q++) ed[q] = e0 + q * NT < ne ? eb[e0 + q * NT] : 0u;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const uint32_t a = ed[q] >> 16, b = ed[q] & 0xFFFFu;
                    if (a == b || S.root[a] != INERT || S.root[b] != INERT) continue;
                    const uint32_t fa = fw[a], ba = bw[a], fb = fw[b], bb = bw[b];
                    if (fa > fb) {
                        atomicMax(&fw[b], fa);
                        ch = true;
                    }
                    if (bb > ba) {
                        atomicMax(&bw[a], bb);
                        ch = true;
                    }
                }
            }
            // what reaches (is reached by) a node's label reaches (is reached by) the node
            for (uint32_t i = tid; i < m; i += NT) {
                if (S.root[i] != INERT) continue;
                const uint32_t f = fw[i], b = bw[i];
                const uint32_t f2 = fw[named(f)], b2 = bw[named(b)];
                if (f2 > f) {
                    atomicMax(&fw[i], f2);
                    ch = true;
                }
                if (b2 > b) {
                    atomicMax(&bw[i], b2);
                    ch = true;
                }
            }
            if (ch) S.chg[it % 3] = 1;
            __syncthreads();
            if (!S.chg[it % 3]) break;
        }
        __syncthreads();  // all have read chg
        if (tid < 3) S.chg[tid] = 0;
        uint32_t left = 0, got = 0;
        for (uint32_t i = tid; i < m; i += NT) {
            if (S.root[i] != INERT) continue;
            if (fw[i] == bw[i]) {
                const uint32_t c = named(fw[i]);
                S.root[i] = (uint16_t)c;
                got += c != i;
            } else {
                left++;
            }
        }
        if (left) atomicAdd(&S.left, left);
        if (got) atomicAdd(&S.got, got);
        __syncthreads();
        if (S.left == 0 || (S.got == 0 && rd > 0)) break;
    }
    __syncthreads();
    for (uint32_t i = tid; i < m; i += NT)
        if (S.root[i] == INERT) S.root[i] = (uint16_t)i;
    __syncthreads();
    // a class may be named by a node that is not in it (a round cut short):
    // name it by its smallest member
    for (uint32_t i = tid; i < m; i += NT) fw[i] = NOIDX;
    __syncthreads();
    for (uint32_t i = tid; i < m; i += NT) atomicMin(&fw[S.root[i]], i);
    __syncthreads();
    for (uint32_t i = tid; i < m; i += NT) bw[i] = fw[S.root[i]];
    __syncthreads();
    for (uint32_t i = tid; i < m; i += NT) S.root[i] = (uint16_t)bw[i];
}

// One range, by the whole workgroup.  Nodes are the halves' classes (BASE:
// vertices); class k of a range is numbered x + k, x its first vertex.
//  1. Live nodes: all of them up to QN; of more, those with an edge from and
//     an edge to another node of the range (the others are in no cycle).
//  2. The live nodes' edges as bits, and their classes by closure.
//  3. Each class of two or more nodes gets a row: its members' targets outside
//     the class, over A and over A^T.  Other nodes keep theirs.
// A range of more than QM nodes, or N live ones, keeps its halves' classes;
// with `defer`, one of more than N live ones is left to a larger N: returns
// false, having written nothing.
template <int N, int NT, bool BASE>
__device__ bool range_classes(QLds<N>& S, const QuotParams& p, uint32_t lev, uint32_t tab0, uint32_t ctab0,
                              uint32_t range, bool defer) {
    const uint32_t tid = threadIdx.x, lane = __lane_id();
    const uint64_t ln = p.n;
    const uint2 R = p.tab[tab0 + range];
    const uint32_t size = 1u << (p.shift + lev), x = R.x, xr = x + size / 2u;
    const uint4* info_prev = BASE ? nullptr : p.info + (lev - 1u) * ln;
    const uint4* infoT_prev = BASE ? nullptr : p.infoT + (lev - 1u) * ln;
    uint4* info_cur = p.info + lev * ln;
    uint4* infoT_cur = p.infoT + lev * ln;
    int32_t* map_cur = p.nmap + (lev & 1u) * ln;
    const int32_t* map_prev = p.nmap + ((lev + 1u) & 1u) * ln;
    uint32_t m0 = size, m = size;
    if (!BASE) {
        m0 = p.ncnt[ctab0 + R.y];
        m = m0 + p.ncnt[ctab0 + R.y + 1u];
    }
    auto node_at = [&](uint32_t i) { return BASE || i < m0 ? x + i : xr + (i - m0); };
    auto row_of = [&](uint32_t v, bool t) {
        if (!BASE) return t ? infoT_prev[v] : info_prev[v];
        const int32_t* rp = t ? p.rpT : p.rp;
        const uint32_t b = (uint32_t)rp[v], e = (uint32_t)rp[v + 1];
        return make_uint4(b, e, 1u, e - b);
    };
    // node number of target v, NOIDX outside the range
    auto local = [&](int32_t v) {
        const uint32_t o = (uint32_t)v - x;
        if (o >= size) return NOIDX;
        if (BASE) return o;
        uint32_t c;
        if (lev == 1u) c = (uint32_t)p.comp[v];
        else c = (uint32_t)map_prev[p.comp[(lev - 2u) * ln + (uint32_t)v]];
        return c < xr ? c - x : m0 + (c - xr);
    };
    if (tid == 0) S.nlive = S.nnew = S.offA = S.offT = S.ne = 0;
    const bool sparse = !BASE && m > (uint32_t)QN;  // nodes to be sifted first
    bool merge = m <= (uint32_t)QM;
    if (sparse && merge) {
        for (uint32_t i = tid; i < m; i += NT) S.live[i] = 0;
        __syncthreads();
        // bit 0: an edge to another node, bit 1: from another node (words of
        // two nodes, so that the bits can be set with 32-bit atomics)
        uint32_t* flag = reinterpret_cast<uint32_t*>(S.live);
        each_row<NT>(
            m,
            [&](uint32_t i) {
                const uint4 r = info_prev[node_at(i)];
                return make_uint2(r.x, r.y);
            },
            [&](uint32_t i, uint32_t k, uint32_t e, uint32_t st, int) {
                int32_t v[4];
                uint32_t l[4];
#pragma unroll
                for (int q = 0; q < 4; q++) v[q] = k + q * st < e ? p.ci[k + q * st] : -1;
#pragma unroll
                for (int q = 0; q < 4; q++) l[q] = v[q] >= 0 ? local(v[q]) : NOIDX;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    if (l[q] == NOIDX || l[q] == i) continue;
                    atomicOr(&flag[i >> 1], 1u << (16u * (i & 1u)));
                    atomicOr(&flag[l[q] >> 1], 2u << (16u * (l[q] & 1u)));
                }
            });
        __syncthreads();
        for (uint32_t i = tid; i < m; i += NT) {
            uint32_t k = INERT;
            if (S.live[i] == 3u) {
                k = atomicAdd(&S.nlive, 1u);
                if (k < (uint32_t)N) S.node[k] = (uint16_t)i;
            }
            S.live[i] = (uint16_t)(k < (uint32_t)N ? k : INERT);
        }
        __syncthreads();
        merge = S.nlive <= (uint32_t)N;
        if (!merge && defer) return false;
    }
    if (!merge) {  // the halves' classes stand
        for (uint32_t i = tid; i < m; i += NT) {
            const uint32_t v = node_at(i);
            map_cur[v] = (int32_t)(x + i);
            info_cur[x + i] = info_prev[v];
            infoT_cur[x + i] = infoT_prev[v];
        }
        if (tid == 0) {
            p.ncnt[tab0 + range] = m;
            if (lev == p.judge) atomicAdd(&p.ctl->nodes, (unsigned long long)m);
        }
        return true;
    }
    const uint32_t nl = sparse ? S.nlive : m;
    auto node_of = [&](uint32_t k) { return node_at(sparse ? S.node[k] : k); };
    // live node of target v, NOIDX for other nodes and outside the range
    auto live = [&](int32_t v) {
        const uint32_t l = local(v);
        if (!sparse || l == NOIDX) return l;
        return S.live[l] == INERT ? NOIDX : (uint32_t)S.live[l];
    };
    for (uint32_t k = tid; k < nl; k += NT) {
        const uint32_t v = node_of(k);
        const uint4 a = row_of(v, false), t = row_of(v, true);
        S.rb[k] = a.x;
        S.re[k] = a.y;
        S.rb[nl + k] = t.x;
        S.re[nl + k] = t.y;
        S.cnt[k] = a.z;
        S.deg[k] = a.w;
        S.deg[N + k] = t.w;
    }
    const bool bits = N == QN || nl <= (uint32_t)QN;
    uint32_t* eb = p.eb + p.rp[x];  // the range's rows leave room for its edges
    if (bits && tid < (uint32_t)(BASE ? QB : QN)) {
#pragma unroll
        for (int q = 0; q < QN / 64; q++) S.u.c.adj[tid][q] = 0ull;
    }
    __syncthreads();
    auto lds_row = [&](uint32_t i) { return make_uint2(S.rb[i], S.re[i]); };
    each_row<NT>(nl, lds_row, [&](uint32_t i, uint32_t k, uint32_t e, uint32_t st, int) {
        int32_t v[4];
        uint32_t l[4];
#pragma unroll
        for (int q = 0; q < 4; q++) v[q] = k + q * st < e ? p.ci[k + q * st] : -1;
#pragma unroll
        for (int q = 0; q < 4; q++) l[q] = v[q] >= 0 ? live(v[q]) : NOIDX;
        if (bits) {
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (l[q] != NOIDX)
                    atomicOr(reinterpret_cast<unsigned long long*>(&S.u.c.adj[i][l[q] >> 6]), 1ull << (l[q] & 63u));
            return;
        }
        uint32_t cnt = 0;
#pragma unroll
        for (int q = 0; q < 4; q++) cnt += l[q] != NOIDX && l[q] != i;
        if (!cnt) return;
        uint32_t o = atomicAdd(&S.ne, cnt);
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (l[q] != NOIDX && l[q] != i) eb[o++] = (i << 16) | l[q];
    });
    __syncthreads();
    if constexpr (BASE) {
        if (nl <= 64u) closure_classes<1, N, NT>(S, nl);
        else closure_classes<2, N, NT>(S, nl);
    } else {
        if (N > QN && !bits) label_classes<N, NT>(S, nl, S.ne, eb);
        else if (nl <= 64u) closure_classes<1, N, NT>(S, nl);
        else if (nl <= 128u) closure_classes<2, N, NT>(S, nl);
        else closure_classes<QN / 64, N, NT>(S, nl);
    }
    __syncthreads();
    for (uint32_t c = tid; c < nl; c += NT) {
        S.u.s.size[c] = 0;
        S.u.s.sumA[c] = S.u.s.sumT[c] = S.u.s.vcnt[c] = S.u.s.degA[c] = S.u.s.degT[c] = 0;
    }
    __syncthreads();
    // sums per class: the first lane's class of each wave by wave sums (a range
    // mostly has one large class), the others by atomics
    for (uint32_t k0 = tid - lane; k0 < nl; k0 += NT) {
        const uint32_t k = k0 + lane;
        const bool in = k < nl;
        const uint32_t c = in ? S.root[k] : NOIDX;
        const uint32_t la = in ? S.re[k] - S.rb[k] : 0u, lt = in ? S.re[nl + k] - S.rb[nl + k] : 0u;
        const uint32_t vc = in ? S.cnt[k] : 0u, da = in ? S.deg[k] : 0u, dt = in ? S.deg[N + k] : 0u;
        const uint32_t c0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)c);
        const bool same = c == c0;
        const uint32_t members = (uint32_t)__popcll(__ballot(same));
        unsigned long long x0 = same ? ((unsigned long long)la << 32) | lt : 0ull;
        unsigned long long x1 = same ? ((unsigned long long)da << 32) | dt : 0ull;
        unsigned long long x2 = same ? vc : 0u;
        x0 = dev::wave_sum64(x0);  // each half stays below 2^32: row lengths of one matrix
        x1 = dev::wave_sum64(x1);
        x2 = dev::wave_sum64(x2);
        if (in && (!same || lane == 0)) {
            atomicAdd(&S.u.s.size[c], same ? members : 1u);
            atomicAdd(&S.u.s.sumA[c], same ? (uint32_t)(x0 >> 32) : la);
            atomicAdd(&S.u.s.sumT[c], same ? (uint32_t)x0 : lt);
            atomicAdd(&S.u.s.degA[c], same ? (uint32_t)(x1 >> 32) : da);
            atomicAdd(&S.u.s.degT[c], same ? (uint32_t)x1 : dt);
            atomicAdd(&S.u.s.vcnt[c], same ? (uint32_t)x2 : vc);
        }
    }
    __syncthreads();
    // class numbers; a merged class's rows get room for all its members': a
    // range's rows never exceed the matrix's entries in the range's rows, so
    // each level has one matrix's worth of room, divided like the matrix
    const uint32_t baseA = p.ext0 * (1u + lev) + (uint32_t)p.rp[x];
    const uint32_t baseT = p.ext0 * (1u + lev) + (uint32_t)p.rpT[x];
    for (uint32_t c = tid; c < nl; c += NT) {
        const uint32_t n = S.u.s.size[c];
        if (n == 0u) continue;
        const uint32_t id = x + atomicAdd(&S.nnew, 1u);
        uint4 a = make_uint4(S.rb[c], S.re[c], S.u.s.vcnt[c], S.u.s.degA[c]);  // one member: c itself
        uint4 t = make_uint4(S.rb[nl + c], S.re[nl + c], S.u.s.vcnt[c], S.u.s.degT[c]);
        if (n > 1u) {
            a.x = a.y = baseA + atomicAdd(&S.offA, S.u.s.sumA[c]);
            t.x = t.y = baseT + atomicAdd(&S.offT, S.u.s.sumT[c]);
            S.u.s.sumA[c] = a.x;
            S.u.s.sumT[c] = t.x;
        }
        info_cur[id] = a;  // a merged class's row end follows
        infoT_cur[id] = t;
        S.u.s.id[c] = id;
    }
    __syncthreads();
    const uint32_t rows = S.offA + S.offT;
    const bool sift = rows >= QSIFT && rows >= 16u * nl;  // targets that several members share go in once
    if (sift)
        for (uint32_t i = tid; i < QSEEN; i += NT) S.u.s.seen[i] = 0u;
    for (uint32_t k = tid; k < nl; k += NT) {
        const uint32_t c = S.root[k], v = node_of(k);
        if (BASE) p.comp[v] = (int32_t)S.u.s.id[c];
        else map_cur[v] = (int32_t)S.u.s.id[c];
        if (S.u.s.size[c] == 1u) S.rb[k] = S.re[k] = S.rb[nl + k] = S.re[nl + k] = 0u;  // no row to build
    }
    if (sparse) {  // the other nodes stay as they are
        for (uint32_t i = tid; i < m; i += NT) {
            if (S.live[i] != INERT) continue;
            const uint32_t v = node_at(i), id = x + atomicAdd(&S.nnew, 1u);
            map_cur[v] = (int32_t)id;
            info_cur[id] = info_prev[v];
            infoT_cur[id] = infoT_prev[v];
        }
    }
    __syncthreads();
    each_row<NT>(2u * nl, lds_row, [&](uint32_t i, uint32_t k, uint32_t e, uint32_t st, int W) {
        const bool t = i >= nl;
        int32_t* cols = t ? p.ciT : p.ci;
        int32_t v[4];
        uint32_t l[4], cnt = 0;
        const uint32_t c = S.root[t ? i - nl : i];
#pragma unroll
        for (int q = 0; q < 4; q++) v[q] = k + q * st < e ? cols[k + q * st] : -1;
#pragma unroll
        for (int q = 0; q < 4; q++) l[q] = v[q] >= 0 ? live(v[q]) : NOIDX;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            if (l[q] != NOIDX && S.root[l[q]] == c) v[q] = -1;
            if (sift && v[q] >= 0) {
                // the place is row + target * an odd number, so it and the target
                // name the row; another pair may take it, and a repeat goes in
                uint32_t* const at = &S.u.s.seen[(2u * c + (t ? 1u : 0u) + (uint32_t)v[q] * 2531u) & (QSEEN - 1u)];
                if (atomicExch(at, (uint32_t)v[q] + 1u) == (uint32_t)v[q] + 1u) v[q] = -1;
            }
            cnt += v[q] >= 0;
        }
        // one cursor step for the lanes that share the row
        uint32_t incl = cnt;
        for (int d = 1; d < W; d <<= 1) {
            const uint32_t y = __shfl_up(incl, d, W);
            if ((lane & (uint32_t)(W - 1)) >= (uint32_t)d) incl += y;
        }
        const uint32_t all = __shfl(incl, W - 1, W);
        if (all == 0u) return;
        uint32_t o = 0;
        if ((lane & (uint32_t)(W - 1)) == 0u) o = atomicAdd(t ? &S.u.s.sumT[c] : &S.u.s.sumA[c], all);
        o = __shfl(o, 0, W) + incl - cnt;
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (v[q] >= 0) cols[o++] = v[q];
    });
    __syncthreads();
    for (uint32_t c = tid; c < nl; c += NT) {
        if (S.u.s.size[c] <= 1u) continue;
        info_cur[S.u.s.id[c]].y = S.u.s.sumA[c];
        infoT_cur[S.u.s.id[c]].y = S.u.s.sumT[c];
    }
    if (tid == 0) {
        p.ncnt[tab0 + range] = S.nnew;
        if (lev == p.judge) atomicAdd(&p.ctl->nodes, (unsigned long long)S.nnew);
    }
    return true;
}

__global__ __launch_bounds__(QNT) void k_quot_base(QuotParams p) {
    __shared__ QLds<QN> S;
    (void)range_classes<QN, QNT, true>(S, p, 0u, 0u, 0u, blockIdx.x, false);
}

// Classes of every vertex of level `lev`'s ranges, from the level below:
// `blocks` blocks from `block` on share the work.
__device__ __forceinline__ void map_level(const QuotParams& p, uint32_t lev, uint32_t tab0, uint32_t ranges,
                                          uint32_t block, uint32_t blocks) {
    const uint32_t sh = p.shift + lev;
    const uint64_t total = (uint64_t)ranges << sh;
    const int32_t* prev = p.comp + (uint64_t)(lev - 1u) * p.n;
    const int32_t* map = p.nmap + (uint64_t)(lev & 1u) * p.n;
    int32_t* cur = p.comp + (uint64_t)lev * p.n;
    for (uint64_t k = (uint64_t)block * blockDim.x + threadIdx.x; k < total; k += (uint64_t)blocks * blockDim.x) {
        const uint32_t v = p.tab[tab0 + (uint32_t)(k >> sh)].x + ((uint32_t)k & ((1u << sh) - 1u));
        cur[v] = map[prev[v]];
    }
}

// The ranges of a level, one workgroup each.  The blocks behind them write the
// classes of the level below (lev >= 2), which this level's own look-ups take
// in two steps instead.
template <int NT>
__global__ __launch_bounds__(NT) void k_quot_level(QuotParams p, uint32_t lev, uint32_t tab0, uint32_t ctab0,
                                                          uint32_t ranges, uint32_t cranges) {
    __shared__ QLds<QN> S;
    if (lev > p.judge && quot_off(p)) return;
    if (blockIdx.x >= ranges) {
        map_level(p, lev - 1u, ctab0, cranges, blockIdx.x - ranges, gridDim.x - ranges);
        return;
    }
    if (!range_classes<QN, NT, false>(S, p, lev, tab0, ctab0, blockIdx.x, p.shift + lev <= QBIG_SHIFT) &&
        threadIdx.x == 0)
        p.blist[atomicAdd(&p.ctl->big[lev], 1u)] = blockIdx.x;
}

// The ranges that k_quot_level left.
__global__ __launch_bounds__(QNT_BIG) void k_quot_big(QuotParams p, uint32_t lev, uint32_t tab0, uint32_t ctab0) {
    __shared__ QLds<QCAP> S;
    const uint32_t cnt = p.ctl->big[lev];
    for (uint32_t i = blockIdx.x; i < cnt; i += gridDim.x) {
        (void)range_classes<QCAP, QNT_BIG, false>(S, p, lev, tab0, ctab0, p.blist[i], false);
        __syncthreads();  // S is read before the next range resets it
    }
}

__global__ __launch_bounds__(QNT_LEVEL) void k_quot_map(QuotParams p, uint32_t lev, uint32_t tab0, uint32_t ranges) {
    if (quot_off(p)) return;
    map_level(p, lev, tab0, ranges, blockIdx.x, gridDim.x);
}

}  // namespace

// Blocks of 64 where most vertices i have an entry with i - 1 or i + 1, as grids
// do, else of 128: such a block holds long paths, and walks in a source's own
// block, one step of a path at a time, bound small matrices.  Where neighbours
// are rarely coupled a walk takes few steps and the level more is all that
// blocks of 64 bring.  (Looks at up to 1,024 rows, 64 entries of each.)
// Execute ms at blocks of 128 -> 64: 64^2 grid 0.326 -> 0.283, 16^2 0.145 ->
// 0.132, 300 x 200 grid 0.79 -> 0.70, 128 2D grids 6.89 -> 6.67, 48^3 2.24 ->
// 2.21, narrow band n = 60,000 0.72 -> 0.64; 33^3 0.764 -> 0.777 and 24^3 0.339
// -> 0.345 are the worst.  Bands of 256, which stay: n = 659,033 4.09 -> 4.25,
// n = 100,003 0.61 -> 0.65, n = 11,948 0.251 -> 0.258.
uint32_t quot_shift(uint32_t W, int64_t n, const int32_t* rp, const int32_t* ci) {
    if (W <= 1u << kQuotShift) return kQuotShift;
    const int64_t step = std::max<int64_t>(n / 1024, 1);
    int64_t rows = 0, hits = 0;
    for (int64_t i = 0; i < n; i += step, rows++)
        for (int32_t k = rp[i], e = k + std::min(rp[i + 1] - k, 64); k < e; k++)
            if (ci[k] == i - 1 || ci[k] == i + 1) {
                hits++;
                break;
            }
    return 2 * hits > rows ? kQuotShiftChain : kQuotShift;
}

// Levels of the largest matrix: a source's block index is at most blocks - 1,
// and only complete blocks are contracted.
uint32_t quot_levels(uint32_t W, uint32_t shift) {
    const uint32_t last = W == 0u ? 0u : (W - 1u) >> shift;
    uint32_t l = 0;
    while (last >> l) l++;
    return l;
}

uint64_t quot_ext(uint64_t nnz, uint32_t levels) { return nnz * levels; }

// Whether entry numbers of the matrix's and the classes' rows fit 32 bits, also
// where a loop steps past a row's end: up to four steps of a workgroup here, and
// a lane group's step in the traversal.  (A number that wrapped would read as
// one before the row's end, and the loop would go on.)
bool quot_fits(uint64_t nnz, uint32_t levels) {
    constexpr uint64_t past = 1ull << 16;
    static_assert(past >= 8ull * QNT_BIG, "a loop's last step and its lanes");
    return nnz + quot_ext(nnz, levels) + past <= (1ull << 32);
}

int64_t quot_bytes(int64_t n, int64_t nnz, uint32_t W, uint32_t shift) {
    const int64_t L = quot_levels(W, shift);
    if (L == 0) return 0;
    return L * n * (4 + 32) + 8 * n + 4 * nnz + 8 * (int64_t)quot_ext((uint64_t)nnz, (uint32_t)L) +
           16 * ((n >> shift) * 2 + L + 1) + (int64_t)sizeof(QuotCtl) + 4096;
}

// Ranges of every level: tab[off[h] ..] = (first vertex, entry of the first
// half among level h - 1's); the halves' entries are neighbours.
void quot_table(const std::vector<uint32_t>& mat_base, uint32_t levels, uint32_t shift, std::vector<uint2>& tab,
                std::vector<uint32_t>& off) {
    tab.clear();
    off.assign((size_t)levels + 1, 0);
    std::vector<uint32_t> child(mat_base.size(), 0), mine(mat_base.size(), 0);
    for (uint32_t h = 0; h < levels; h++) {
        off[h] = (uint32_t)tab.size();
        for (size_t b = 0; b + 1 < mat_base.size(); b++) {
            const uint32_t nb = mat_base[b + 1] - mat_base[b];
            const uint32_t cnt = (nb == 0u ? 0u : (nb - 1u) >> shift) >> h;
            mine[b] = (uint32_t)tab.size() - off[h];
            for (uint32_t q = 0; q < cnt; q++)
                tab.push_back(make_uint2(mat_base[b] + (q << (shift + h)), child[b] + 2u * q));
        }
        child = mine;
    }
    off[levels] = (uint32_t)tab.size();
}

// p.ctl is zero on entry.
hipError_t launch_quot(const QuotParams& p, const std::vector<uint32_t>& off, hipStream_t s) {
    auto map_blocks = [](uint64_t vertices) {
        return (uint32_t)std::min<uint64_t>((vertices + QNT_LEVEL - 1) / QNT_LEVEL, 1024);
    };
    hipLaunchKernelGGL(k_quot_base, dim3(off[1]), dim3(QNT), 0, s, p);
    uint32_t h = 1;
    for (; h < p.levels && off[h + 1] > off[h]; h++) {
        const uint32_t ranges = off[h + 1] - off[h], below = off[h] - off[h - 1];
        const uint32_t mb = h >= 2 ? map_blocks((uint64_t)below << (p.shift + h - 1)) : 0u;
        auto* level = ranges <= QFEW ? k_quot_level<QNT_BIG> : k_quot_level<QNT_LEVEL>;
        hipLaunchKernelGGL(level, dim3(ranges + mb), dim3(ranges <= QFEW ? QNT_BIG : QNT_LEVEL), 0, s, p, h, off[h],
                           off[h - 1], ranges, below);
        if (p.shift + h <= QBIG_SHIFT)
            hipLaunchKernelGGL(k_quot_big, dim3(std::min(ranges, QBIG_GRID)), dim3(QNT_BIG), 0, s, p, h, off[h],
                               off[h - 1]);
    }
    if (h >= 2) {
        const uint32_t ranges = off[h] - off[h - 1];
        hipLaunchKernelGGL(k_quot_map, dim3(map_blocks((uint64_t)ranges << (p.shift + h - 1))), dim3(QNT_LEVEL), 0,
                           s, p, h - 1u, off[h - 1], ranges);
    }
    return hipGetLastError();
}

}  // namespace gsofa

// gsofa_reach.hip -- two-pass reachability traversal (GSOFA_MODE_REACH).
//
// The fill-path theorem splits row s of struct(L+U) into two reachability
// questions that need no labels:
//   U_s = {m > s : m is reached from s through vertices below s}, and with it
//         R_<(s) (the vertices below s so reached) and TE_alg;
//   L_s = {m < s : s is reached from m through vertices below m in A^T}, since
//         a path s -> ... -> m of A whose intermediates lie below m is a path
//         m -> ... -> s of A^T whose intermediates lie below its source m.
// So one kernel answers both: over A it yields U rows, |R| and TE exactly as
// the reference's traversal does for U (with_space_optimization/
// symbfact.cuh:883-1082, the "m > src" branch at :992-1009); over A^T it
// yields L columns, from whose records the same sorted rows are built.  Each
// (vertex, source) pair is expanded at most once, where the reference's max-id
// labels re-expand a vertex each time its label drops (2-10 times per pair on
// 3D nested-dissection grids).
//
// Execution model (CDNA4, persistent grid of co-resident workgroups: one of
// 1024 threads per CU with the largest tables, or two of 512 threads or four of
// 256 with a part of it each, so one runs while another waits at a barrier):
// * A workgroup owns MB source slots (32, 64, 128 or 256: the bits of a mask
//   of one, two or four 64-bit words) and runs a mini-group of up to MB
//   sources of one matrix, in one of the two passes, through all of its
//   levels alone.  The next mini-group comes from one global counter over a
//   work table that interleaves the passes' chunks, deepest first, so both
//   passes share one launch and its tail.
// * With 32 and 64 slots a mini-group's nodes (the vertices and classes that its
//   sources reach, a few hundred on banded and 2D matrices, up to thousands on
//   3D ones) are kept in an LDS table for its whole traversal, with their
//   visited and pending bits (walk_nodes): a lane group pops a node, maps each
//   edge's target to its node, ORs the new bits into it and queues it if it had
//   none pending.  A level is one barrier, and per hop only the graph is read
//   from memory: edges, their classes, new nodes' rows.  What bounds it: those
//   three dependent reads, 2 to 3 us a level, and for wide levels the LDS
//   operations per edge.  Execute ms, before -> now: 64^2 grid in natural order
//   0.41 -> 0.33; 181^2 0.84 -> 0.64; 27^3 0.76 -> 0.59; 33^3 1.08 -> 0.79; band
//   of 100,003 0.79 -> 0.70; 128 2D grids 11.1 -> 7.2; 48^3, whose deep groups
//   outgrow it, 2.30 -> 2.13.
// * A mini-group goes on in memory from where its nodes outgrow the table
//   (nodes_to_memory), and every one with more slots starts there, as follows.
// * Per vertex, one word holds the MB slots' visited bits with the
//   mini-group's stamp beside it; an older stamp reads as "nothing visited",
//   so the array is never cleared between mini-groups (the reference's
//   source-stamped markers, symbfact.cuh:2126, generalised to a bit per slot).
// * A level runs in rounds of two phases separated by workgroup barriers:
//     A. combine: lane groups of G lanes pop frontier vertices (all lanes of
//        a group load the same queue entry and mask, so nothing is
//        broadcast between lanes); a step covers G*E edges of the vertex,
//        lane j taking edges j, j+G, ... with all E loads issued first; each
//        target is found or inserted in an LDS hash table of the round's
//        distinct targets and the vertex's slot mask ORed into the target's
//        mask (ds_or);
//     B. relax: one lane per table entry: new = mask & ~visited; the new bits
//        of slots whose source lies above the target push it to the next
//        frontier (its R_<(s) membership), the others are U entries (fills
//        from level 1 on: level 0 expands the sources themselves, whose
//        neighbours are A's own entries).
//   Targets are unique within a round, so the visited word, the next-level
//   mask and the queue append need no global atomics.  The round's counters
//   alternate by parity and the level's by level parity, so a round costs two
//   barriers and a level no more.
// * Nothing is written per entry during the search.  A vertex above the group
//   goes to a list when it is first reached; at the group's end the final
//   visited word of each, and of the group's own vertices, is all entries of
//   that vertex for the group.  The words become records (vertex, first
//   source, mask of 64 sources), sorted by vertex with an LDS bitmap, from
//   which gsofa_rows.hip writes the rows; the A pass also counts its rows' U
//   entries, the A^T pass adds to its targets' L counts.
// * Vertices below the block of the mini-group's lowest source are not walked
//   one by one: strongly connected classes of block ranges stand for them
//   (gsofa_quot.hip).  Combine maps each target below that block to its
//   class, relax takes a class's row, vertex count and row-length sum from
//   the class table.  |R| and TE add those weights, so they count vertices.
// * A class's row can hold thousands of targets, which one lane group would
//   take alone while the workgroup waits: rows over SPLIT_ROW are expanded in
//   SPLIT_PARTS parts by as many groups.
// * Sources of a mini-group form an arithmetic sequence first, first-stride,
//   ... (the cyclic source map of symbfact.cuh:1084-1099 within a share), so
//   "source j lies above m" is the prefix of slots j < ceil((first-m)/stride).
#include <algorithm>

#include "gsofa_device.h"
#include "gsofa_internal.h"

namespace gsofa {

namespace {

using namespace dev;

// Workgroup shapes (threads, hash slots of the target table; a round takes
// at most half the slots in new targets, so the load stays below 1/2 +
// threads/slots).  16 waves share a CU in each:
//   wide: one 1024-thread workgroup per CU and the largest table that fits
//         the CU's 160 KB of LDS at 64 slots: fewest rounds per level;
//   pair: two 512-thread workgroups per CU with half the table each: one
//         workgroup runs while the other waits at a barrier;
//   quad: four 256-thread workgroups per CU with a quarter of it, where a
//         level's frontier is a few hundred targets and barriers are most of
//         its time.
// reach_shape picks one.
constexpr int NT_WIDE = 1024, NH_WIDE = 11264;
constexpr int NT_PAIR = 512, NH_PAIR = 5632;
constexpr int NT_QUAD = 256, NH_QUAD = 2656;
constexpr uint32_t FULLI = 0xFFFFFFFFu;
constexpr uint32_t PASS_T = 0x80000000u;  // chunk stride bit: the A^T pass
// Lane groups: lanes per vertex and edges per lane and step.  Execute ms with
// (48^3 grid, 128 2D grids, band n = 659,033, 64 slots) at pair 2 x 6: 3.82,
// 25.0, 7.6; 4 x 3: 3.22, 19.7, 6.6; 8 x 2: 2.89, 17.1, 6.4; 16 x 1: 2.92,
// 18.7, 7.2.  At quad 2 x 6: 4.23, 16.0, 6.1; 4 x 3: 3.69, 13.6, 5.7; 8 x 2:
// 3.53, 12.9, 6.0; 16 x 1: 3.58, 15.2, 7.0.  At wide, which runs the few
// groups of small matrices, 4 x 3 takes 0.50 ms on a 64^2 grid, 16 x 1 0.55.
template <int NT>
constexpr int lanes_per_vertex() { return NT == NT_PAIR ? 8 : 4; }
template <int NT>
constexpr int edges_per_lane() { return NT == NT_PAIR ? 2 : 3; }

template <class M>
struct MaskOps;
// Bit helpers shared by the scalar mask types.
template <class M, int B>
struct ScalarBits {
    static __device__ __forceinline__ M bit(uint32_t j) { return (M)1 << j; }
    static __device__ __forceinline__ M prefix(uint32_t c) {  // the low c bits
        return c >= (uint32_t)B ? ~(M)0 : (((M)1 << c) - (M)1);
    }
    static __device__ __forceinline__ M low_clear(M b) { return b & (b - (M)1); }
    template <class F>  // f(j) for every set bit j, in increasing order
    static __device__ __forceinline__ void for_each_bit(M m, F f) {
        if constexpr (B == 128) {
            for (uint64_t b = (uint64_t)m; b; b &= b - 1ull) f((uint32_t)__builtin_ctzll(b));
            for (uint64_t b = (uint64_t)(m >> 64); b; b &= b - 1ull) f(64u + (uint32_t)__builtin_ctzll(b));
        } else {
            for (M b = m; b; b &= b - (M)1) f((uint32_t)(B == 64 ? __builtin_ctzll(b) : __builtin_ctz(b)));
        }
    }
};
template <>
struct MaskOps<uint32_t> : ScalarBits<uint32_t, 32> {
    using V = uint2;  // visited word: (mask, stamp)
    static constexpr int BITS = 32;
    static __device__ __forceinline__ uint32_t get(const V& e, uint32_t st) { return e.y == st ? e.x : 0u; }
    static __device__ __forceinline__ V make(uint32_t m, uint32_t st) { return make_uint2(m, st); }
    static __device__ __forceinline__ uint32_t popc(uint32_t m) { return (uint32_t)__popc(m); }
    static __device__ __forceinline__ uint32_t ctz(uint32_t m) { return (uint32_t)__builtin_ctz(m); }
};
template <>
struct MaskOps<uint64_t> : ScalarBits<uint64_t, 64> {
    using V = uint4;  // visited word: (mask lo, mask hi, stamp, -)
    static constexpr int BITS = 64;
    static __device__ __forceinline__ uint64_t get(const V& e, uint32_t st) {
        return e.z == st ? (((uint64_t)e.y << 32) | e.x) : 0ull;
    }
    static __device__ __forceinline__ V make(uint64_t m, uint32_t st) {
        return make_uint4((uint32_t)m, (uint32_t)(m >> 32), st, 0u);
    }
    static __device__ __forceinline__ uint32_t popc(uint64_t m) { return (uint32_t)__popcll(m); }
    static __device__ __forceinline__ uint32_t ctz(uint64_t m) { return (uint32_t)__builtin_ctzll(m); }
};
typedef unsigned __int128 u128;
struct __align__(16) V128 {  // visited word of 128 slots: mask halves, stamp (32 B)
    uint64_t lo, hi;
    uint32_t stamp, pad[3];
};
template <>
struct MaskOps<u128> : ScalarBits<u128, 128> {
    using V = V128;
    static constexpr int BITS = 128;
    static __device__ __forceinline__ u128 get(const V& e, uint32_t st) {
        return e.stamp == st ? (((u128)e.hi << 64) | e.lo) : (u128)0;
    }
    static __device__ __forceinline__ V make(u128 m, uint32_t st) {
        V v;
        v.lo = (uint64_t)m;
        v.hi = (uint64_t)(m >> 64);
        v.stamp = st;
        v.pad[0] = v.pad[1] = v.pad[2] = 0u;
        return v;
    }
    static __device__ __forceinline__ uint32_t popc(u128 m) {
        return (uint32_t)(__popcll((uint64_t)m) + __popcll((uint64_t)(m >> 64)));
    }
    static __device__ __forceinline__ uint32_t ctz(u128 m) {
        const uint64_t lo = (uint64_t)m;
        return lo ? (uint32_t)__builtin_ctzll(lo) : 64u + (uint32_t)__builtin_ctzll((uint64_t)(m >> 64));
    }
};

// 256 slots: four 64-bit words.
struct M256 {
    uint64_t w[4];
    M256() = default;
    __device__ __forceinline__ constexpr M256(int z) : w{(uint64_t)z, 0ull, 0ull, 0ull} {}
    __device__ __forceinline__ explicit operator bool() const { return (w[0] | w[1] | w[2] | w[3]) != 0ull; }
};
__device__ __forceinline__ M256 operator&(const M256& a, const M256& b) {
    M256 r;
    for (int k = 0; k < 4; k++) r.w[k] = a.w[k] & b.w[k];
    return r;
}
__device__ __forceinline__ M256 operator|(const M256& a, const M256& b) {
    M256 r;
    for (int k = 0; k < 4; k++) r.w[k] = a.w[k] | b.w[k];
    return r;
}
__device__ __forceinline__ M256 operator~(const M256& a) {
    M256 r;
    for (int k = 0; k < 4; k++) r.w[k] = ~a.w[k];
    return r;
}
__device__ __forceinline__ bool operator==(const M256& a, const M256& b) {
    return ((a.w[0] ^ b.w[0]) | (a.w[1] ^ b.w[1]) | (a.w[2] ^ b.w[2]) | (a.w[3] ^ b.w[3])) == 0ull;
}
struct __align__(16) V256 {  // visited word of 256 slots: mask words, stamp (48 B)
    uint64_t w[4];
    uint32_t stamp, pad[3];
};
template <>
struct MaskOps<M256> {
    using V = V256;
    static constexpr int BITS = 256;
    static __device__ __forceinline__ M256 get(const V& e, uint32_t st) {
        M256 r(0);
        if (e.stamp == st)
            for (int k = 0; k < 4; k++) r.w[k] = e.w[k];
        return r;
    }
    static __device__ __forceinline__ V make(const M256& m, uint32_t st) {
        V v;
        for (int k = 0; k < 4; k++) v.w[k] = m.w[k];
        v.stamp = st;
        v.pad[0] = v.pad[1] = v.pad[2] = 0u;
        return v;
    }
    static __device__ __forceinline__ uint32_t popc(const M256& m) {
        return (uint32_t)(__popcll(m.w[0]) + __popcll(m.w[1]) + __popcll(m.w[2]) + __popcll(m.w[3]));
    }
    static __device__ __forceinline__ uint32_t ctz(const M256& m) {
        for (int k = 0; k < 3; k++)
            if (m.w[k]) return 64u * (uint32_t)k + (uint32_t)__builtin_ctzll(m.w[k]);
        return 192u + (uint32_t)__builtin_ctzll(m.w[3]);
    }
    static __device__ __forceinline__ M256 bit(uint32_t j) {
        M256 r(0);
        r.w[j >> 6] = 1ull << (j & 63u);
        return r;
    }
    static __device__ __forceinline__ M256 prefix(uint32_t c) {
        M256 r;
        for (int k = 0; k < 4; k++) {
            const uint32_t lo = 64u * (uint32_t)k;
            r.w[k] = c >= lo + 64u ? ~0ull : c <= lo ? 0ull : ((1ull << (c - lo)) - 1ull);
        }
        return r;
    }
    template <class F>
    static __device__ __forceinline__ void for_each_bit(const M256& m, F f) {
        for (int k = 0; k < 4; k++)
            for (uint64_t b = m.w[k]; b; b &= b - 1ull) f(64u * (uint32_t)k + (uint32_t)__builtin_ctzll(b));
    }
    static __device__ __forceinline__ M256 low_clear(M256 b) {
        for (int k = 0; k < 4; k++)
            if (b.w[k]) {
                b.w[k] &= b.w[k] - 1ull;
                break;
            }
        return b;
    }
};

// 64-bit word k of a mask.
__device__ __forceinline__ uint64_t mask_word(uint32_t m, int) { return m; }
__device__ __forceinline__ uint64_t mask_word(uint64_t m, int) { return m; }
__device__ __forceinline__ uint64_t mask_word(u128 m, int k) { return (uint64_t)(k ? m >> 64 : m); }
__device__ __forceinline__ uint64_t mask_word(const M256& m, int k) { return m.w[k]; }

// OR into an LDS mask (128 and 256 slots: per 64-bit word that has bits).
__device__ __forceinline__ void mask_or(uint32_t* p, uint32_t v) { atomicOr(p, v); }
__device__ __forceinline__ void mask_or(uint64_t* p, uint64_t v) {
    atomicOr(reinterpret_cast<unsigned long long*>(p), (unsigned long long)v);
}
__device__ __forceinline__ void mask_or(u128* p, u128 v) {
    unsigned long long* q = reinterpret_cast<unsigned long long*>(p);
    if ((uint64_t)v) atomicOr(q, (unsigned long long)(uint64_t)v);
    if ((uint64_t)(v >> 64)) atomicOr(q + 1, (unsigned long long)(uint64_t)(v >> 64));
}
__device__ __forceinline__ void mask_or(M256* p, const M256& v) {
    unsigned long long* q = reinterpret_cast<unsigned long long*>(p);
    for (int k = 0; k < 4; k++)
        if (v.w[k]) atomicOr(q + k, (unsigned long long)v.w[k]);
}

// One- and two-word masks (32, 64 slots) merge bits that reach a vertex still
// queued for the current level into that level's mask, so it expands them in
// the same pop: on 3D nested-dissection grids, where a vertex gets bits from
// different sources at neighbouring levels, that halves the traversal.  The
// two masks of a vertex (this level's, the next's) then sit side by side, so
// relax reads both with one access.  Wider masks, whose sources' searches
// mostly advance together (banded matrices), keep the two levels' masks in
// separate arrays and do not merge: the extra reads cost more there.
template <class M>
constexpr bool merges() { return sizeof(M) <= 8; }

// Hash slots of the target table for a shape and mask width: the largest
// table that fits the CU's LDS (4 B key, the mask, 2 B entry per slot).
template <class M>
constexpr int tab_slots(int threads) {
    return sizeof(M) == 32   ? (threads == NT_WIDE ? 4224 : threads == NT_PAIR ? 2048 : 960)
           : sizeof(M) == 16 ? (threads == NT_WIDE ? 7168 : threads == NT_PAIR ? 3584 : 1696)
           : threads == NT_WIDE ? NH_WIDE
           : threads == NT_PAIR ? NH_PAIR
                                : NH_QUAD;
}

// Rows longer than SPLIT_ROW are expanded by SPLIT_PARTS lane groups instead of
// one: the vertex goes to a short LDS list rather than the queue, and the
// level's pops past the queue's end take one part each.  At most SPLIT_MAX
// such vertices per level (any more are queued whole).
constexpr uint32_t SPLIT_ROW = 192, SPLIT_PARTS = 32, SPLIT_MAX = 32;

// A mini-group's nodes, all of them, in LDS (one- and two-word masks): node
// table slots for the space of the target table at 64 slots, at most FT in use.
template <class M>
constexpr int node_slots(int threads) {
    return ((threads == NT_WIDE ? NH_WIDE : threads == NT_PAIR ? NH_PAIR : NH_QUAD) * 14 - 8 * threads) /
           (18 + 2 * (int)sizeof(M)) / WAVE * WAVE;
}
constexpr uint32_t node_room(uint32_t slots) { return slots / 8u * 7u; }  // nodes, at most

// Rows of over two steps are walked in parts, by as many lane groups as there
// are parts: a level of few nodes, as most are once classes stand for the
// vertices, would otherwise last as long as its longest row.
constexpr uint32_t PART_STEPS = 2, PART_ROWS = 64;  // such rows of a level, at most
template <class M, int F, int NT>
struct RNodes {
    M vis[F];                            // sources that have visited the node
    M pend[F];                           // of those, the ones it is still to be expanded for
    uint2 row[F];                        // a queued node's row; at the group's end a bitmap and its prefix
    uint32_t key[F];                     // node + 1; 0 = empty
    uint16_t q[2][F];                    // queues, by level parity
    uint16_t ent[F];                     // slots in use, in the order of insertion
    M pmask[PART_ROWS];                  // masks of this level's rows in parts
    uint32_t plen[2][PART_ROWS];         // edges of a part, by level parity
    uint16_t pnode[2][PART_ROWS];        // their nodes
    uint16_t part[2][NT];                // the parts: (row << 10) | part of it
};

template <class M, int H, int F, int NT>
struct RLds {
    union {
        struct {                         // all zero between rounds but for ent
            uint32_t hkey[H];            // target + 1 (window-local); 0 = empty
            M hmask[H];                  // OR of the masks folded into the target this round
            uint16_t ent[H];             // occupied hash slots in insertion order
        };
        RNodes<M, F, NT> n;                 // vis, pend and key zero between mini-groups
    };
    uint32_t nq[3], ncur[3];             // queue sizes and cursors, by level modulo 3
    uint32_t nrow[3], npart[3];          // rows in parts and parts, likewise
    uint32_t used, over[3];              // nodes in the table; it ran full in a level
    uint32_t s_cnt[MaskOps<M>::BITS];    // A pass: U entries per slot
    uint32_t wsum[16];                   // per-wave sums of a block scan
    uint32_t nup, tmax;                  // vertices above the group reached so far; the largest
    unsigned long long acc[8];           // workgroup totals: fills, checks, -, expansions,
                                         // TE and |R| of the A pass, of the A^T pass
    unsigned long long cte, creach;      // the current mini-group's TE and |R|
    uint32_t qcnt[2];                    // queue sizes, by buffer
    uint32_t cursor[2];                  // pop cursors, by level parity
    uint32_t tcnt[2];                    // inserts of this round, by round parity
    uint32_t held[2];                    // some group holds unfolded edges, by round parity
    uint32_t chunk;
    uint32_t spn[2];                     // split vertices, by level parity
    uint4 sp[2][SPLIT_MAX];              // (vertex, row begin, row end, weight)
    unsigned long long rbase;            // the group's first record
};

// Hash slot of window-local target m, inserting it if new; FULLI when it is
// new and the round already holds T targets.  Linear probing.
template <class M, int H, int F, int NT>
__device__ __forceinline__ uint32_t rtab_find(RLds<M, H, F, NT>& S, uint32_t* tcnt, uint32_t m) {
    constexpr int T = H / 2;
    const uint32_t key = m + 1u;
    uint32_t s = (uint32_t)(((uint64_t)(m * 2654435761u) * (uint32_t)H) >> 32);
    {
        const uint32_t cur = S.hkey[s];  // usual case: present at its first slot
        if (cur == key) return s;
    }
    for (int probe = 0; probe < H; probe++) {
        const uint32_t cur = S.hkey[s];
        if (cur == key) return s;
        if (cur == 0u) {
            if (*tcnt >= (uint32_t)T) return FULLI;
            const uint32_t prev = atomicCAS(&S.hkey[s], 0u, key);
            if (prev == 0u) {
                S.ent[atomicAdd(tcnt, 1u)] = (uint16_t)s;
                return s;
            }
            if (prev == key) return s;
        }
        s = s + 1u == (uint32_t)H ? 0u : s + 1u;
    }
    return FULLI;
}

// Slots j < count whose source first - j*stride lies above global vertex mg.
template <class M>
__device__ __forceinline__ M above_mask(uint32_t mg, uint32_t first, uint32_t stride, uint32_t count) {
    if (mg >= first) return (M)0;
    const uint32_t d = first - mg;
    uint32_t c = stride == 1u ? d : (d + stride - 1u) / stride;
    c = c < count ? c : count;
    return MaskOps<M>::prefix(c);
}

// The calling lane group's bits of a wave ballot (bit k: lane k of the group).
template <int G>
__device__ __forceinline__ uint32_t grp_ballot(bool x, uint32_t grp) {
    return (uint32_t)(__ballot(x) >> (G * grp)) & ((1u << G) - 1u);
}

// The frontier vertex a lane group holds across rounds (group-uniform: every
// lane of the group loads the same queue entry and mask, so no broadcast is
// needed): its slot mask, edge cursor, row end and, per lane, the edges of
// its current step not yet folded.
template <class M>
struct RGrp {
    bool held;           // a vertex is in progress
    bool done;           // the queue is exhausted for this level
    uint32_t pos, end, pend;
    M vm;
};

struct RTally {
    unsigned long long fills, checks, expansions, te, reach;
};

// The mini-group being run: its chunk, matrix window and pass.
struct RCur {
    const int32_t* rp;
    const int32_t* ci;
    uint32_t first, count, stride, mat, wb;
    bool tpass;
    // classes of the vertices below block jb (local vertex below): the group's
    // sources all lie at or above it
    const int32_t* comp;
    const uint4* info;
    uint32_t jb, below, top, shift;
    uint64_t cn;  // stride of the per-level arrays

    __device__ __forceinline__ uint32_t level_of(uint32_t m) const {
        const uint32_t h = 31u - (uint32_t)__builtin_clz((m >> shift) ^ jb);
        return h < top ? h : top;
    }
    // row and (vertices, row lengths) of a node
    __device__ __forceinline__ uint2 row(uint32_t m) const {
        if (m < below) {
            const uint4 in = info[(uint64_t)level_of(m) * cn + wb + m];
            return make_uint2(in.x, in.y);
        }
        return make_uint2((uint32_t)rp[wb + m], (uint32_t)rp[wb + m + 1u]);
    }
    __device__ __forceinline__ uint2 weight(uint32_t m) const {
        if (m < below) {
            const uint4 in = info[(uint64_t)level_of(m) * cn + wb + m];
            return make_uint2(in.z, in.w);
        }
        return make_uint2(1u, (uint32_t)rp[wb + m + 1u] - (uint32_t)rp[wb + m]);
    }
    // the node (local) that stands for local vertex m
    __device__ __forceinline__ uint32_t node(uint32_t m) const {
        return m < below ? (uint32_t)comp[(uint64_t)level_of(m) * cn + wb + m] - wb : m;
    }
};

// Phase A: lane groups of G lanes pop frontier vertices one at a time; a
// step of a group covers the next G*E edges of its vertex, lane j taking
// edges j, j+G, ..., j+(E-1)G of the step (all E loads issued before the
// first fold).  Each target is found or inserted in the table and the
// vertex's mask folded into it, until the queue is exhausted or the table is
// full.  Wave-uniform control flow; the groups hold independent vertices.
template <int H, int F, int G, int E, class M, int NT>
__device__ void rcombine(RLds<M, H, F, NT>& S, RGrp<M>& hv, const RCur& c, M* maskc, const uint4* qc, uint32_t qsize,
                         uint32_t size, const uint4* sp, uint32_t* cursor, uint32_t rb, RTally& t) {
    using O = MaskOps<M>;
    constexpr int T = H / 2;
    const uint32_t lane = __lane_id();
    const uint32_t grp = lane / G;
    const uint32_t j = lane % G;
    constexpr uint32_t ALL = (1u << E) - 1u;  // a lane's edges of one step
    for (;;) {
        const bool want = !hv.held && !hv.done && S.tcnt[rb] < (uint32_t)T;
        const uint64_t wl = __ballot(want && j == 0u);
        uint32_t base = 0;
        if (lane == 0 && wl) base = atomicAdd(cursor, (uint32_t)__popcll(wl));
        base = bcast0(base);
        uint32_t m[E];     // targets of the current step
        bool fresh = false;  // m holds the first step of a vertex just popped
        if (want) {
            const uint32_t idx = base + (uint32_t)__popcll(wl & ((1ull << (G * grp)) - 1ull));
            if (idx >= size) {
                hv.done = true;
            } else {
                uint4 e;
                const bool whole = idx < qsize;
                if (whole) {
                    e = qc[idx];
                } else {  // one part of a split row; the first carries the weight
                    const uint32_t part = (idx - qsize) % SPLIT_PARTS;
                    e = sp[(idx - qsize) / SPLIT_PARTS];
                    const uint32_t len = e.z - e.y;
                    const uint32_t per = ((len + SPLIT_PARTS - 1u) / SPLIT_PARTS + (uint32_t)(G * E) - 1u) /
                                         (uint32_t)(G * E) * (uint32_t)(G * E);
                    const uint32_t o = part * per < len ? part * per : len;
                    e.z = len - o > per ? e.y + o + per : e.z;
                    e.y += o;
                    if (part != 0u) e.w = 0u;
                }
                // the mask and the first step's edges load together
                const M mk = maskc[(merges<M>() ? 2u : 1u) * e.x];
#pragma unroll
                for (int k = 0; k < E; k++) {
                    const uint32_t ek = e.y + j + (uint32_t)(G * k);
                    m[k] = ek < e.z ? (uint32_t)c.ci[ek] - c.wb : FULLI;
                }
#pragma unroll
                for (int k = 0; k < E; k++)
                    if (m[k] != FULLI) m[k] = c.node(m[k]);
                fresh = true;
                hv.pos = e.y;
                hv.end = e.z;
                hv.pend = ALL;
                hv.vm = mk;
                hv.held = e.y < e.z;
                if (j == 0u) {
                    if (whole) maskc[(merges<M>() ? 2u : 1u) * e.x] = (M)0;  // consumed; refilled two levels later
                    t.checks += (unsigned long long)e.w * O::popc(mk);
                    t.expansions++;
                }
            }
        }
        if (!__ballot(hv.held)) {
            // no group holds edges: pop again while the queue and the table allow
            if (__ballot(!hv.done && S.tcnt[rb] < (uint32_t)T)) continue;
            return;
        }
        bool failed = false;
        if (hv.held) {
            if (!fresh) {
#pragma unroll
                for (int k = 0; k < E; k++) {
                    const uint32_t e = hv.pos + j + (uint32_t)(G * k);
                    m[k] = FULLI;
                    if (((hv.pend >> k) & 1u) && e < hv.end) m[k] = (uint32_t)c.ci[e] - c.wb;
                }
#pragma unroll
                for (int k = 0; k < E; k++)
                    if (m[k] != FULLI) m[k] = c.node(m[k]);
            }
            uint32_t left = 0;
#pragma unroll
            for (int k = 0; k < E; k++) {
                if (m[k] != FULLI) {
                    const uint32_t hs = rtab_find(S, &S.tcnt[rb], m[k]);
                    if (hs == FULLI) left |= 1u << k;
                    else mask_or(&S.hmask[hs], hv.vm);
                }
            }
            hv.pend = left;  // the unplaced edges stay for the next round
            failed = left != 0u;
        }
        const uint32_t fm = grp_ballot<G>(failed, grp);
        if (hv.held && !fm) {
            hv.pos += (uint32_t)(G * E);
            hv.pend = ALL;
            hv.held = hv.pos < hv.end;
        }
        if (__ballot(fm != 0u)) return;  // the table is full for everyone
    }
}

// Table slot of node m, inserting it if new; FULLI (and *over set) when the
// table is full.
template <class M, int H, int F, int NT>
__device__ __forceinline__ uint32_t node_find(RLds<M, H, F, NT>& S, uint32_t* over, uint32_t m) {
    constexpr uint32_t FT = node_room((uint32_t)F);
    const uint32_t key = m + 1u;
    uint32_t s = (uint32_t)(((uint64_t)(m * 2654435761u) * (uint32_t)F) >> 32);
    for (int probe = 0; probe < F; probe++) {
        const uint32_t cur = S.n.key[s];
        if (cur == key) return s;
        if (cur == 0u) {
            if (S.used >= FT) break;
            const uint32_t prev = atomicCAS(&S.n.key[s], 0u, key);
            if (prev == 0u) {
                S.n.ent[atomicAdd(&S.used, 1u)] = (uint16_t)s;  // at most F keys are ever inserted
                return s;
            }
            if (prev == key) return s;
        }
        s = s + 1u == (uint32_t)F ? 0u : s + 1u;
    }
    *over = 1u;
    return FULLI;
}

__device__ __forceinline__ uint32_t mask_or_rtn(uint32_t* p, uint32_t v) { return atomicOr(p, v); }
__device__ __forceinline__ uint64_t mask_or_rtn(uint64_t* p, uint64_t v) {
    return atomicOr(reinterpret_cast<unsigned long long*>(p), (unsigned long long)v);
}
__device__ __forceinline__ uint32_t mask_take(uint32_t* p) { return atomicExch(p, 0u); }
__device__ __forceinline__ uint64_t mask_take(uint64_t* p) {
    return atomicExch(reinterpret_cast<unsigned long long*>(p), 0ull);
}

// A mini-group's whole traversal on the node table.  A popped node's bits go
// straight to its targets' visited words; who sets a pending bit of a node with
// none queues it.  So a level is one phase and one barrier and nothing but the
// graph itself is read from memory: edges, their classes, the new nodes' rows.
// If the table ran full: in level 0, the group starts again elsewhere; later, it
// goes on from what the table holds (nodes_to_memory), where every node that the
// level walked is pending again with all its bits, since its edges may be lost.
enum class Walk { DONE, FULL_AT_ONCE, OUTGREW };
template <int RB, int H, int F, int G, int E, class M>
__device__ Walk walk_nodes(RLds<M, H, F, RB>& S, const RCur& c, RTally& t, unsigned long long& levels) {
    using O = MaskOps<M>;
    const uint32_t tid = threadIdx.x, lane = __lane_id();
    const uint32_t grp = lane / G, j = lane % G;
    RTally own{0, 0, 0, 0, 0};
    // a row of over PART edges to level lv's parts; false: no room left
    constexpr uint32_t STEP = (uint32_t)(G * E), PART = PART_STEPS * STEP;
    auto in_parts = [&](uint32_t lv, uint32_t node, uint32_t len, M mask) {
        uint32_t per = (len + RB / 4u - 1u) / (RB / 4u);
        per = per < PART ? PART : (per + STEP - 1u) / STEP * STEP;
        const uint32_t parts = (len + per - 1u) / per, q = lv & 1u;
        const uint32_t r = atomicAdd(&S.nrow[lv % 3u], 1u);
        if (r >= PART_ROWS) return false;
        const uint32_t o = atomicAdd(&S.npart[lv % 3u], parts);
        const bool fits = o + parts <= (uint32_t)RB;
        for (uint32_t k = 0; k < parts && o + k < (uint32_t)RB; k++)
            S.n.part[q][o + k] = fits ? (uint16_t)((r << 10) | k) : (uint16_t)0xFFFF;
        S.n.pnode[q][r] = (uint16_t)(fits ? node : 0xFFFFu);
        S.n.plen[q][r] = per;
        if (mask) S.n.pmask[r] = mask;
        return fits;
    };
    if (tid < 3u) S.nq[tid] = tid == 0 ? c.count : 0u;
    if (tid >= 3u && tid < 6u) S.ncur[tid - 3u] = 0;
    if (tid >= 6u && tid < 9u) S.nrow[tid - 6u] = 0;
    if (tid >= 9u && tid < 12u) S.npart[tid - 9u] = 0;
    if (tid >= 12u && tid < 15u) S.over[tid - 12u] = 0;
    __syncthreads();
    if (tid < c.count) {  // level 0: the sources, each for its own slot
        const uint32_t sg = c.first - tid * c.stride;
        const uint32_t k = node_find(S, &S.over[2], sg - c.wb);  // distinct, and far fewer than slots
        const uint32_t r0 = (uint32_t)c.rp[sg], r1 = (uint32_t)c.rp[sg + 1];
        S.n.vis[k] = O::bit(tid);
        S.n.row[k] = make_uint2(r0, r1);
        S.n.q[0][tid] = (uint16_t)(r1 - r0 > PART && in_parts(0u, k, r1 - r0, O::bit(tid)) ? 0xFFFFu : k);
        own.te = r1 - r0;
    }
    uint32_t lev = 0;
    bool full;
    for (;; lev++) {
        __syncthreads();
        const uint32_t b = lev % 3u, nb = (lev + 1u) % 3u;
        const uint32_t qsize = S.nq[b], nrow = S.nrow[b] < PART_ROWS ? S.nrow[b] : PART_ROWS;
        const uint32_t size = qsize + (S.npart[b] < (uint32_t)RB ? S.npart[b] : (uint32_t)RB);
        full = S.over[(lev + 2u) % 3u] != 0u;  // in the level before: this one's flag may be set by now
        if (size == 0u || full) break;
        if (tid == 0) {  // the counters of the level after the next: last read a barrier ago
            const uint32_t z = (lev + 2u) % 3u;
            S.nq[z] = S.ncur[z] = S.nrow[z] = S.npart[z] = 0;
        }
        const uint16_t* qc = S.n.q[lev & 1u];
        uint16_t* qn = S.n.q[(lev + 1u) & 1u];
        const uint32_t par = lev & 1u;
        if (nrow && lev) {
            if (tid < nrow && S.n.pnode[par][tid] != 0xFFFFu) S.n.pmask[tid] = mask_take(&S.n.pend[S.n.pnode[par][tid]]);
            __syncthreads();
        }
        bool held = false, done = false;
        uint32_t pos = 0, end = 0;
        M vm = (M)0;
        for (;;) {
            const bool want = !held && !done;
            const uint64_t wl = __ballot(want && j == 0u);
            if (wl) {
                uint32_t base = 0;
                if (lane == 0) base = atomicAdd(&S.ncur[b], (uint32_t)__popcll(wl));
                base = bcast0(base);
                if (want) {
                    const uint32_t idx = base + (uint32_t)__popcll(wl & ((1ull << (G * grp)) - 1ull));
                    if (idx >= size) {
                        done = true;
                    } else if (idx < qsize) {
                        const uint32_t k = qc[idx];
                        if (k != 0xFFFFu) {  // not one that is walked in parts
                            const uint2 r = S.n.row[k];
                            pos = r.x;
                            end = r.y;
                            M m = (M)0;
                            if (j == 0u) m = lev ? mask_take(&S.n.pend[k]) : O::bit(idx);
                            vm = __shfl(m, 0, G);
                            held = pos < end;
                            if (j == 0u) own.expansions++;
                        }
                    } else {
                        const uint32_t x = S.n.part[par][idx - qsize];
                        if (x != 0xFFFFu) {
                            const uint32_t per = S.n.plen[par][x >> 10];
                            const uint2 r = S.n.row[S.n.pnode[par][x >> 10]];
                            pos = r.x + (x & 1023u) * per;
                            end = r.y - pos > per ? pos + per : r.y;
                            vm = S.n.pmask[x >> 10];
                            held = true;
                            if ((x & 1023u) == 0u && j == 0u) own.expansions++;
                        }
                    }
                }
            }
            if (!__ballot(held)) {
                if (__ballot(!done)) continue;
                break;
            }
            // one step of every group that holds a node
            uint32_t m[E];
#pragma unroll
            for (int k = 0; k < E; k++) {
                const uint32_t ek = pos + j + (uint32_t)(G * k);
                m[k] = held && ek < end ? (uint32_t)c.ci[ek] - c.wb : FULLI;
            }
#pragma unroll
            for (int k = 0; k < E; k++)
                if (m[k] != FULLI) m[k] = c.node(m[k]);
            uint32_t push[E];
            uint2 row[E];
#pragma unroll
            for (int k = 0; k < E; k++) {
                push[k] = FULLI;
                if (m[k] == FULLI) continue;
                const uint32_t sl = node_find(S, &S.over[b], m[k]);
                if (sl == FULLI) continue;
                M nw = vm & ~S.n.vis[sl];
                if (!nw) continue;
                nw = nw & ~mask_or_rtn(&S.n.vis[sl], nw);
                if (!nw) continue;
                const M bl = nw & above_mask<M>(m[k] + c.wb, c.first, c.stride, c.count);
                if (lev) own.fills += O::popc(nw & ~bl);
                if (bl && !mask_or_rtn(&S.n.pend[sl], bl)) push[k] = sl;
            }
#pragma unroll
            for (int k = 0; k < E; k++)
                if (push[k] != FULLI) row[k] = c.row(m[k]);
#pragma unroll
            for (int k = 0; k < E; k++) {
                bool enq = push[k] != FULLI;
                if (enq) {
                    S.n.row[push[k]] = row[k];
                    const uint32_t len = row[k].y - row[k].x;
                    if (len > PART && in_parts(lev + 1u, push[k], len, (M)0)) enq = false;
                }
                const uint64_t em = __ballot(enq);
                if (em) {
                    uint32_t qb = 0;
                    if (lane == 0) qb = atomicAdd(&S.nq[nb], (uint32_t)__popcll(em));
                    qb = bcast0(qb);
                    if (enq) qn[qb + rank_in(em)] = (uint16_t)push[k];
                }
            }
            if (held) {
                pos += (uint32_t)(G * E);
                held = pos < end;
            }
        }
    }
    if (full && lev < 2u) return Walk::FULL_AT_ONCE;
    t.fills += own.fills;
    t.expansions += own.expansions;
    t.te += own.te;
    t.checks += own.te;
    levels += tid == 0 ? lev : 0u;
    if (full) {
        const uint32_t b = (lev + 2u) % 3u, par = (lev + 1u) & 1u, qsize = S.nq[b];
        const uint32_t nrow = S.nrow[b] < PART_ROWS ? S.nrow[b] : PART_ROWS;
        for (uint32_t x = tid; x < qsize + nrow; x += RB) {  // a node is in the queue or in parts
            const uint32_t k = x < qsize ? S.n.q[par][x] : S.n.pnode[par][x - qsize];
            if (k != 0xFFFFu)
                S.n.pend[k] |= S.n.vis[k] & above_mask<M>(S.n.key[k] - 1u + c.wb, c.first, c.stride, c.count);
        }
        __syncthreads();
        return Walk::OUTGREW;
    }
    // TE and |R|: every node below a source that visited it, with its weights
    const uint32_t fl = c.first - c.wb, used = S.used;
    for (uint32_t x = tid; x < used; x += RB) {
        const uint32_t i = S.n.ent[x], m = S.n.key[i] - 1u;
        if (m > fl) continue;
        const M bl = S.n.vis[i] & above_mask<M>(m + c.wb, c.first, c.stride, c.count);
        if (!bl) continue;
        const uint2 w = c.weight(m);
        t.reach += (unsigned long long)O::popc(bl) * w.x;
        t.te += (unsigned long long)O::popc(bl) * w.y;
        t.checks += (unsigned long long)O::popc(bl) * w.y;  // every node once for every source that visits it
    }
    return Walk::DONE;
}

// A group that outgrew its table goes on in memory: its nodes' visited words, the
// pending ones as level `cur` = 0's queue, those above the group on their list.
// Starting it again there instead walked up to the whole group twice.  Traversal
// ms again -> on (before there was a table): directed cycle of 5,000 19.1 -> 12.1
// (12.2), one-directional band of 60,000 with 2,000 entries back 6.9 -> 4.9 (4.5),
// hubs n = 8,000 2.06 -> 1.76 (6.2), 48^3 grid 1.44 -> 1.33.
template <int RB, int H, int F, class M>
__device__ void nodes_to_memory(RLds<M, H, F, RB>& S, const RCur& c, typename MaskOps<M>::V* vis, M* nmask0, uint4* q0,
                                uint32_t* ulist, uint32_t stamp, RTally& t) {
    using O = MaskOps<M>;
    static_assert(merges<M>(), "masks side by side");
    const uint32_t lane = __lane_id(), fl = c.first - c.wb, used = S.used;
    for (uint32_t x0 = threadIdx.x - lane; x0 < used; x0 += RB) {
        bool up = false, enq = false;
        uint32_t m = 0;
        uint4 e = make_uint4(0u, 0u, 0u, 0u);
        if (x0 + lane < used) {
            const uint32_t i = S.n.ent[x0 + lane];
            m = S.n.key[i] - 1u;
            const M v = S.n.vis[i], pd = S.n.pend[i];
            vis[m] = O::make(v, stamp);
            const M bl = v & above_mask<M>(m + c.wb, c.first, c.stride, c.count);
            up = m > fl;
            if (bl) {
                const uint2 w = c.weight(m);
                t.reach += (unsigned long long)O::popc(bl) * w.x;
                t.te += (unsigned long long)O::popc(bl) * w.y;
                t.checks += (unsigned long long)O::popc(bl & ~pd) * w.y;
                if (pd) {
                    const uint2 r = S.n.row[i];
                    nmask0[2u * m] = pd;
                    e = make_uint4(m, r.x, r.y, w.y);
                    enq = true;
                    if (r.y - r.x > SPLIT_ROW) {
                        const uint32_t k = atomicAdd(&S.spn[0], 1u);
                        if (k < SPLIT_MAX) {
                            S.sp[0][k] = e;
                            enq = false;
                        }
                    }
                }
            }
        }
        const uint64_t em = __ballot(enq), um = __ballot(up);
        if (em) {
            uint32_t qb = 0;
            if (lane == 0) qb = atomicAdd(&S.qcnt[0], (uint32_t)__popcll(em));
            qb = bcast0(qb);
            if (enq) q0[qb + rank_in(em)] = e;
        }
        if (um) {
            uint32_t ub = 0;
            if (lane == 0) ub = atomicAdd(&S.nup, (uint32_t)__popcll(um));
            ub = bcast0(ub);
            if (up) {
                ulist[ub + rank_in(um)] = m;
                atomicMax(&S.tmax, m);
            }
        }
    }
}

// The group's entries from the node table, which is cleared: records in order
// of the vertex by ranks in an LDS bitmap over the vertices above the group,
// a window of 32 F of them at a time; counts per row.
template <int RB, int H, int F, class M>
__device__ void emit_nodes(RLds<M, H, F, RB>& S, const RCur& c, const RchParams& p, uint32_t ck) {
    using O = MaskOps<M>;
    static_assert(sizeof(M) <= 8, "one record word");
    const uint32_t tid = threadIdx.x, lane = __lane_id(), w = tid / WAVE;
    const uint32_t fl = c.first - c.wb, lo = fl - (c.count - 1u), used = S.used;
    const bool rec = p.rec_cap != 0ull;
    uint32_t* bm = reinterpret_cast<uint32_t*>(S.n.row);
    uint32_t* before = bm + F;
    uint32_t nup = 0, top = 0;
    for (uint32_t x = tid; x < used; x += RB) {
        const uint32_t m = S.n.key[S.n.ent[x]] - 1u;
        if (m <= fl) continue;
        nup++;
        top = m > top ? m : top;
    }
    nup = dev::wave_incl_scan(nup);
#pragma unroll
    for (int d = 1; d < WAVE; d <<= 1) {
        const uint32_t o = __shfl_xor(top, d, WAVE);
        top = o > top ? o : top;
    }
    if (lane == WAVE - 1 && nup) {
        atomicAdd(&S.nup, nup);
        atomicMax(&S.tmax, top);
    }
    __syncthreads();
    const uint32_t items = c.count + S.nup;
    const uint32_t all = rec && S.nup ? ((S.tmax - fl - 1u) >> 5) + 1u : 0u;
    if (rec && tid == 0) {
        const unsigned long long o = aadd64(&p.ctrl->fill_pos, (unsigned long long)items);
        const bool fits = o + (unsigned long long)items <= p.rec_cap;
        S.rbase = fits ? o : ~0ull;
        p.grp[ck] = make_uint4((uint32_t)o, (uint32_t)(o >> 32), fits ? items : 0u, 0u);
    }
    uint32_t acc = 0, sorted = c.count;
    for (uint32_t w0 = 0; w0 == 0u || w0 < all; w0 += F) {
        const uint32_t nw = all - w0 < (uint32_t)F ? all - w0 : (uint32_t)F;
        if (rec) {
            for (uint32_t i = tid; i < nw; i += RB) bm[i] = 0u;
            __syncthreads();
            for (uint32_t x = tid; x < used; x += RB) {
                const uint32_t m = S.n.key[S.n.ent[x]] - 1u, o = m - fl - 1u;
                if (m > fl && (o >> 5) - w0 < nw) atomicOr(&bm[(o >> 5) - w0], 1u << (o & 31u));
            }
            __syncthreads();
            const uint32_t per = (nw + RB - 1u) / RB;
            const uint32_t b0 = tid * per < nw ? tid * per : nw;
            const uint32_t b1 = b0 + per < nw ? b0 + per : nw;
            uint32_t cnt = 0;
            for (uint32_t b = b0; b < b1; b++) cnt += (uint32_t)__popc(bm[b]);
            const uint32_t incl = wave_incl_scan(cnt);
            if (lane == WAVE - 1) S.wsum[w] = incl;
            __syncthreads();
            uint32_t pos = sorted + incl - cnt;
            for (uint32_t k = 0; k < (uint32_t)(RB / WAVE); k++) {
                if (k < w) pos += S.wsum[k];
                sorted += S.wsum[k];
            }
            for (uint32_t b = b0; b < b1; b++) {
                before[b] = pos;
                pos += (uint32_t)__popc(bm[b]);
            }
            __syncthreads();
        }
        const uint64_t r0 = rec ? S.rbase : ~0ull;
        for (uint32_t x0 = w * WAVE; x0 < used; x0 += RB) {
            const uint32_t i = x0 + lane < used ? S.n.ent[x0 + lane] : 0u;
            const uint32_t m = x0 + lane < used ? S.n.key[i] - 1u : 0u, o = m - fl - 1u;
            bool in = false;
            uint32_t at = 0;
            M mk = (M)0;
            if (m > fl) {
                in = !rec || (o >> 5) - w0 < nw;
                if (in) {
                    mk = S.n.vis[i];
                    if (rec) at = before[(o >> 5) - w0] + (uint32_t)__popc(bm[(o >> 5) - w0] & ((1u << (o & 31u)) - 1u));
                }
            } else if (x0 + lane < used && m >= lo && w0 == 0u) {
                in = true;
                at = m - lo;
                mk = S.n.vis[i] & ~O::prefix(c.count - at);  // sources below the vertex
            }
            const uint64_t wd = mask_word(mk, 0);
            if (in && r0 != ~0ull) p.rec[r0 + at] = make_uint4(c.wb + m, c.first, (uint32_t)wd, (uint32_t)(wd >> 32));
            if (!__ballot(wd != 0ull)) continue;
            if (c.tpass) {
                if (wd) aadd64(&p.cntL[c.wb + m], (1ull << 32) | (unsigned long long)__popcll(wd));
            } else {
#pragma unroll
                for (int j = 0; j < O::BITS; j++) {
                    const uint32_t n = (uint32_t)__popcll(__ballot((wd >> j) & 1ull));
                    if (lane == (uint32_t)j) acc += n;
                }
            }
        }
        __syncthreads();  // the window's ranks are read
    }
    if (!c.tpass && acc) atomicAdd(&S.s_cnt[lane], acc);
    for (uint32_t x = tid; x < used; x += RB) {
        const uint32_t i = S.n.ent[x];
        S.n.key[i] = 0u;
        S.n.vis[i] = S.n.pend[i] = (M)0;
    }
    __syncthreads();
    if (tid == 0) S.used = 0;
    if (!c.tpass && tid < c.count) p.cntU[c.first - tid * c.stride] = S.s_cnt[tid];
}

template <int RB, int H, int F, int G, int E, class M>
__global__ __launch_bounds__(RB, sizeof(M) <= 16 ? 4 : 1) void k_reach_blk(RchParams p) {
    static_assert(H / 2 + RB <= H, "insert overshoot stays within the entry list");
    static_assert(H <= 65536, "entries are 16-bit slot numbers");
    static_assert(WAVE % G == 0 && G < 32 && E >= 1 && E < 32, "lane groups tile a wave; a lane's edges fit its pending bits");
    using O = MaskOps<M>;
    using VW = typename O::V;
    using Lds = RLds<M, H, F, RB>;
    __shared__ Lds S;
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = __lane_id();
    const uint32_t w = tid / WAVE;
    const uint32_t W = p.W;
    VW* vis = reinterpret_cast<VW*>(p.vis) + (uint64_t)blockIdx.x * W;
    M* nmask0 = reinterpret_cast<M*>(p.nmask) + (uint64_t)blockIdx.x * 2 * W;
    uint4* q0 = p.q + (uint64_t)blockIdx.x * 2 * W;
    uint32_t epoch = p.bstate[blockIdx.x];
    RTally t{0, 0, 0, 0, 0};
    unsigned long long levels = 0;
    constexpr bool NODES = sizeof(M) <= 8;
    constexpr uint32_t TAB_WORDS = (uint32_t)(offsetof(Lds, nq) / 4);
    auto clear_tables = [&] {
        for (uint32_t i = tid; i < TAB_WORDS; i += RB) reinterpret_cast<uint32_t*>(&S)[i] = 0u;
    };
    uint32_t wait = 0;  // mini-groups to go before the node table is tried again
    clear_tables();
    if (tid == 0) S.used = 0;
    if (tid < 8) S.acc[tid] = 0;
    if (tid == 0) {
        S.qcnt[0] = S.qcnt[1] = 0;
        S.tcnt[0] = S.tcnt[1] = S.held[0] = S.held[1] = 0;
        S.spn[0] = S.spn[1] = 0;
    }
    uint32_t rb = 0;  // round parity
    const bool classes = p.quot.levels != 0u && !quot_off(p.quot);
    for (;;) {
        if (tid == 0) {
            S.chunk = atomicAdd(&p.ctrl->src_next, 1u);
            S.cte = S.creach = 0;
            S.cursor[0] = S.cursor[1] = 0;
            S.nup = S.tmax = 0;
        }
        if (tid < (uint32_t)O::BITS) S.s_cnt[tid] = 0;
        __syncthreads();
        const uint32_t ck = S.chunk;
        if (ck >= p.n_chunks) break;
        const BlkChunk C = p.chunks[ck];
        RCur c;
        c.tpass = (C.stride & PASS_T) != 0u;
        c.rp = c.tpass ? p.rpT : p.rp;
        c.ci = c.tpass ? p.ciT : p.ci;
        c.first = C.first;
        c.count = C.count;
        c.stride = C.stride & ~PASS_T;
        c.mat = C.mat;
        c.wb = p.mat_base[C.mat];
        c.comp = p.quot.comp;
        c.info = c.tpass ? p.quot.infoT : p.quot.info;
        c.cn = p.quot.n;
        c.top = p.quot.levels - 1u;
        c.shift = p.quot.shift;
        c.jb = classes ? (c.first - (c.count - 1u) * c.stride - c.wb) >> c.shift : 0u;
        c.below = c.jb << c.shift;
        bool nodes = false;  // the node table holds the whole group
        bool part = false;   // or its first levels
        if constexpr (NODES) {
            if (wait == 0u) {
                const Walk r = walk_nodes<RB, H, F, G, E, M>(S, c, t, levels);
                nodes = r == Walk::DONE;
                part = r == Walk::OUTGREW;
                if (!nodes) wait = 8u;  // the sizes of neighbouring groups are alike
            }
        }
        // No vertex above the group is ever queued, so the queue arrays' entries
        // past the group's largest source hold the list of those reached (in
        // the first array) and its sorted copy (in the second).
        const uint32_t fl = c.first - c.wb;
        uint32_t* const ulist = reinterpret_cast<uint32_t*>(q0 + fl + 1u);
        uint32_t* const slist = reinterpret_cast<uint32_t*>(q0 + W + fl + 1u);
        uint32_t stamp = 0;
        if (!nodes) {
        if (epoch >= p.loops) {  // stamps exhausted: clear this workgroup's visited words
            for (uint32_t i = tid; i < W; i += RB) vis[i] = O::make((M)0, 0u);
            epoch = 0;
            __syncthreads();  // cleared before the sources are stamped
        }
        epoch++;
        stamp = epoch;
        if constexpr (NODES) {
            if (wait == 8u) {  // the table is left
                if (part) nodes_to_memory<RB>(S, c, vis, nmask0, q0, ulist, stamp, t);
                __syncthreads();
                clear_tables();
                if (tid == 0) S.used = 0;
                __syncthreads();
            }
        }
        // level 0: the sources themselves, each visited by and queued for its own slot
        if (!part && tid < c.count) {
            const uint32_t sg = c.first - tid * c.stride;
            const uint32_t s = sg - c.wb;
            const M bit = O::bit(tid);
            vis[s] = O::make(bit, stamp);
            nmask0[(merges<M>() ? 2u : 1u) * s] = bit;  // level 0 uses the first mask
            const uint32_t r0 = (uint32_t)c.rp[sg], r1 = (uint32_t)c.rp[sg + 1];
            q0[tid] = make_uint4(s, r0, r1, r1 - r0);
            t.te += r1 - r0;
        }
        if (!part && tid == 0) S.qcnt[0] = c.count;
        __syncthreads();

        uint32_t cur = 0;
        for (uint32_t lev = part ? 2u : 0u;; lev++) {  // level 0 alone is told apart; cur is its parity
            // final since the last barrier; reset during this level's relax
            const uint32_t nxt = cur ^ 1u;
            const uint32_t qsize = S.qcnt[cur];
            const uint32_t nsp = S.spn[cur] < SPLIT_MAX ? S.spn[cur] : SPLIT_MAX;
            const uint32_t size = qsize + SPLIT_PARTS * nsp;
            // the previous level's split vertices: no part is left, so their
            // masks are cleared here, before this level's relax fills that array
            if (w == 0) {
                const uint32_t done = S.spn[nxt] < SPLIT_MAX ? S.spn[nxt] : SPLIT_MAX;
                if (tid < done)
                    nmask0[merges<M>() ? 2ull * S.sp[nxt][tid].x + nxt : (uint64_t)nxt * W + S.sp[nxt][tid].x] = (M)0;
                wave_sync();
                if (tid == 0) S.spn[nxt] = 0;
            }
            if (size == 0) break;
            // this level's and the next level's masks: side by side per vertex
            // (merging widths, index 2v) or two arrays (index v)
            constexpr uint32_t MS = merges<M>() ? 2u : 1u;
            M* maskc = nmask0 + (merges<M>() ? (uint64_t)cur : (uint64_t)cur * W);
            M* maskn = nmask0 + (merges<M>() ? (uint64_t)nxt : (uint64_t)nxt * W);
            const uint4* qc = q0 + (uint64_t)cur * W;
            uint4* qn = q0 + (uint64_t)nxt * W;
            uint32_t* cursor = &S.cursor[lev & 1u];
            RGrp<M> hv;
            hv.held = false;
            hv.done = false;
            hv.pend = 0u;
            hv.pos = hv.end = 0u;
            hv.vm = (M)0;
            for (;;) {  // rounds, two barriers each
                rcombine<H, F, G, E, M>(S, hv, c, maskc, qc, qsize, size, S.sp[cur], cursor, rb, t);
                if (hv.held && (lane % G) == 0u) atomicOr(&S.held[rb], 1u);
                __syncthreads();
                // final for this round: the cursor moves only in phase A
                const bool more = S.held[rb] != 0u || *cursor < size;
                // ---- B. relax: one lane per table entry
                const uint32_t tc = S.tcnt[rb];
                const uint32_t ntab = tc < (uint32_t)H ? tc : (uint32_t)H;
                for (uint32_t b0 = w * WAVE; b0 < ntab; b0 += RB) {
                    const uint32_t i = b0 + lane;
                    const bool ok = i < ntab;
                    uint32_t m = 0;
                    M mk = (M)0;
                    if (ok) {
                        const uint32_t hs = S.ent[i];
                        m = S.hkey[hs] - 1u;
                        mk = S.hmask[hs];
                        S.hkey[hs] = 0u;
                        S.hmask[hs] = (M)0;
                    }
                    const uint32_t mg = m + c.wb;
                    M up = (M)0;
                    uint32_t r0 = 0, r1 = 0, wt = 0;
                    bool enq = false, above = false;
                    if (ok) {
                        const VW vw = vis[m];
                        const M mc = merges<M>() ? maskc[MS * m] : (M)0;
                        const M mn = maskn[MS * m];
                        uint32_t vc = 1;  // vertices of the node
                        if (m < c.below) {
                            const uint4 in = c.info[(uint64_t)c.level_of(m) * c.cn + mg];
                            r0 = in.x;
                            r1 = in.y;
                            vc = in.z;
                            wt = in.w;
                        } else {
                            r0 = (uint32_t)c.rp[mg];
                            r1 = (uint32_t)c.rp[mg + 1];
                            wt = r1 - r0;
                        }
                        const M vv = O::get(vw, stamp);
                        const M nw = mk & ~vv;
                        if (nw) {
                            vis[m] = O::make(vv | nw, stamp);
                            const M bl = nw & above_mask<M>(mg, c.first, c.stride, c.count);
                            up = lev ? (nw & ~bl) : (M)0;  // level 0: A's own entries
                            above = m > fl && !vv;
                            if (bl) {
                                if (merges<M>() && lev != 0u && mc && r1 - r0 <= SPLIT_ROW) {
                                    // still queued for this level and not yet
                                    // popped: it expands these bits too, one
                                    // expansion fewer (not at level 0, whose
                                    // edges are A's own entries of the sources)
                                    maskc[MS * m] = mc | bl;
                                } else {
                                    maskn[MS * m] = mn | bl;
                                    enq = mn == (M)0;
                                }
                                const uint32_t nb = O::popc(bl);
                                t.reach += (unsigned long long)nb * vc;
                                t.te += (unsigned long long)nb * wt;
                                if (enq && r1 - r0 > SPLIT_ROW) {
                                    const uint32_t k = atomicAdd(&S.spn[nxt], 1u);
                                    if (k < SPLIT_MAX) {
                                        S.sp[nxt][k] = make_uint4(m, r0, r1, wt);
                                        enq = false;
                                    }
                                }
                            }
                        }
                    }
                    const uint64_t em = __ballot(enq);
                    if (em) {
                        uint32_t qb = 0;
                        if (lane == 0) qb = atomicAdd(&S.qcnt[nxt], (uint32_t)__popcll(em));
                        qb = bcast0(qb);
                        if (enq) qn[qb + rank_in(em)] = make_uint4(m, r0, r1, wt);
                    }
                    t.fills += O::popc(up);
                    const uint64_t um = __ballot(above);
                    if (um) {
                        uint32_t ub = 0;
                        if (lane == 0) ub = atomicAdd(&S.nup, (uint32_t)__popcll(um));
                        ub = bcast0(ub);
                        if (above) {
                            ulist[ub + rank_in(um)] = m;
                            atomicMax(&S.tmax, m);
                        }
                    }
                }
                // counters of the next round, the consumed queue and the next
                // level's cursor, cleared while others still relax: each was
                // last read before this round's first barrier
                if (tid == 0) {
                    S.tcnt[rb ^ 1u] = 0;
                    S.held[rb ^ 1u] = 0;
                    S.qcnt[cur] = 0;
                    S.cursor[(lev + 1u) & 1u] = 0;
                }
                __syncthreads();
                rb ^= 1u;
                if (!more) break;
            }
            cur = nxt;
            levels++;
        }
        }
        // the mini-group's TE and |R| (per matrix for the A pass); counts-only
        // fills per source row
        const unsigned long long te = wave_sum64(t.te), rc = wave_sum64(t.reach);
        if (lane == 0 && (te | rc)) {
            atomicAdd(&S.cte, te);
            atomicAdd(&S.creach, rc);
        }
        t.te = t.reach = 0;
        __syncthreads();
        if (tid == 0) {
            atomicAdd(&S.acc[c.tpass ? 6 : 4], S.cte);
            atomicAdd(&S.acc[c.tpass ? 7 : 5], S.creach);
            if (!c.tpass && p.mat_te) {
                aadd64(&p.mat_te[c.mat], S.cte);
                aadd64(&p.mat_reach[c.mat], S.creach);
            }
        }
        if constexpr (NODES) {
            if (nodes) {
                emit_nodes<RB, H, F, M>(S, c, p, ck);
                continue;
            }
        }
        // ---- the group's entries, from the final visited words: items are the
        // group's own vertices in increasing order, then those above it
        constexpr int NW = O::BITS > 64 ? O::BITS / 64 : 1;
        const uint32_t nup = S.nup, items = c.count + nup;
        const bool rec = p.rec_cap != 0ull;
        if (rec) {
            // sorted by LDS bitmap windows over the vertices from fl + 1 on
            // (the target table's masks, all zero between rounds)
            uint32_t* bm = reinterpret_cast<uint32_t*>(S.hmask);
            constexpr uint32_t BW = (uint32_t)(H * sizeof(M) / 4);
            const uint32_t all = nup ? ((S.tmax - fl - 1u) >> 5) + 1u : 0u;
            uint32_t sorted = 0;
            for (uint32_t w0 = 0; w0 < all; w0 += BW) {
                const uint32_t nw = all - w0 < BW ? all - w0 : BW;
                for (uint32_t i = tid; i < nup; i += RB) {
                    const uint32_t o = ulist[i] - fl - 1u;
                    if ((o >> 5) - w0 < nw) atomicOr(&bm[(o >> 5) - w0], 1u << (o & 31u));
                }
                __syncthreads();
                const uint32_t per = (nw + RB - 1u) / RB;
                const uint32_t b0 = tid * per < nw ? tid * per : nw;
                const uint32_t b1 = b0 + per < nw ? b0 + per : nw;
                uint32_t cnt = 0;
                for (uint32_t b = b0; b < b1; b++) cnt += (uint32_t)__popc(bm[b]);
                const uint32_t incl = wave_incl_scan(cnt);
                if (lane == WAVE - 1) S.wsum[w] = incl;
                __syncthreads();
                uint32_t pos = sorted + incl - cnt;
                for (uint32_t k = 0; k < (uint32_t)(RB / WAVE); k++) {
                    if (k < w) pos += S.wsum[k];
                    sorted += S.wsum[k];
                }
                for (uint32_t b = b0; b < b1; b++) {
                    for (uint32_t x = bm[b]; x; x &= x - 1u)
                        slist[pos++] = fl + 1u + ((w0 + b) << 5) + (uint32_t)__builtin_ctz(x);
                    bm[b] = 0u;
                }
                __syncthreads();
            }
            if (tid == 0) {
                const unsigned long long o = aadd64(&p.ctrl->fill_pos, (unsigned long long)NW * items);
                const bool fits = o + (unsigned long long)NW * items <= p.rec_cap;
                S.rbase = fits ? o : ~0ull;
                p.grp[ck] = make_uint4((uint32_t)o, (uint32_t)(o >> 32), fits ? items : 0u, 0u);
            }
            __syncthreads();
        }
        const uint64_t r0 = rec ? S.rbase : ~0ull;
        const uint32_t* up_list = rec ? slist : ulist;
        uint32_t acc[NW] = {};
        for (uint32_t i0 = w * WAVE; i0 < items; i0 += RB) {
            const uint32_t i = i0 + lane;
            uint32_t m = 0;
            M mk = (M)0;
            if (i < items) {
                m = i < c.count ? fl - (c.count - 1u - i) : up_list[i - c.count];
                mk = O::get(vis[m], stamp);
                if (i < c.count) mk = mk & ~O::prefix(c.count - i);  // sources below the vertex
            }
#pragma unroll
            for (int k = 0; k < NW; k++) {
                const uint64_t wd = mask_word(mk, k);
                if (i < items) {
                    if (r0 != ~0ull)
                        p.rec[r0 + (uint64_t)k * items + i] =
                            make_uint4(c.wb + m, c.first - 64u * (uint32_t)k, (uint32_t)wd, (uint32_t)(wd >> 32));
                    if (c.tpass && wd) aadd64(&p.cntL[c.wb + m], (1ull << 32) | (unsigned long long)__popcll(wd));
                }
                if (!c.tpass) {
#pragma unroll
                    for (int j = 0; j < (O::BITS < 64 ? O::BITS : 64); j++) {
                        const uint32_t n = (uint32_t)__popcll(__ballot((wd >> j) & 1ull));
                        if (lane == (uint32_t)j) acc[k] += n;
                    }
                }
            }
        }
        if (!c.tpass) {
#pragma unroll
            for (int k = 0; k < NW; k++)
                if (acc[k]) atomicAdd(&S.s_cnt[64 * k + (int)lane], acc[k]);
            __syncthreads();
            if (tid < c.count) p.cntU[c.first - tid * c.stride] = S.s_cnt[tid];
        }
        __syncthreads();
        if (NODES && wait && --wait == 0u) {
            clear_tables();
            __syncthreads();
        }
    }
    if (t.fills) atomicAdd(&S.acc[0], t.fills);
    if (t.checks) atomicAdd(&S.acc[1], t.checks);
    if (t.expansions) atomicAdd(&S.acc[3], t.expansions);
    __syncthreads();
    if (tid == 0) {
        Ctrl* ct = p.ctrl;
        if (S.acc[0]) aadd64(&ct->fill_count, S.acc[0]);
        if (S.acc[1]) aadd64(&ct->edge_checks, S.acc[1]);
        if (S.acc[3]) aadd64(&ct->expansions, S.acc[3]);
        if (S.acc[4]) aadd64(&ct->te, S.acc[4]);
        if (S.acc[5]) aadd64(&ct->reach, S.acc[5]);
        if (S.acc[6]) aadd64(&ct->te_t, S.acc[6]);
        if (S.acc[7]) aadd64(&ct->reach_t, S.acc[7]);
        aadd64(&ct->levels, levels);
        p.bstate[blockIdx.x] = epoch;
    }
}

}  // namespace

bool rch_bits_valid(int bits) { return bits == 32 || bits == 64 || bits == 128 || bits == 256; }
bool rch_threads_valid(int threads) { return threads == NT_WIDE || threads == NT_PAIR; }

bool rch_shape_valid(int threads) { return rch_threads_valid(threads) || threads == NT_QUAD; }

// The shape for `chunks` mini-groups (both passes) of matrices of up to W
// vertices, whose groups reach `reach` vertices at or above themselves on
// average (from the record bound) and the largest of them `largest`, on `cus`
// CUs:
//   quad  where several mini-groups queue per CU and they are narrow;
//   wide  where the largest group's nodes fit only its table;
//   pair  otherwise.
// With 128 and 256 slots, which use no node table, wide while every mini-group
// has a CU of its own.  More workgroups hold more per-vertex arrays, so a shape
// is taken only while those stay within `room` bytes (quad 8 GiB, pair half the
// room and 32 GiB); pair's 256-slot kernel has registers for one workgroup per
// CU.  Execute ms at 64 slots, wide / pair / quad where taken: 16^2 grid 0.162 /
// 0.156; 64^2 grid 0.346 / 0.332; band n = 11,948 0.32 / 0.30; 181^2 grid 0.77 /
// 0.64; 33^3 grid (largest group about 3,000) 0.79 / 1.06; 48^3 (6,000 and
// more) 2.8 / 2.3; band n = 100,003 1.02 / 0.73 / 0.70; 128 2D grids 17.6 / 9.3
// / 7.2.
int reach_shape(uint64_t chunks, uint64_t reach, uint64_t largest, uint32_t W, int bits, uint32_t cus, int64_t room) {
    if (bits > 64 && chunks <= cus) return NT_WIDE;
    const int64_t quad = reach_bytes((uint32_t)std::min<uint64_t>(4ull * cus, chunks), W, bits);
    if (chunks >= 8ull * cus && reach <= 512 && quad <= std::min<int64_t>(room, 8ll << 30)) return NT_QUAD;
    if (bits <= 64) {
        const uint64_t need = largest + 256;  // with the nodes below the group
        const bool m64 = bits == 64;
        const uint64_t in_pair = node_room((uint32_t)(m64 ? node_slots<uint64_t>(NT_PAIR) : node_slots<uint32_t>(NT_PAIR)));
        const uint64_t in_wide = node_room((uint32_t)(m64 ? node_slots<uint64_t>(NT_WIDE) : node_slots<uint32_t>(NT_WIDE)));
        if (need > in_pair && need <= in_wide) return NT_WIDE;
    }
    const int64_t pair = reach_bytes((uint32_t)std::min<uint64_t>(2ull * cus, chunks), W, bits);
    return bits < 256 && pair <= std::min<int64_t>(room / 2, 32ll << 30) ? NT_PAIR : NT_WIDE;
}

namespace {
template <int NT, class M>
const void* kptr() {
    return reinterpret_cast<const void*>(
        &k_reach_blk<NT, tab_slots<M>(NT), node_slots<M>(NT), lanes_per_vertex<NT>(), edges_per_lane<NT>(), M>);
}
template <int NT, class M>
void klaunch(const RchParams& p, hipStream_t s) {
    hipLaunchKernelGGL((k_reach_blk<NT, tab_slots<M>(NT), node_slots<M>(NT), lanes_per_vertex<NT>(), edges_per_lane<NT>(), M>),
                       dim3(p.nblocks), dim3(NT), 0, s, p);
}
template <int NT>
const void* kptr_bits(int bits) {
    return bits == 256   ? kptr<NT, M256>()
           : bits == 128 ? kptr<NT, u128>()
           : bits == 64  ? kptr<NT, uint64_t>()
                         : kptr<NT, uint32_t>();
}
template <int NT>
void klaunch_bits(const RchParams& p, int bits, hipStream_t s) {
    if (bits == 256) klaunch<NT, M256>(p, s);
    else if (bits == 128) klaunch<NT, u128>(p, s);
    else if (bits == 64) klaunch<NT, uint64_t>(p, s);
    else klaunch<NT, uint32_t>(p, s);
}
}  // namespace

const void* rch_kernel_ptr(int bits, int threads) {
    return threads == NT_QUAD ? kptr_bits<NT_QUAD>(bits) : threads == NT_PAIR ? kptr_bits<NT_PAIR>(bits) : kptr_bits<NT_WIDE>(bits);
}
uint32_t rch_pass_bit() { return PASS_T; }
// Per workgroup: visited words (8, 16 or 32 B), two next-level masks, two
// 16-byte frontier queues, per vertex of the window.
int64_t reach_bytes(uint32_t nb, uint32_t W, int bits) {
    const int64_t vw = rch_visit_bytes(bits), mw = bits / 8;
    return (int64_t)nb * ((vw + 2 * mw + 32) * (int64_t)W + 8);
}

int64_t rch_visit_bytes(int bits) { return bits == 256 ? 48 : bits == 128 ? 32 : bits == 64 ? 16 : 8; }

hipError_t launch_reach(const RchParams& p, int bits, int threads, hipStream_t s) {
    if (!rch_bits_valid(bits) || !rch_shape_valid(threads)) return hipErrorInvalidValue;
    if (threads == NT_QUAD) klaunch_bits<NT_QUAD>(p, bits, s);
    else if (threads == NT_PAIR) klaunch_bits<NT_PAIR>(p, bits, s);
    else klaunch_bits<NT_WIDE>(p, bits, s);
    return hipGetLastError();
}

}  // namespace gsofa

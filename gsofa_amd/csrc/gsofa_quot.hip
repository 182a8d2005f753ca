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
// Each matrix's vertices are cut into blocks of
// 2^kQuotShift.  Level h holds the
// complete, aligned ranges of 2^h blocks; a range's classes are found in the
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
// many nodes keeps its halves' classes, and the label rounds below stop at a
// fixed count.
//
// What bounds it: latency.  A level is two launches; a range is a chain of
// dependent gathers (column, class, node number) and barriers of one
// workgroup, 20-100 us a level however many ranges it has, until ranges
// outnumber the CUs.
//
// Measured, traversal of one execute walking vertices -> classes (the
// classes' construction included): band n = 659,033 780 -> 5.8 ms, band
// n = 100,003 32.3 -> 1.5, 48^3 grid 64.9 -> 3.3, 128 2D grids 278 -> 33.5,
// 181^2 grid 16.4 -> 1.0, n = 11,948 1.13 -> 0.37.  At 48^3 the construction
// takes 0.73 ms of the 3.3, at the 128 grids 1.8 of 33.5.
#include <algorithm>

#include "gsofa_device.h"
#include "gsofa_internal.h"

namespace gsofa {

namespace {

using dev::WAVE;

constexpr uint16_t NOROOT = 0xFFFFu;
constexpr uint32_t NOIDX = 0xFFFFFFFFu;
constexpr int ROUNDS = 4;       // label rounds per range
constexpr int ITERS = 96;       // label iterations per round, at most
constexpr uint32_t SHORT_ROW = 64;   // rows up to here: 8 lanes each
constexpr uint32_t MID_ROW = 2048;   // rows up to here: one wave each; longer ones: the workgroup
constexpr int QBASE_CAP = 1 << kQuotShift;  // vertices of a level-0 range
constexpr int QCAP = 4096;           // nodes of a higher range whose classes are merged
constexpr int QBASE_NT = 256, QNT = 1024;

template <int CAP>
struct QLds {
    int32_t node[CAP];
    uint32_t rb[CAP], re[CAP];      // the node's row
    uint32_t fw[CAP], bw[CAP];      // labels; then the class's first member and size
    uint32_t a0[CAP], a1[CAP], a2[CAP];  // class sums and row cursor
    uint16_t root[CAP];
    unsigned long long ebase;
    uint32_t total, ne, left, got, nnew;
    uint32_t chg[3];
};

// f(i, k, end, step) covers edges k, k + step, .. k + 3 step (below end) of
// node i; every edge of every row is covered once by the workgroup.
template <int NT, class F>
__device__ __forceinline__ void each_row(const uint32_t* rb, const uint32_t* re, uint32_t m, F f) {
    const uint32_t tid = threadIdx.x, lane = __lane_id(), w = tid / WAVE;
    for (uint32_t i = tid / 8u; i < m; i += NT / 8) {
        const uint32_t b = rb[i], e = re[i];
        if (e - b > SHORT_ROW) continue;
        for (uint32_t k = b + (tid & 7u); k < e; k += 32u) f(i, k, e, 8u);
    }
    uint32_t turn = 0;
    for (uint32_t t0 = 0; t0 < m; t0 += WAVE) {
        const uint32_t i0 = t0 + lane;
        const uint32_t len = i0 < m ? re[i0] - rb[i0] : 0u;
        for (uint64_t b = __ballot(len > SHORT_ROW && len <= MID_ROW); b; b &= b - 1ull) {
            if (turn++ % (uint32_t)(NT / WAVE) != w) continue;
            const uint32_t i = t0 + (uint32_t)__builtin_ctzll(b);
            for (uint32_t k = rb[i] + lane; k < re[i]; k += 4u * WAVE) f(i, k, re[i], (uint32_t)WAVE);
        }
        for (uint64_t b = __ballot(len > MID_ROW); b; b &= b - 1ull) {
            const uint32_t i = t0 + (uint32_t)__builtin_ctzll(b);
            for (uint32_t k = rb[i] + tid; k < re[i]; k += 4u * NT) f(i, k, re[i], (uint32_t)NT);
        }
    }
}

// One workgroup per range.  Nodes are the halves' classes (BASE: vertices).
//  1. The edges among the range's nodes go to a list (node pairs).
//  2. Classes by label rounds: every node carries the largest label that
//     reaches it and the largest that it reaches; where both are the same
//     node c, the node is strongly connected with c.  Labels of heavy nodes
//     are larger, so the range's main class is found in the first round and
//     is not hidden behind single vertices that only lead into or out of it.
//     Assigned nodes leave the graph; the next round looks at the rest.
//  3. Each class of two or more nodes gets a row: its members' targets
//     outside the class, over A and over A^T.  Other nodes keep theirs.
template <int CAP, int NT, bool BASE>
__global__ __launch_bounds__(NT) void k_quot_classes(QuotParams p, uint32_t lev, uint32_t tab0, uint32_t ctab0) {
    __shared__ QLds<CAP> S;
    if (!BASE && quot_off(p)) return;
    const uint32_t tid = threadIdx.x;
    const uint2 R = p.tab[tab0 + blockIdx.x];
    const uint32_t size = 1u << (kQuotShift + lev);
    const uint32_t x = R.x;
    const int32_t* comp_prev = BASE ? nullptr : p.comp + (uint64_t)(lev - 1u) * p.n;
    const uint4* info_prev = BASE ? nullptr : p.info + (uint64_t)(lev - 1u) * p.n;
    const uint4* infoT_prev = BASE ? nullptr : p.infoT + (uint64_t)(lev - 1u) * p.n;
    uint4* info_cur = p.info + (uint64_t)lev * p.n;
    uint4* infoT_cur = p.infoT + (uint64_t)lev * p.n;
    const int32_t* nodes_prev = p.nodes + (uint64_t)((lev + 1u) & 1u) * p.n;
    int32_t* nodes_cur = p.nodes + (uint64_t)(lev & 1u) * p.n;
    uint32_t m0 = size, m = size;
    if (!BASE) {
        m0 = p.ncnt[ctab0 + R.y];
        m = m0 + p.ncnt[ctab0 + R.y + 1u];
    }
    const uint32_t xr = x + size / 2u;
    auto node_at = [&](uint32_t i) {
        return BASE ? (int32_t)(x + i) : i < m0 ? nodes_prev[x + i] : nodes_prev[xr + i - m0];
    };
    if (m > (uint32_t)CAP) {  // too many nodes: the halves' classes stand
        for (uint32_t i = tid; i < m; i += NT) {
            const int32_t v = node_at(i);
            p.nmap[v] = v;
            nodes_cur[x + i] = v;
            info_cur[v] = info_prev[v];
            infoT_cur[v] = infoT_prev[v];
        }
        if (tid == 0) p.ncnt[tab0 + blockIdx.x] = m;
        return;
    }
    auto row_of = [&](int32_t v, bool t) {
        if (!BASE) return t ? infoT_prev[v] : info_prev[v];
        const int32_t* rp = t ? p.rpT : p.rp;
        const uint32_t b = (uint32_t)rp[v], e = (uint32_t)rp[v + 1];
        return make_uint4(b, e, 1u, e - b);
    };
    if (tid == 0) {
        S.total = S.ne = S.nnew = 0;
        S.chg[0] = S.chg[1] = S.chg[2] = 0;
    }
    __syncthreads();
    {
        uint32_t len = 0;
        for (uint32_t i = tid; i < m; i += NT) {
            const int32_t v = node_at(i);
            const uint4 r = row_of(v, false);
            S.node[i] = v;
            S.rb[i] = r.x;
            S.re[i] = r.y;
            S.a2[i] = r.z;
            S.root[i] = NOROOT;
            if (!BASE) p.nidx[v] = (int32_t)i;
            len += r.y - r.x;
        }
        if (len) atomicAdd(&S.total, len);
    }
    __syncthreads();  // also: this workgroup's nidx writes are done
    if (tid == 0) S.ebase = atomicAdd(&p.ctl->eb[lev], (unsigned long long)S.total);
    __syncthreads();
    uint32_t* eb = p.eb + S.ebase;
    // local node of target v, NOIDX outside the range
    auto local = [&](int32_t v) {
        const uint32_t o = (uint32_t)v - x;
        if (o >= size) return NOIDX;
        return BASE ? o : (uint32_t)p.nidx[comp_prev[v]];
    };
    // ---- 1. edges among the nodes
    each_row<NT>(S.rb, S.re, m, [&](uint32_t i, uint32_t k, uint32_t e, uint32_t st) {
        int32_t v[4];
        uint32_t t[4];
        uint32_t cnt = 0;
#pragma unroll
        for (int q = 0; q < 4; q++) v[q] = k + q * st < e ? p.ci[k + q * st] : -1;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            t[q] = v[q] >= 0 ? local(v[q]) : NOIDX;
            if (t[q] == i) t[q] = NOIDX;
            cnt += t[q] != NOIDX;
        }
        if (!cnt) return;
        uint32_t o = atomicAdd(&S.ne, cnt);
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (t[q] != NOIDX) eb[o++] = (i << 16) | t[q];
    });
    __syncthreads();
    const uint32_t ne = S.ne;
    // ---- 2. classes
    // label: weight class, then a permuted node number (its inverse names the node)
    constexpr uint32_t PM = 2531u;  // odd: a bijection modulo CAP
    uint32_t inv = PM;              // PM * inv = 1 modulo 2^32, by Newton's iteration
    for (int k = 0; k < 4; k++) inv *= 2u - PM * inv;
    auto label = [&](uint32_t i) {
        return ((31u - (uint32_t)__builtin_clz(S.a2[i] | 1u)) << 16) | ((i * PM) & (uint32_t)(CAP - 1));
    };
    auto named = [&](uint32_t l) { return (l * inv) & (uint32_t)(CAP - 1); };
    for (int rd = 0; rd < ROUNDS; rd++) {
        for (uint32_t i = tid; i < m; i += NT)
            if (S.root[i] == NOROOT) S.fw[i] = S.bw[i] = label(i);
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
                    if (a == b || S.root[a] != NOROOT || S.root[b] != NOROOT) continue;
                    const uint32_t fa = S.fw[a], ba = S.bw[a], fb = S.fw[b], bb = S.bw[b];
                    if (fa > fb) {
                        atomicMax(&S.fw[b], fa);
                        ch = true;
                    }
                    if (bb > ba) {
                        atomicMax(&S.bw[a], bb);
                        ch = true;
                    }
                }
            }
            // what reaches (is reached by) a node's label reaches (is reached by) the node
            for (uint32_t i = tid; i < m; i += NT) {
                if (S.root[i] != NOROOT) continue;
                const uint32_t f = S.fw[i], b = S.bw[i];
                const uint32_t f2 = S.fw[named(f)], b2 = S.bw[named(b)];
                if (f2 > f) {
                    atomicMax(&S.fw[i], f2);
                    ch = true;
                }
                if (b2 > b) {
                    atomicMax(&S.bw[i], b2);
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
            if (S.root[i] != NOROOT) continue;
            if (S.fw[i] == S.bw[i]) {
                const uint32_t c = named(S.fw[i]);
                S.root[i] = (uint16_t)c;
                got += c != i;
            } else {
                left++;
            }
        }
        if (left) atomicAdd(&S.left, left);
        if (got) atomicAdd(&S.got, got);
        __syncthreads();
        const bool stop = S.left == 0 || (S.got == 0 && rd > 0);
        __syncthreads();
        if (stop) break;
    }
    // class c: the members with root c; fw: its first member, bw: its size
    for (uint32_t i = tid; i < m; i += NT) {
        S.fw[i] = NOIDX;
        S.bw[i] = 0;
        if (S.root[i] == NOROOT) S.root[i] = (uint16_t)i;
    }
    __syncthreads();
    for (uint32_t i = tid; i < m; i += NT) {
        atomicMin(&S.fw[S.root[i]], i);
        atomicAdd(&S.bw[S.root[i]], 1u);
    }
    __syncthreads();
    for (uint32_t i = tid; i < m; i += NT) {
        const uint32_t c = S.root[i], f = S.fw[c];
        const int32_t v = S.node[i], nv = S.node[f];
        if (BASE) p.comp[v] = nv;
        else p.nmap[v] = nv;
        if (f == i) {
            nodes_cur[x + atomicAdd(&S.nnew, 1u)] = v;
            if (S.bw[c] == 1u) {  // not merged: keeps its rows
                info_cur[v] = row_of(v, false);
                infoT_cur[v] = row_of(v, true);
            }
        }
    }
    // ---- 3. rows of merged classes, over A then over A^T
    for (int side = 0; side < 2; side++) {
        const bool t = side == 1;
        __syncthreads();
        for (uint32_t i = tid; i < m; i += NT) {
            S.a0[i] = S.a1[i] = 0;
            if (!t) S.a2[i] = 0;
        }
        __syncthreads();
        for (uint32_t i = tid; i < m; i += NT) {
            const uint32_t c = S.root[i];
            const bool merged = S.bw[c] > 1u;
            const uint4 r = merged ? row_of(S.node[i], t) : make_uint4(0u, 0u, 0u, 0u);
            S.rb[i] = r.x;  // unmerged nodes: an empty row
            S.re[i] = r.y;
            if (!merged) continue;
            atomicAdd(&S.a0[c], r.y - r.x);
            atomicAdd(&S.a1[c], r.w);
            if (!t) atomicAdd(&S.a2[c], r.z);
        }
        __syncthreads();
        uint4* info = t ? infoT_cur : info_cur;
        int32_t* cols = t ? p.ciT : p.ci;
        for (uint32_t i = tid; i < m; i += NT) {
            const uint32_t c = S.root[i];
            if (S.fw[c] != i || S.bw[c] == 1u) continue;
            // room for every member's row; the levels' rows never exceed the
            // matrix's entries, so the reserve of one matrix per level holds
            const uint32_t b = p.ext0 + (uint32_t)atomicAdd(t ? &p.ctl->extT : &p.ctl->ext, (unsigned long long)S.a0[c]);
            info[S.node[i]] = make_uint4(b, b, S.a2[c], S.a1[c]);
            S.a0[c] = b;
        }
        __syncthreads();
        each_row<NT>(S.rb, S.re, m, [&](uint32_t i, uint32_t k, uint32_t e, uint32_t st) {
            int32_t v[4];
            uint32_t cnt = 0;
            const uint32_t c = S.root[i];
#pragma unroll
            for (int q = 0; q < 4; q++) v[q] = k + q * st < e ? cols[k + q * st] : -1;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                if (v[q] < 0) continue;
                const uint32_t l = local(v[q]);
                if (l != NOIDX && S.root[l] == c) v[q] = -1;
                else cnt++;
            }
            if (!cnt) return;
            uint32_t o = atomicAdd(&S.a0[c], cnt);
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (v[q] >= 0) cols[o++] = v[q];
        });
        __syncthreads();
        for (uint32_t i = tid; i < m; i += NT) {
            const uint32_t c = S.root[i];
            if (S.fw[c] == i && S.bw[c] > 1u) info[S.node[i]].y = S.a0[c];
        }
    }
    if (tid == 0) {
        p.ncnt[tab0 + blockIdx.x] = S.nnew;
        if (BASE) atomicAdd(&p.ctl->nodes0, (unsigned long long)S.nnew);
    }
}

// Classes of every vertex of the level's ranges, from the level below.
__global__ __launch_bounds__(256) void k_quot_map(QuotParams p, uint32_t lev, uint32_t tab0, uint32_t ranges) {
    if (quot_off(p)) return;
    const uint32_t sh = kQuotShift + lev;
    const uint64_t total = (uint64_t)ranges << sh;
    const int32_t* prev = p.comp + (uint64_t)(lev - 1u) * p.n;
    int32_t* cur = p.comp + (uint64_t)lev * p.n;
    for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k < total;
         k += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t v = p.tab[tab0 + (uint32_t)(k >> sh)].x + ((uint32_t)k & ((1u << sh) - 1u));
        cur[v] = p.nmap[prev[v]];
    }
}

}  // namespace

// Levels of the largest matrix: a source's block index is at most blocks - 1,
// and only complete blocks are contracted.
uint32_t quot_levels(uint32_t W) {
    const uint32_t last = W == 0u ? 0u : (W - 1u) >> kQuotShift;
    uint32_t l = 0;
    while (last >> l) l++;
    return l;
}

uint64_t quot_ext(uint64_t nnz, uint32_t levels) { return nnz * levels; }

int64_t quot_bytes(int64_t n, int64_t nnz, uint32_t W) {
    const int64_t L = quot_levels(W);
    if (L == 0) return 0;
    return L * n * (4 + 32) + 16 * n + 4 * nnz + 8 * (int64_t)quot_ext((uint64_t)nnz, (uint32_t)L) +
           12 * ((n >> kQuotShift) * 2 + L + 1) + (int64_t)sizeof(QuotCtl) + 4096;
}

// Ranges of every level: tab[off[h] ..] = (first vertex, entry of the first
// half among level h - 1's); the halves' entries are neighbours.
void quot_table(const std::vector<uint32_t>& mat_base, uint32_t levels, std::vector<uint2>& tab, std::vector<uint32_t>& off) {
    tab.clear();
    off.assign((size_t)levels + 1, 0);
    std::vector<uint32_t> child(mat_base.size(), 0), mine(mat_base.size(), 0);
    for (uint32_t h = 0; h < levels; h++) {
        off[h] = (uint32_t)tab.size();
        for (size_t b = 0; b + 1 < mat_base.size(); b++) {
            const uint32_t nb = mat_base[b + 1] - mat_base[b];
            const uint32_t cnt = (nb == 0u ? 0u : (nb - 1u) >> kQuotShift) >> h;
            mine[b] = (uint32_t)tab.size() - off[h];
            for (uint32_t q = 0; q < cnt; q++)
                tab.push_back(make_uint2(mat_base[b] + (q << (kQuotShift + h)), child[b] + 2u * q));
        }
        child = mine;
    }
    off[levels] = (uint32_t)tab.size();
}

hipError_t launch_quot(const QuotParams& p, const std::vector<uint32_t>& off, hipStream_t s) {
    hipError_t e = launch_fill(reinterpret_cast<uint32_t*>(p.ctl), sizeof(QuotCtl) / 4, 0u, s);
    if (e != hipSuccess) return e;
    for (uint32_t h = 0; h < p.levels; h++) {
        const uint32_t ranges = off[h + 1] - off[h];
        if (ranges == 0) break;
        if (h == 0) {
            hipLaunchKernelGGL((k_quot_classes<QBASE_CAP, QBASE_NT, true>), dim3(ranges), dim3(QBASE_NT), 0, s, p, h,
                               off[h], 0u);
        } else {
            hipLaunchKernelGGL((k_quot_classes<QCAP, QNT, false>), dim3(ranges), dim3(QNT), 0, s, p, h, off[h],
                               off[h - 1]);
            const uint64_t total = (uint64_t)ranges << (kQuotShift + h);
            hipLaunchKernelGGL(k_quot_map, dim3((uint32_t)std::min<uint64_t>((total + 255) / 256, 2048)), dim3(256),
                               0, s, p, h, off[h], ranges);
        }
    }
    return hipGetLastError();
}

}  // namespace gsofa

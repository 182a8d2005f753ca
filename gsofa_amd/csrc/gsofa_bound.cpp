// gsofa_bound.cpp -- per-row upper bounds of the L/U structure, on the host,
// before any traversal.
//
// No counterpart in the reference, which sizes its frontier pool from a
// memory budget and recovers from overflow by spilling to the host
// (with_space_optimization/symbfact.cuh:2079, 2170-2380).  Here the fill
// stream and the output columns are sized once, from bounds that hold for
// every input:
//
// A fill path of A (a directed path i -> ... -> j whose intermediates are all
// below min(i, j); Rose and Tarjan, SIAM J. Appl. Math. 34, 1978) is also a
// path of the undirected graph of S = A + A^T with the same property, so
// struct(L + U) lies inside struct(C + C^T) for the Cholesky factor C of S.
// Row i of L therefore has at most rc(i) entries and row i of U at most
// cc(i), where rc / cc are the strict row / column counts of C.  Both come
// from the elimination tree of S in O(nnz(S) alpha(n)) time with the
// skeleton-leaf method of Gilbert, Ng and Peyton (SIAM J. Matrix Anal.
// Appl. 15, 1994):
//   * row i's pattern in C is its row subtree T_i: the union of the tree
//     paths from each j < i adjacent to i up to (not including) i.  Its
//     leaves are the adjacent j that have no adjacent descendant; in
//     postorder, j is one iff first(j) (the smallest postorder number in j's
//     subtree) exceeds the postorder number of the previous adjacent vertex
//     of row i;
//   * |T_i| = sum over its leaves l_1 < l_2 < ... (postorder) of
//     depth(l_t) - depth(q_t), with q_1 = i and q_t = lca(l_{t-1}, l_t);
//   * cc(k) = #{i : k in T_i} = the subtree sum at k of weights +1 at every
//     leaf, -1 at every lca(l_{t-1}, l_t) and -1 at i (once per nonempty T_i);
//   * the lca of an earlier vertex with the current one (in postorder) is
//     the representative of its set in a union-find whose vertices are
//     linked to their parent when finished (Tarjan's offline lca).
#include <algorithm>
#include <cstdint>
#include <vector>

#include "gsofa.h"

namespace gsofa {

namespace {

int32_t find_root(std::vector<int32_t>& anc, int32_t x) {
    int32_t r = x;
    while (anc[r] != r) r = anc[r];
    while (anc[x] != r) {  // compress the path just walked
        const int32_t nx = anc[x];
        anc[x] = r;
        x = nx;
    }
    return r;
}

}  // namespace

// rp/ci: packed rows (sorted, duplicate-free) of A, rpT/ciT of its transpose, n
// rows.  On return Lb[i] >= |L_i|, Ub[i] >= |U_i| (both strict, A's own entries
// included); the elimination tree of A + A^T goes to *parent_out if given.
// S's rows are never built: row i of S is row i of A and row i of A^T, and an
// entry met in both changes nothing the second time (its path to i is walked
// and compressed, and j is no leaf of T_i twice).
void lu_row_bounds(int32_t n, const int32_t* rp, const int32_t* ci, const int32_t* rpT, const int32_t* ciT,
                   std::vector<int64_t>& Lb, std::vector<int64_t>& Ub, std::vector<int32_t>* parent_out) {
    Lb.assign((size_t)n, 0);
    Ub.assign((size_t)n, 0);
    if (parent_out) parent_out->clear();
    if (n <= 0) return;
    const int32_t* const rows[2] = {rp, rpT};
    const int32_t* const cols[2] = {ci, ciT};
    // elimination tree of S (Liu's ancestor algorithm with path compression);
    // split[t][i]: row i's first entry above the diagonal
    std::vector<int32_t> parent((size_t)n, -1), anc((size_t)n, -1), split[2];
    split[0].resize((size_t)n);
    split[1].resize((size_t)n);
    for (int32_t i = 0; i < n; i++)
        for (int t = 0; t < 2; t++) {
            const int32_t* c = cols[t];
            int32_t p = rows[t][i];
            const int32_t e = rows[t][i + 1];
            for (; p < e && c[p] < i; p++) {
                int32_t r = c[p];
                for (;;) {
                    const int32_t a = anc[(size_t)r];
                    if (a == i) break;
                    anc[(size_t)r] = i;
                    if (a < 0) {
                        parent[(size_t)r] = i;
                        break;
                    }
                    r = a;
                }
            }
            split[t][(size_t)i] = p < e && c[p] == i ? p + 1 : p;
        }
    // depth (parents are numbered above their children) and a postorder
    std::vector<int32_t> depth((size_t)n, 0), head((size_t)n, -1), nxt((size_t)n, -1);
    for (int32_t j = n - 1; j >= 0; j--) {
        const int32_t pj = parent[(size_t)j];
        depth[(size_t)j] = pj < 0 ? 0 : depth[(size_t)pj] + 1;
        if (pj >= 0) {  // children listed in increasing order
            nxt[(size_t)j] = head[(size_t)pj];
            head[(size_t)pj] = j;
        }
    }
    std::vector<int32_t> post((size_t)n), first((size_t)n, -1);
    int32_t k = 0;
    for (int32_t root = 0; root < n; root++) {
        if (parent[(size_t)root] != -1) continue;
        // down to the next unvisited child, else number the vertex and go up
        for (int32_t v = root;;) {
            const int32_t c = head[(size_t)v];
            if (c >= 0) {
                head[(size_t)v] = nxt[(size_t)c];
                v = c;
                continue;
            }
            if (first[(size_t)v] < 0) first[(size_t)v] = k;  // a leaf starts its subtree
            post[(size_t)k++] = v;
            const int32_t up = parent[(size_t)v];
            if (up < 0) break;
            if (first[(size_t)up] < 0) first[(size_t)up] = first[(size_t)v];
            v = up;
        }
    }
    // skeleton leaves, row counts and column-count weights, in postorder
    std::vector<int32_t> last_adj((size_t)n, -1), prev_leaf((size_t)n, -1), set((size_t)n);
    int64_t* w = Ub.data();
    for (int32_t v = 0; v < n; v++) set[(size_t)v] = v;
    for (int32_t q = 0; q < n; q++) {
        const int32_t j = post[(size_t)q], fj = first[(size_t)j], dj = depth[(size_t)j];
        for (int t = 0; t < 2; t++) {
            const int32_t e = rows[t][j + 1];
            for (int32_t p = split[t][(size_t)j]; p < e; p++) {
                const int32_t i = cols[t][p];  // S(i, j) != 0 with i > j
                const bool leaf = fj > last_adj[(size_t)i];
                last_adj[(size_t)i] = q;
                if (!leaf) continue;
                w[j] += 1;
                const int32_t pl = prev_leaf[(size_t)i];
                int32_t top;  // where the path from j joins what row i already holds
                if (pl < 0) {
                    top = i;
                    w[i] -= 1;
                } else {
                    top = find_root(set, pl);
                    w[top] -= 1;
                }
                Lb[(size_t)i] += dj - depth[(size_t)top];
                prev_leaf[(size_t)i] = j;
            }
        }
        if (parent[(size_t)j] >= 0) set[(size_t)j] = parent[(size_t)j];
    }
    for (int32_t j = 0; j < n; j++)  // subtree sums: children precede parents
        if (parent[(size_t)j] >= 0) w[parent[(size_t)j]] += w[j];
    if (parent_out) parent_out->swap(parent);
}

// Records of one reach-mode pass at most (per mask word of 64 or 32 sources, a
// record for every vertex that a group of `bits` sources reaches at or above
// itself; groups are cut from each matrix's last vertex down).  A source's
// vertices above it lie in its column of C, and a column's entries but the
// parent lie in the parent's column, so a group reaches its own vertices and
// the columns of those whose parent is outside the group.  *largest: vertices
// of the group with the longest such column, its own and that column's (for the
// deep groups, whose columns mostly lie in one another, all they reach).
uint64_t reach_record_bound(const std::vector<uint32_t>& mat_base, const std::vector<int32_t>& parent,
                            const std::vector<int64_t>& Ub, int bits, uint64_t* largest) {
    uint64_t sum = 0;
    *largest = 0;
    for (size_t b = 0; b + 1 < mat_base.size(); b++) {
        for (int64_t hi = (int64_t)mat_base[b + 1]; hi > (int64_t)mat_base[b]; hi -= bits) {
            const int64_t lo = std::max<int64_t>(hi - bits, (int64_t)mat_base[b]);
            uint64_t items = (uint64_t)(hi - lo), column = 0;
            for (int64_t j = lo; j < hi; j++)
                if (parent[(size_t)j] < 0 || parent[(size_t)j] >= hi) {
                    items += (uint64_t)Ub[(size_t)j];
                    column = std::max(column, (uint64_t)Ub[(size_t)j]);
                }
            *largest = std::max(*largest, (uint64_t)(hi - lo) + column);
            sum += items;
        }
    }
    return sum * (uint64_t)(bits > 64 ? bits / 64 : 1);
}

// Of the sources gid, gid + N, ...: the largest subtree of the elimination tree
// (all that a source can reach below itself) over their mean.
double subtree_skew(int32_t N, int32_t gid, const std::vector<int32_t>& parent) {
    const int32_t n = (int32_t)parent.size();
    std::vector<int32_t> below((size_t)n, 1);
    for (int32_t i = 0; i < n; i++)
        if (parent[(size_t)i] >= 0) below[(size_t)parent[(size_t)i]] += below[(size_t)i];
    double sum = 0, most = 0;
    int64_t count = 0;
    for (int64_t i = gid; i < n; i += N, count++) {
        sum += below[(size_t)i];
        most = std::max<double>(most, below[(size_t)i]);
    }
    return sum > 0 ? most * (double)count / sum : 1;
}

}  // namespace gsofa

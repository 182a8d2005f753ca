"""GPU parity of reach mode over vertex classes (strongly connected classes of
block ranges stand for their vertices) against the CPU oracle: block and range
edges, patterns without classes, patterns that keep too many nodes to merge,
rows long enough to be split over lane groups, batches and replays."""
import numpy as np
import pytest

from gpu_util import assert_same_structure

pytestmark = pytest.mark.gpu

BLOCK = 256


def _oracle(A):
    from oracle import oracle
    return oracle.symbfact(A.colbeg, A.colend, A.csr, A.n)


def _from_edges(n, rows, cols):
    import gsofa_amd as g
    d = np.arange(n, dtype=np.int64)
    key = np.unique(np.concatenate([np.asarray(rows, np.int64) * n + cols, d * n + d]))
    end = np.cumsum(np.bincount(key // n, minlength=n))
    return g.CsrMatrix(n, np.concatenate([[0], end[:-1]]), end, key % n)


def _check(A, **kw):
    import gsofa_amd as g
    print("case: n", A.n, "nnz", A.nnz, kw, flush=True)
    r = g.symbfact(A, mode="reach", **kw)
    assert r.edge_checks >= r.te_alg
    assert_same_structure(r, _oracle(A))


@pytest.mark.parametrize("bits", [32, 64, 128, 256])
@pytest.mark.parametrize("n", [BLOCK, BLOCK + 1, 2 * BLOCK, 2 * BLOCK + 1, 3 * BLOCK - 1, 4 * BLOCK + 1, 9 * BLOCK + 77])
def test_range_edges(n, bits):
    import gsofa_amd as g
    _check(g.gen_band(n, 30, 4.0, n + bits), block_slots=bits)


@pytest.mark.parametrize("threads", [512, 1024])
@pytest.mark.parametrize("lam", [1.2, 2.0, 3.0])
def test_few_classes(lam, threads):
    """Sparse one-directional bands: most vertices stay classes of their own,
    at the lowest density so many that classes are not used at all."""
    import gsofa_amd as g
    _check(g.gen_band(20011, 200, lam, 7), block_slots=64, workgroup_threads=threads)


@pytest.mark.parametrize("nodes", [2, 63, 64, 65, 127, 128, 129, 193, 255, 256])
def test_closure_sizes(nodes):
    """Ranges of two blocks of 128 with that many nodes: in each block the last
    vertices are one cycle, the others have edges to later ones only, and sparse
    edges between the blocks close cycles of every length among the nodes."""
    rng = np.random.default_rng(nodes)
    n, half = 2048 + 77, 128
    rows, cols = [], []
    for b in range(n // half):
        m = nodes // 2 if b % 2 == 0 else nodes - nodes // 2
        first = m - 1 if m < half else half  # of the cycle
        c = b * half + np.arange(first, half)
        if len(c) > 1:
            rows.append(c), cols.append(np.roll(c, -1))
        u = rng.integers(0, half, (2, 40))
        u = np.sort(u[:, u.max(axis=0) < first], axis=0)
        rows.append(b * half + u[0]), cols.append(b * half + u[1])
        v = rng.integers(0, half, (2, 48))
        v[0, 0] = v[1, 0] = 0
        rows.append(b * half + v[0]), cols.append((b ^ 1) * half + v[1])
    u = rng.integers(0, n, (2, 600))
    rows.append(u[0]), cols.append(u[1])
    rows, cols = np.concatenate(rows), np.concatenate(cols)
    keep = cols < n
    for bits in (32, 64, 256):
        _check(_from_edges(n, rows[keep], cols[keep]), block_slots=bits)


@pytest.mark.parametrize("n", [128, 129, 192, 193, 256, 257, 1024, 1025, 2111, 4161])
def test_chain_blocks(n):
    """Rows mostly coupled to their neighbours take blocks of 64 vertices: one
    direction, both, and every third link cut, with a few long entries."""
    rng = np.random.default_rng(n)
    i = np.arange(n - 1)
    far = rng.integers(0, n, (2, n // 16))
    for links, back in ((i, i[::2]), (i, i), (i[i % 3 != 0], i[:0]), (i[:0], i)):
        rows = np.concatenate([links, back + 1, far[0]])
        cols = np.concatenate([links + 1, back, far[1]])
        for bits in (32, 64, 128):
            _check(_from_edges(n, rows, cols), block_slots=bits)


def test_too_many_nodes():
    """Ranges of over 256 live nodes keep their halves' classes: pairs (2i, 2i+1)
    are strongly connected, the pairs form an acyclic chain of chains."""
    n = 12001
    i = np.arange(0, n - 1, 2)
    rows = np.concatenate([i, i + 1, i[:-9]])
    cols = np.concatenate([i + 1, i, i[:-9] + 18])
    _check(_from_edges(n, rows, cols), block_slots=32)
    _check(_from_edges(n, cols, rows), block_slots=32)


def test_acyclic():
    n = 1500
    rng = np.random.default_rng(3)
    i, j = rng.integers(0, n, 6000), rng.integers(0, n, 6000)
    lo, hi = np.minimum(i, j), np.maximum(i, j)
    _check(_from_edges(n, lo, hi))
    _check(_from_edges(n, hi, lo))


@pytest.mark.parametrize("bits", [32, 64, 256])
@pytest.mark.parametrize("hubs,length", [(1, 193), (3, 2900), (60, 250)])
def test_long_rows(hubs, length, bits):
    """Hub rows and columns longer than the split length, more of them than
    the split list holds, below, among and above the other vertices."""
    n = 3001
    rng = np.random.default_rng(hubs)
    rows, cols = [], []
    for h in rng.choice(n, hubs, replace=False):
        t = rng.choice(n, length, replace=False)
        rows += [np.full(length, h), t]
        cols += [t, np.full(length, h)]
    i = np.arange(n - 1)
    rows += [i, i[::3] + 1]
    cols += [i + 1, i[::3]]
    _check(_from_edges(n, np.concatenate(rows), np.concatenate(cols)), block_slots=bits)


@pytest.mark.parametrize("kw", [dict(), dict(graph=True), dict(counts_only=True)])
def test_batch_of_sizes(kw):
    """Matrices below, at and above a block in one plan, executed three times."""
    import gsofa_amd as g
    import gsofa_amd.configs as cf
    mats = [cf.batch_matrix(s, s) for s in (1, 15, 16, 17, 40, 70)] + [g.gen_band(2 * BLOCK + 1, 20, 3.0, 1),
                                                                      cf.grid64_natural()]
    orc = [_oracle(A) for A in mats]
    print("case: batch", kw, flush=True)
    with g.Plan(mats, mode="reach", **kw) as p:
        for _ in range(3):
            p.execute()
            for b, o in enumerate(orc):
                r = p.fetch_matrix(b)
                if kw.get("counts_only"):
                    assert r.fill_count == o.fill_count and r.te_alg == o.te_alg and r.reach == o.reach
                    np.testing.assert_array_equal(r.row_fill, o.row_fill)
                else:
                    assert_same_structure(r, o)


@pytest.mark.parametrize("bits", [32, 64, 128, 256])
def test_narrow_groups(bits):
    """Thousands of narrow mini-groups take four workgroups per CU."""
    import gsofa_amd as g
    if bits == 256:
        mats = [g.gen_band(14001, 12, 3.0, s) for s in range(5)] * 4
    else:
        mats = [g.gen_grid(s, s, 1, nd_leaf=64, extra_prob=0.05, extra_dist=3, seed=s) for s in (3, 150, 171, 256)]
        mats.append(g.gen_grid(257, 255, 1, nd_leaf=64, seed=9))
    print("case: narrow groups, bits", bits, flush=True)
    with g.Plan(mats, mode="reach", block_slots=bits) as p:
        p.execute()
        for b, A in enumerate(mats[:5]):
            r = p.fetch_matrix(b)
            assert r.grid_blocks > 512
            assert_same_structure(r, _oracle(A))

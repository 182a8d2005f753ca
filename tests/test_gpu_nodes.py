"""GPU parity of reach mode around the limits of a group's node table in LDS:
groups that outgrow it between groups that fit, rows walked in parts (also the
sources' own), and vertices above a group that span several bitmap windows."""
import numpy as np
import pytest

from gpu_util import assert_same_structure

pytestmark = pytest.mark.gpu


def _oracle(A):
    from oracle import oracle
    return oracle.symbfact(A.colbeg, A.colend, A.csr, A.n)


def _from_edges(n, rows, cols):
    import gsofa_amd as g
    d = np.arange(n, dtype=np.int64)
    key = np.unique(np.concatenate([np.asarray(rows, np.int64) * n + cols, d * n + d]))
    end = np.cumsum(np.bincount(key // n, minlength=n))
    return g.CsrMatrix(n, np.concatenate([[0], end[:-1]]), end, key % n)


def _star(n):
    """Vertex 0 and every other vertex of a second matrix' worth of rows: source s
    reaches all n - s vertices above it, so the low groups outgrow every table."""
    i = np.arange(1, n, dtype=np.int64)
    z = np.zeros(n - 1, np.int64)
    far = np.full((n - 1) // 3 + 1, n - 1, np.int64)
    return _from_edges(n, np.concatenate([i, z, i[::3][: far.size]]), np.concatenate([z, i, far[: i[::3].size]]))


STAR = {}


def _star_case(n):
    if n not in STAR:
        A = _star(n)
        STAR[n] = (A, _oracle(A))
    return STAR[n]


@pytest.mark.parametrize("bits,threads", [(32, 512), (32, 1024), (64, 512), (64, 1024), (64, 0), (128, 0)])
def test_groups_larger_than_the_table(bits, threads):
    import gsofa_amd as g
    A, o = _star_case(5500)
    print("case", bits, threads, flush=True)
    with g.Plan(A, mode="reach", block_slots=bits, workgroup_threads=threads) as p:
        for _ in range(2):
            p.execute()
            assert_same_structure(p.fetch(), o)
    with g.Plan(A, mode="reach", block_slots=bits, workgroup_threads=threads, counts_only=True) as p:
        p.execute()
        r = p.fetch()
        assert (r.fill_count, r.te_alg, r.reach) == (o.fill_count, o.te_alg, o.reach)
        np.testing.assert_array_equal(r.row_fill, o.row_fill)


@pytest.mark.parametrize("n", [1, 2, 24, 25, 33, 48, 49, 130])
@pytest.mark.parametrize("bits", [32, 64])
def test_small_stars(n, bits):
    """Rows of up to n entries around the length from which parts are made."""
    import gsofa_amd as g
    A = _star(n) if n > 1 else _from_edges(1, [0], [0])
    for threads in (512, 1024):
        assert_same_structure(g.symbfact(A, mode="reach", block_slots=bits, workgroup_threads=threads), _oracle(A))


@pytest.mark.parametrize("bits", [32, 64])
def test_windows(bits):
    import gsofa_amd as g
    n = 150001
    rng = np.random.default_rng(3)
    i = np.arange(n, dtype=np.int64)
    j = np.minimum(i + rng.integers(1, 20, n), n - 1)
    f = i[:: 40]
    rows = np.concatenate([i, j, f, n - 1 - f % 7, f[::5]])
    cols = np.concatenate([j, i, n - 1 - f % 5, f, np.minimum(f[::5] + 60000, n - 1)])
    A = _from_edges(n, rows, cols)
    o = _oracle(A)
    for threads in (0, 512):
        print("case", bits, threads, A.nnz, flush=True)
        assert_same_structure(g.symbfact(A, mode="reach", block_slots=bits, workgroup_threads=threads), o)


@pytest.mark.parametrize("bits", [32, 64, 256])
@pytest.mark.parametrize("n,band,lam", [(1500, 200, 12.0), (6011, 250, 9.0), (5000, 2500, 14.0)])
def test_shared_targets(n, band, lam, bits):
    """Classes whose members share targets, which their rows hold once."""
    import gsofa_amd as g
    A = g.gen_band(n, band, lam, n)
    assert_same_structure(g.symbfact(A, mode="reach", block_slots=bits), _oracle(A))

"""Columns of L and U for the hand-off from the traversal's records, against
transposes of the rows: every mask width, columns that many groups reach, runs
repeated, replayed and fetched in either order, and the same from a run without
records (block mode)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _csc(rowptr, col, n):
    rows = np.repeat(np.arange(n, dtype=np.int64), np.diff(rowptr))
    order = np.lexsort((rows, col.astype(np.int64)))
    colptr = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(col, minlength=n), out=colptr[1:])
    return colptr, rows[order].astype(np.int32)


def _check(r, h):
    for rp, col, cp, row in ((r.L_rowptr, r.L_col, h.xlcol, h.lrow), (r.U_rowptr, r.U_col, h.xucol, h.urow)):
        want = _csc(rp, col, r.n)
        np.testing.assert_array_equal(cp, want[0])
        np.testing.assert_array_equal(row, want[1])
    first = h.xsup[:-1]
    np.testing.assert_array_equal(np.diff(h.xsub), 1 + np.diff(r.U_rowptr)[first])
    np.testing.assert_array_equal(h.sub[h.xsub[:-1]], first)


def _arrow(n, seed):
    """Both triangles' last rows and columns are reached from every group."""
    import gsofa_amd as g
    rng = np.random.default_rng(seed)
    i = np.arange(n, dtype=np.int64)
    j = np.minimum(i + rng.integers(1, 9, n), n - 1)
    rows = np.concatenate([i, i, j[::2], np.full(n, n - 1), i])
    cols = np.concatenate([i, j, i[::2], i, np.full(n, n - 2)])
    key = np.unique(rows * n + cols)
    end = np.cumsum(np.bincount(key // n, minlength=n))
    return g.CsrMatrix(n, np.concatenate([[0], end[:-1]]), end, key % n)


@pytest.mark.parametrize("bits", [32, 64, 128, 256])
@pytest.mark.parametrize("n", [2, 65, 257, 9001])
def test_columns(n, bits):
    import gsofa_amd as g
    for A in (_arrow(n, n + bits), g.gen_band(n, min(40, n - 1), 3.0, n)):
        print("case", n, bits, A.nnz, flush=True)
        with g.Plan(A, mode="reach", block_slots=bits) as p:
            for order in (0, 1):
                p.execute()
                h = p.fetch_supernodal() if order else None
                r = p.fetch()
                _check(r, h or p.fetch_supernodal())
                _check(r, p.fetch_supernodal())


def test_columns_of_replays_and_block_mode():
    import gsofa_amd as g
    A = g.gen_grid(15, 14, 13, nd_leaf=32, extra_prob=0.05, extra_dist=2, seed=4)
    with g.Plan(A, graph=True) as p:
        for _ in range(4):
            p.execute()
            _check(p.fetch(), p.fetch_supernodal())
    for kw in ({"mode": "block"}, {"mode": "reach", "output_capacity": 1000}):
        with g.Plan(A, **kw) as p:
            p.execute()
            _check(p.fetch(), p.fetch_supernodal())

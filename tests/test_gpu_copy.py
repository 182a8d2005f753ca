"""GPU parity of results around the sizes where their copy to the host changes
hands: one kernel, one thread's chunks, several threads; and of calls that copy
at the same time."""
import threading

import numpy as np
import pytest

from gpu_util import assert_same_structure

pytestmark = pytest.mark.gpu


def _full_band(n, b):
    """Every entry within b of the diagonal, a few above it left out."""
    import gsofa_amd as g
    i = np.repeat(np.arange(n, dtype=np.int64), 2 * b + 1)
    j = i + np.tile(np.arange(-b, b + 1, dtype=np.int64), n)
    ok = (j >= 0) & (j < n) & ((j <= i) | ((i + 3 * j) % 7 != 0))
    key = i[ok] * n + j[ok]
    end = np.cumsum(np.bincount(key // n, minlength=n))
    return g.CsrMatrix(n, np.concatenate([[0], end[:-1]]), end, key % n)


def _oracle(A):
    from oracle import oracle
    return oracle.symbfact(A.colbeg, A.colend, A.csr, A.n)


# 8 * b + 28 bytes a row: below, at and above 512 KB; 1 and 4 MB; several threads
SIZES = [(1, 0), (2, 1), (2001, 28), (2080, 28), (4201, 28), (8300, 60), (20011, 61), (50021, 62)]


@pytest.mark.parametrize("n,b", SIZES)
def test_result_sizes(n, b):
    import gsofa_amd as g
    A = _full_band(n, b)
    print("case", n, b, flush=True)
    o = _oracle(A)
    assert_same_structure(g.symbfact(A), o)
    with g.Plan(A) as plan:
        plan.execute()
        h = plan.fetch_supernodal()
        r = plan.fetch()
    assert_same_structure(r, o)
    key = np.sort(np.asarray(o.L_col, np.int64) * n + np.repeat(np.arange(n), np.diff(o.L_rowptr)))
    np.testing.assert_array_equal(h.lrow, (key % n).astype(np.int32))
    np.testing.assert_array_equal(h.xlcol[1:], np.cumsum(np.bincount(key // n, minlength=n)))


def test_wide_ranges():
    """Columns further apart than 16 bits, within rows and where rows meet."""
    import gsofa_amd as g
    n = 140003
    rng = np.random.default_rng(8)
    i = np.arange(n, dtype=np.int64)
    f = i[::3]
    rows = np.concatenate([i, i, f, np.minimum(f + 1, n - 1), i[-400:]])
    cols = np.concatenate([i, np.minimum(i + 1, n - 1), n - 1 - f % 37, f, rng.integers(0, n - 400, 400)])
    key = np.unique(rows * n + cols)
    end = np.cumsum(np.bincount(key // n, minlength=n))
    A = g.CsrMatrix(n, np.concatenate([[0], end[:-1]]), end, key % n)
    o = _oracle(A)
    assert np.abs(np.diff(o.U_col)).max() > 65536
    assert_same_structure(g.symbfact(A), o)
    with g.Plan(A) as plan:
        plan.execute()
        h = plan.fetch_supernodal()
    key = np.sort(np.asarray(o.U_col, np.int64) * n + np.repeat(np.arange(n), np.diff(o.U_rowptr)))
    np.testing.assert_array_equal(h.urow, (key % n).astype(np.int32))


def test_concurrent_results():
    import gsofa_amd as g
    mats = [_full_band(n, b) for n, b in SIZES[2:7]]
    want = [_oracle(A) for A in mats]
    got = {}

    def work(k):
        for q in range(len(mats)):
            got[k, q] = g.symbfact(mats[(q + k) % len(mats)])
    th = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for (k, q), r in sorted(got.items()):
        assert_same_structure(r, want[(q + k) % len(mats)])
    assert len(got) == 4 * len(mats)

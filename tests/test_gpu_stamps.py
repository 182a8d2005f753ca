"""GPU: the clear of the visited words when a workgroup's stamps run out, in
reach mode.  Stamps are used up by the groups that are run in memory alone: all
of 128 and 256 slots, and with 32 and 64 those that outgrow the node table.
GSOFA_OFFSET_SPAN lowers the span to a few groups."""
import numpy as np
import pytest

from gpu_util import assert_same_structure

pytestmark = pytest.mark.gpu


def _oracle(A):
    from oracle import oracle
    return oracle.symbfact(A.colbeg, A.colend, A.csr, A.n)


@pytest.fixture(scope="module")
def star():
    """Source s reaches all n - s vertices above it, through vertex 0: the low
    groups hold 5,500 nodes, more than any table (4,984 at most)."""
    import gsofa_amd as g
    n = 5500
    i = np.arange(n, dtype=np.int64)
    rows = np.concatenate([i, i[1:], np.zeros(n - 1, np.int64)])
    cols = np.concatenate([i, np.zeros(n - 1, np.int64), i[1:]])
    key = np.unique(rows * n + cols)
    end = np.cumsum(np.bincount(key // n, minlength=n))
    A = g.CsrMatrix(n, np.concatenate([[0], end[:-1]]), end, key % n)
    return A, _oracle(A)


@pytest.mark.parametrize("span", [1, 2, 5])
@pytest.mark.parametrize("slots", [32, 64, 128, 256])
def test_star(star, monkeypatch, slots, span):
    import gsofa_amd as g
    A, o = star
    print("case: star, slots", slots, "span", span, flush=True)
    monkeypatch.setenv("GSOFA_OFFSET_SPAN", str(span))
    # few workgroups: each runs many groups one after the other
    with g.Plan(A, mode="reach", block_slots=slots, grid_blocks=4) as p:
        for _ in range(3):
            p.execute()
            assert_same_structure(p.fetch(), o)


@pytest.mark.parametrize("span", [1, 2, 5])
@pytest.mark.parametrize("slots", [128, 256])
def test_bcsstk18(bcsstk18, monkeypatch, slots, span):
    import gsofa_amd as g
    o = _oracle(bcsstk18)
    print("case: bcsstk18, slots", slots, "span", span, flush=True)
    monkeypatch.setenv("GSOFA_OFFSET_SPAN", str(span))
    with g.Plan(bcsstk18, mode="reach", block_slots=slots, grid_blocks=8) as p:
        for _ in range(3):
            p.execute()
            assert_same_structure(p.fetch(), o)

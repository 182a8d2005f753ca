"""GPU parity of cyclic shares: few sources a workgroup with labels in LDS or (2
and 4 slots) in memory, up to the sizes where one changes to the other, rows
longer than a step takes, levels with more targets than a round's table, every
share in one execute and replays."""
import numpy as np
import pytest

from gpu_util import assert_same_structure

pytestmark = pytest.mark.gpu


def _oracle(A, **kw):
    from oracle import oracle
    return oracle.symbfact(A.colbeg, A.colend, A.csr, A.n, **kw)


def _slots(r):
    return r.chunk // r.grid_blocks


def _hub(n, extra, seed):
    """Two hubs above n - 2 vertices that have few entries of their own: the
    hubs' frontiers and rows take all of them."""
    import gsofa_amd as g
    rng = np.random.default_rng(seed)
    i = np.arange(n, dtype=np.int64)
    a = rng.integers(0, n - 2, extra * n // 2)
    b = np.maximum(a - rng.integers(1, 4, a.size), 0)
    low = np.arange(n - 2, dtype=np.int64)
    rows = np.concatenate([i, a, low, np.full(n - 2, n - 1), np.full((n - 2) // 2, n - 2), low[::3]])
    cols = np.concatenate([i, b, np.full(n - 2, n - 1), low, low[: (n - 2) // 2], np.full(low[::3].size, n - 2)])
    key = np.unique(rows * n + cols)
    end = np.cumsum(np.bincount(key // n, minlength=n))
    return g.CsrMatrix(n, np.concatenate([[0], end[:-1]]), end, key % n)


@pytest.mark.parametrize("side,N,gid,slots", [(12, 3, 0, 1), (12, 7, 6, 1), (17, 2, 1, 1), (22, 2, 0, 2), (3, 5, 4, None)])
def test_grid3d_shares(side, N, gid, slots):
    import gsofa_amd as g
    A = g.gen_grid(side, side, side, nd_leaf=32, extra_prob=0.02, extra_dist=3, seed=side)
    print("case", side, N, gid, flush=True)
    r = g.symbfact(A, n_virtual_gpu=N, virtual_gpu_id=gid)
    assert r.mode == "block" and (slots is None or _slots(r) == slots)
    o = _oracle(A, n_virtual_gpu=N, virtual_gpu_id=gid)
    assert_same_structure(r, o, check_super=False)
    c = g.symbfact(A, n_virtual_gpu=N, virtual_gpu_id=gid, counts_only=True)
    assert (c.fill_count, c.te_alg, c.reach) == (o.fill_count, o.te_alg, o.reach)
    for k in ("row_fill", "row_te", "row_reach"):
        np.testing.assert_array_equal(getattr(c, k), getattr(o, k))


@pytest.mark.parametrize("n,extra,slots", [(43, 2, 1), (4099, 2, 1), (9001, 4, 2), (12000, 2, 2), (17000, 2, 1), (30001, 2, 4)])
def test_hubs(n, extra, slots):
    import gsofa_amd as g
    A = _hub(n, extra, n)
    for N, gid in ((2, (n - 1) % 2), (3, 1)):
        print("case", n, N, gid, flush=True)
        r = g.symbfact(A, n_virtual_gpu=N, virtual_gpu_id=gid)
        assert N == 3 or _slots(r) == slots
        assert_same_structure(r, _oracle(A, n_virtual_gpu=N, virtual_gpu_id=gid), check_super=False)


@pytest.mark.parametrize("n,band,N,slots", [(700, 40, 3, 2), (5000, 60, 4, 4), (11003, 100, 8, 2), (21001, 60, 4, 8)])
def test_band_shares(n, band, N, slots):
    import gsofa_amd as g
    A = g.gen_band(n, band, 5.0, n)
    r = g.symbfact(A, n_virtual_gpu=N, virtual_gpu_id=N - 1)
    assert _slots(r) == slots
    assert_same_structure(r, _oracle(A, n_virtual_gpu=N, virtual_gpu_id=N - 1), check_super=False)


def test_four_slots_in_memory():
    import gsofa_amd as g
    A = g.gen_grid(134, 134, 1, nd_leaf=32, extra_prob=0.02, extra_dist=3, seed=3)
    r = g.symbfact(A, n_virtual_gpu=2, virtual_gpu_id=1)
    assert _slots(r) == 1
    A = g.gen_grid(140, 140, 1, nd_leaf=32, extra_prob=0.02, extra_dist=3, seed=3)
    r = g.symbfact(A, n_virtual_gpu=2, virtual_gpu_id=1)
    assert _slots(r) == 4
    assert_same_structure(r, _oracle(A, n_virtual_gpu=2, virtual_gpu_id=1), check_super=False)


@pytest.mark.parametrize("shares", [1, 3])
@pytest.mark.parametrize("slots", [8, 0])
def test_all_shares_and_replays(shares, slots):
    import gsofa_amd as g
    A = g.gen_grid(14, 14, 14, nd_leaf=32, extra_prob=0.02, extra_dist=3, seed=9)
    o = _oracle(A)
    with g.Plan(A, mode="block", n_virtual_gpu=shares, block_slots=slots, graph=True) as p:
        for _ in range(4):
            p.execute()
            assert_same_structure(p.fetch(), o)

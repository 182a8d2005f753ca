"""GPU parity of reach mode where a group outgrows its node table in LDS after
some levels and goes on in memory from there: chains, wide levels whose last
edges are lost, long rows among the pending ones, groups that fit between."""
import numpy as np
import pytest

from gpu_util import assert_same_structure

pytestmark = pytest.mark.gpu

ROOM = 4984  # nodes that the largest table holds (32 sources, 1,024 threads)


def _oracle(A):
    from oracle import oracle
    return oracle.symbfact(A.colbeg, A.colend, A.csr, A.n)


def _from_edges(n, rows, cols):
    import gsofa_amd as g
    d = np.arange(n, dtype=np.int64)
    key = np.unique(np.concatenate([np.asarray(rows, np.int64) * n + cols, d * n + d]))
    end = np.cumsum(np.bincount(key // n, minlength=n))
    return g.CsrMatrix(n, np.concatenate([[0], end[:-1]]), end, key % n)


def _cycle():
    """One directed cycle: a level a node, the last of them too many."""
    n = ROOM + 200
    i = np.arange(n)
    return _from_edges(n, i, (i + 1) % n)


def _random():
    """Levels of thousands of nodes, no classes."""
    n = 12000
    rng = np.random.default_rng(8)
    return _from_edges(n, rng.integers(0, n, 2 * n), rng.integers(0, n, 2 * n))


def _long_rows():
    """A path to rows of 150 to 700 entries, over the lengths that are walked in
    parts and split, which together reach more nodes than fit."""
    n = 9000
    rng = np.random.default_rng(9)
    rows, cols = [np.full(3, n - 1), np.arange(1, 40)], [np.array([0, 5, 9]), np.arange(0, 39)]
    for k in range(40):
        e = rng.integers(40, n - 1, rng.integers(150, 700))
        rows += [np.full(e.size, k), e[::4]]
        cols += [e, np.full(e[::4].size, rng.integers(0, 40))]
    rows.append(np.arange(0, 39))
    cols.append(np.arange(1, 40))
    more = rng.integers(40, n, (2, 2 * n))
    return _from_edges(n, np.concatenate(rows + [more[0]]), np.concatenate(cols + [more[1]]))


MAKE = {"cycle": _cycle, "random": _random, "long rows": _long_rows}
CASES = {}


def _case(name):
    if name not in CASES:
        A = MAKE[name]()
        o = _oracle(A)
        # a source's own nodes, with no classes to stand for them, are too many
        assert (o.row_reach + np.diff(o.U_rowptr)).max() > ROOM, name
        CASES[name] = (A, o)
    return CASES[name]


@pytest.mark.parametrize("threads", [512, 1024, 0])
@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("name", list(MAKE))
def test_outgrows_after_some_levels(name, bits, threads):
    import gsofa_amd as g
    A, o = _case(name)
    print("case", name, bits, threads, flush=True)
    with g.Plan(A, mode="reach", block_slots=bits, workgroup_threads=threads, graph=True) as p:
        for _ in range(3):
            p.execute()
            assert_same_structure(p.fetch(), o)
    with g.Plan(A, mode="reach", block_slots=bits, workgroup_threads=threads, counts_only=True) as p:
        p.execute()
        r = p.fetch()
        assert (r.fill_count, r.te_alg, r.reach) == (o.fill_count, o.te_alg, o.reach)
        np.testing.assert_array_equal(r.row_fill, o.row_fill)


@pytest.mark.parametrize("span", [0, 1])
def test_between_groups_that_fit(monkeypatch, span):
    """Few workgroups take groups of all kinds in turn, at span 1 with the visited
    words cleared before each group that goes to memory."""
    import gsofa_amd as g
    mats, want = [], []
    rng = np.random.default_rng(10)
    for k, name in enumerate(list(MAKE) + ["cycle"]):
        A, o = _case(name)
        n = 40 + 60 * k
        B = _from_edges(n, rng.integers(0, n, 3 * n), rng.integers(0, n, 3 * n))
        mats += [A, B]
        want += [o, _oracle(B)]
    if span:
        monkeypatch.setenv("GSOFA_OFFSET_SPAN", str(span))
    print("case: batch, span", span, flush=True)
    with g.Plan(mats, mode="reach", grid_blocks=5) as p:
        for _ in range(2):
            p.execute()
            for i, o in enumerate(want):
                assert_same_structure(p.fetch_matrix(i), o)

"""GPU: a device allocation that fails ends its call with GSOFA_ERR_ALLOC alone.
GSOFA_FAIL_ALLOC=k, read when a plan or a server worker's arena is made, fails
its k-th allocation once; whatever runs next on the same plan or server must
find every array it needs."""
import pytest

from gpu_util import assert_same_structure

pytestmark = pytest.mark.gpu

ERR_ALLOC = -2


def _oracle(A):
    from oracle import oracle
    return oracle.symbfact(A.colbeg, A.colend, A.csr, A.n)


@pytest.fixture(scope="module")
def cases():
    import gsofa_amd as g
    mats = [g.gen_band(3000, 40, 4.0, 11), g.gen_grid(9, 9, 9, nd_leaf=64, seed=7), g.gen_band(4000, 60, 4.0, 12)]
    return [(A, _oracle(A)) for A in mats]


def test_server_after_a_failed_batch(cases, monkeypatch):
    """Every allocation of the first batch (an arena makes 39) and of the third,
    larger one in turn: one request fails, and those behind it, smaller ones among
    them that the failed one's sizes would have held, do not."""
    import gsofa_amd as g
    failed = 0
    for k in range(1, 44):
        print("case: server, allocation", k, flush=True)
        monkeypatch.setenv("GSOFA_FAIL_ALLOC", str(k))
        with g.Server(mem_gb=4.0, max_inflight=1) as srv:
            errors = []
            for A, o in cases + cases[1:]:
                try:
                    r, _ = srv.wait(srv.submit(A))
                except g.GsofaError as e:
                    errors.append(e.code)
                    continue
                assert_same_structure(r, o)
            assert errors in ([], [ERR_ALLOC])
            failed += len(errors)
    assert failed >= 39


@pytest.mark.parametrize("kw", [dict(mode="reach", output_capacity=10), dict(mode="block", output_capacity=10),
                                dict(n_virtual_gpu=3, spill=True, output_capacity=10), dict(mode="block")],
                         ids=["reach", "block", "spill", "bounded"])
def test_plan_after_a_failed_execute(cases, monkeypatch, kw):
    """Every allocation of a plan and its first execute in turn; the second
    execute gives the whole result."""
    import gsofa_amd as g
    A, o = cases[1]
    failed = 0
    for k in range(1, 50):
        print("case: plan", kw, "allocation", k, flush=True)
        monkeypatch.setenv("GSOFA_FAIL_ALLOC", str(k))
        try:
            p = g.Plan(A, **kw)
        except g.GsofaError as e:
            assert e.code == ERR_ALLOC
            continue
        with p:
            try:
                p.execute()
            except g.GsofaError as e:
                assert e.code == ERR_ALLOC
                failed += 1
                with pytest.raises(g.GsofaError):
                    p.fetch()
                p.execute()
            assert_same_structure(p.fetch(), o)
    assert failed >= 3

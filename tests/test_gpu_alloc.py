"""GPU: a device allocation that fails ends its call with GSOFA_ERR_ALLOC alone.
GSOFA_FAIL_ALLOC=k, read when a plan or a server worker's arena is made, fails
its k-th allocation once; whatever runs next on the same plan or server must
find every array it needs."""
import ctypes as C

import numpy as np
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


def _free_bytes():
    from gsofa_amd import _lib
    free, total = C.c_size_t(), C.c_size_t()
    assert _lib.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _columns(p):
    h = p.fetch_supernodal()
    return [getattr(h, k) for k in ("xsup", "supno", "xsub", "sub", "xlcol", "lrow", "xucol", "urow")]


@pytest.mark.parametrize("mode", ["reach", "block"])
def test_given_capacity_is_what_is_reserved(cases, mode):
    """output_capacity reserves 8 bytes an entry in every mode; all else of this
    plan is some 40 allocations of under 2 MB each."""
    import gsofa_amd as g
    A, o = cases[1]
    cap = 1 << 28
    with g.Plan(A) as p:
        p.execute()
        want = _columns(p)
    before = _free_bytes()
    with g.Plan(A, mode=mode, output_capacity=cap) as p:
        assert before - _free_bytes() <= 8 * cap + (128 << 20)
        p.execute()
        r = p.fetch()
        assert r.passes == 1
        assert_same_structure(r, o)
        for a, b in zip(_columns(p), want):
            np.testing.assert_array_equal(a, b)


def test_columns_without_room_for_the_lists(cases, monkeypatch):
    """The allocation that fails is, from some k on, that of the hand-off's longer
    record lists: the columns then come from the rows."""
    import gsofa_amd as g
    A, _ = cases[1]
    with g.Plan(A) as p:
        p.execute()
        want = _columns(p)
    for k in range(30, 50):
        print("case: hand-off, allocation", k, flush=True)
        monkeypatch.setenv("GSOFA_FAIL_ALLOC", str(k))
        try:
            p = g.Plan(A, mode="reach", output_capacity=1 << 16)
        except g.GsofaError as e:
            assert e.code == ERR_ALLOC
            continue
        with p:
            try:
                p.execute()
            except g.GsofaError as e:
                assert e.code == ERR_ALLOC
                p.execute()
            for _ in range(2):
                for a, b in zip(_columns(p), want):
                    np.testing.assert_array_equal(a, b)
            p.execute()
            for a, b in zip(_columns(p), want):
                np.testing.assert_array_equal(a, b)

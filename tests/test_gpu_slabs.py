"""GPU: device memory of released plans is kept for the plans after them (what
it holds by then is any), within a bound, and is given back."""
import ctypes as C
import threading

import pytest

from conftest import random_matrix
from gpu_util import assert_same_structure

pytestmark = pytest.mark.gpu


def _oracle(A):
    from oracle import oracle
    return oracle.symbfact(A.colbeg, A.colend, A.csr, A.n)


@pytest.fixture(scope="module")
def cases():
    import gsofa_amd as g
    import numpy as np
    rng = np.random.default_rng(3)
    mats = [g.gen_grid(14, 14, 14, nd_leaf=64, extra_prob=0.05, extra_dist=2, seed=2), g.gen_band(3000, 90, 6.0, 5),
            g.gen_grid(60, 60, 1, seed=4), random_matrix(rng, 700, 0.01)[0], g.gen_band(2000, 40, 4.0, 6)]
    return [(A, _oracle(A)) for A in mats]


@pytest.fixture
def pool():
    import gsofa_amd as g
    from gsofa_amd import _lib
    L = _lib.lib()

    class Pool:
        made = L._ZN5gsofa10slabs_madeEv
        release = staticmethod(g.release_memory)

        @staticmethod
        def idle():
            return L._ZN5gsofa10slabs_idleEi(0)
    Pool.made.restype = C.c_uint64
    L._ZN5gsofa10slabs_idleEi.restype = C.c_size_t
    L._ZN5gsofa10slabs_idleEi.argtypes = [C.c_int]
    Pool.release()
    assert Pool.idle() == 0
    yield Pool
    Pool.release()
    assert Pool.idle() == 0


def test_one_shot_calls_reuse_it(cases, pool):
    import gsofa_amd as g
    from gsofa_amd import _lib
    free, total = C.c_size_t(), C.c_size_t()
    before = pool.made()
    for A, o in cases:  # once each: no more than one slab a matrix
        assert_same_structure(g.symbfact(A), o)
    first = pool.made() - before
    assert 1 <= first <= len(cases)
    for _ in range(3):  # and in any order after that: no new one
        for A, o in reversed(cases):
            assert_same_structure(g.symbfact(A), o)
    assert pool.made() - before == first
    assert _lib.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    assert 0 < pool.idle() <= total.value // 16


def test_plans_alive_do_not_share(cases, pool):
    """A released plan's memory goes to one plan at a time; hand-offs and replays
    of those that live are unharmed."""
    import gsofa_amd as g
    plans = []
    for A, o in cases:
        with g.Plan(A) as p:
            p.execute()
        plans.append(g.Plan(A, graph=True))  # in the memory just released
    for _ in range(3):
        for p, (A, o) in zip(plans, cases):
            p.execute()
            assert_same_structure(p.fetch(), o)
    for p in plans:
        p.close()


def test_threads(cases, pool):
    import gsofa_amd as g
    bad = []

    def work(k):
        for i in range(12):
            A, o = cases[(i + k) % len(cases)]
            try:
                assert_same_structure(g.symbfact(A), o)
            except AssertionError as e:
                bad.append((k, i, str(e)))
    th = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad


def test_given_back_before_an_allocation_fails(cases, pool):
    import gsofa_amd as g
    A, o = cases[0]
    g.symbfact(A)
    assert pool.idle() > 0
    with pytest.raises(g.GsofaError) as e:  # 2^40 bytes
        g.Plan(A, mode="reach", output_capacity=1 << 37)
    assert e.value.code == -2
    assert pool.idle() == 0
    assert_same_structure(g.symbfact(A), o)

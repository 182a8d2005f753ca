"""GPU: the host memory behind results is made once and kept: pinned staging
buffers."""
import ctypes as C
import threading

import pytest

from gpu_util import assert_same_structure

pytestmark = pytest.mark.gpu


def _oracle(A):
    from oracle import oracle
    return oracle.symbfact(A.colbeg, A.colend, A.csr, A.n)


def test_staging_buffers_are_kept():
    """Large results fetched from six threads at once, over and over: the staging
    buffers made are those of four large copies, one more and two a thread."""
    import gsofa_amd as g
    from gsofa_amd import _lib
    made = _lib.lib()._ZN5gsofa10stage_madeEv
    made.restype = C.c_uint64
    A = g.gen_grid(27, 27, 27, nd_leaf=64, extra_prob=0.05, extra_dist=2, seed=2)
    o = _oracle(A)
    with g.Plan(A) as keep:  # buffers go back with the last plan
        keep.execute()
        before = made()
        plans = [g.Plan(A) for _ in range(6)]
        for p in plans:
            p.execute()
        out = {}

        def work(k):
            for _ in range(8):
                out[k] = plans[k].fetch()
        th = [threading.Thread(target=work, args=(k,)) for k in range(6)]
        for t in th:
            t.start()
        for t in th:
            t.join()
        assert made() - before <= 96 + 1 + 2 * 6
        for p in plans:
            p.close()
    for r in out.values():
        assert r.L_col.nbytes + r.U_col.nbytes > 24 << 20  # copied by twelve threads where there are buffers
        assert_same_structure(r, o)

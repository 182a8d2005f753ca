"""Entry numbers of class rows (32 bits) leave room for a loop's step past a
row's end; without it the number wraps and the loop does not end."""
import ctypes as C

import pytest

STEP = 4 * 1024 + 4 * 1024  # four steps of the largest workgroup, and its lanes' offsets


def _fits():
    from gsofa_amd import _lib
    f = _lib.lib()._ZN5gsofa9quot_fitsEmj
    f.argtypes, f.restype = [C.c_uint64, C.c_uint32], C.c_bool
    return f


@pytest.mark.parametrize("levels", [1, 7, 13, 19])
def test_last_step_stays_below_32_bits(levels):
    fits = _fits()
    most = (2 ** 32 - 1) // (levels + 1)
    for nnz in [most - d for d in (0, 1, 100, STEP // (levels + 1) // 2)] + [1, 1000, 10 ** 8 // levels]:
        ends_at = nnz * (levels + 1)
        assert fits(nnz, levels) <= (ends_at + STEP < 2 ** 32)
    # and what is clear of the limit is not refused
    assert fits((2 ** 32 - 2 ** 16) // (levels + 1), levels)
    assert not fits((2 ** 32 - 2 ** 16) // (levels + 1) + 1, levels)

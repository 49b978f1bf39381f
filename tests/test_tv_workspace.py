"""The workspace of the TV prox (gn_tv_work_bytes) around the size from which the dual field
is kept once; the library is loaded, nothing runs on a GPU."""
import ctypes

import pytest


@pytest.mark.parametrize("ndim", [2, 3])
def test_large_arrays_keep_the_field_once(ndim):
    from mripy_amd import _lib
    L = _lib.load()

    def fields(n, nt=1):
        shape = (ctypes.c_int64 * 3)(*([2] * (ndim - 1) + [n // nt >> (ndim - 1)] + [1] * (3 - ndim)))
        return L.gn_tv_work_bytes(ndim, shape, nt) / (16 * n)
    big = 1 << 29
    assert fields(1 << 20) == fields(big) == fields(big, 64) == 2 * ndim
    # field and divergence, as two kernels a step need
    assert fields(big + 8) == fields(2 * big) == fields(2 * big, 64) == fields(4 * big - 8) == ndim + 1

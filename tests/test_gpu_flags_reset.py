"""The error-set flag of one compress does not survive into the next on rows
outside the register top-k's shapes (cols % 4 != 0), where the separation's
row kernel clears it: an all-zero matrix has no error set, before and after a
matrix that has one."""
import ctypes

import numpy as np
import pytest

import bitsqz_amd as B

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(1, 129), (37, 1001)])
def test_flag_of_the_last_compress_is_gone(rows, cols):
    L = B.lib()
    B.compress_release()
    B.check(B.compress_initialize(rows, cols, 0.01, 0.02, -1, 1, B.QUANT_NONE, B.QUANT_NONE, B.NF4, B.INPUT_HOST), "init")
    try:
        x = np.random.default_rng(rows).standard_normal((rows, cols)).astype(np.float32)
        sizes = []
        for m in (np.zeros_like(x), x, np.zeros_like(x)):
            obj = ctypes.POINTER(B.PackedHeader)()
            B.check(L.bsq_compress(m.ctypes.data_as(ctypes.c_void_p), ctypes.byref(obj), None), "compress")
            handle = ctypes.cast(obj, ctypes.c_void_p)
            sizes.append(L.bsq_get_packed_size(handle))
            L.bsq_free(handle)
        assert sizes[0] == sizes[2] < sizes[1]
    finally:
        B.compress_release()

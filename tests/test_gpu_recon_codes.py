"""Packed factors at any byte address: bsq_device_decompress takes the
sections' pointers from the caller, who may have copied them into buffers of
their own.  Codes that start one, two or three bytes off a word must decode to
the bytes that the compress runtime's own arrays give."""
import ctypes

import numpy as np
import pytest

import bitsqz_amd as B
from _svdcase import lowrank

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("uv", [B.NF4, B.NF4_DQ])
@pytest.mark.parametrize("q", [24, 64, 72, 100])  # ranks below a slice, whole groups of eight, a remainder
def test_codes_off_word_alignment(q, uv):
    rows, cols = 131, 260
    x = lowrank(rows, cols, 120, 0.8, 0.01, seed=q)
    B.compress_release()
    B.decompress_release()
    B.check(B.compress_initialize(rows, cols, 0.0, 0.0, q, 1, uv, B.QUANT_NONE, B.QUANT_NONE, B.INPUT_DEVICE), "init")
    B.check(B.decompress_initialize(rows, cols, 0.0, 0.0, q, uv, B.QUANT_NONE, B.QUANT_NONE), "init")
    try:
        src, dst = B.DeviceBuffer.from_array(x), B.DeviceBuffer(rows * cols * 4)
        packed = B.device_compress(src)

        def decoded():
            B.device_decompress(packed, dst, rows * cols)
            B.device_synchronize()
            return dst.download(np.uint8, rows * cols * 4).tobytes()

        expect = decoded()
        own = [packed.d_codes[i] for i in range(4)]
        for off in (1, 2, 3):
            keep = []
            for i in (0, 2):  # U, V
                n = (packed.count[i] + 1) // 2
                keep.append(B.DeviceBuffer(n + off))
                at = ctypes.c_void_p(keep[-1].ptr.value + off)
                B.check(B.lib().bsq_memcpy_d2d(at, own[i], n), "copy")
                packed.d_codes[i] = at.value
            B.check(B.lib().bsq_stream_synchronize(None), "the copies' stream")
            assert decoded() == expect, off
    finally:
        B.compress_release()
        B.decompress_release()

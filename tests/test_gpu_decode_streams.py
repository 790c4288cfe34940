"""One decompress runtime, two streams: device-resident decodes run on the
compress runtime's stream, a host object's decode on the decompress runtime's
own.  Both use the runtime's buffers for the factors, so a host object decoded
while device-resident decodes are in flight, and the other way round, must give
the bytes that each gives alone."""
import numpy as np
import pytest

import bitsqz_amd as B
from _svdcase import lowrank

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q,uv,s", [(64, B.NF4, B.NF4), (128, B.QUANT_NONE, B.QUANT_NONE), (96, B.NF4_DQ, B.QUANT_NONE)])
def test_host_decode_beside_device_decodes(q, uv, s):
    rows, cols = 2048, 1536
    n = rows * cols
    a, b = (lowrank(rows, cols, 160, 0.7, 0.01, seed=i) for i in (q, q + 1))
    B.compress_release()
    B.decompress_release()
    B.check(B.compress_initialize(rows, cols, 0.0, 0.0, q, 1, uv, s, B.QUANT_NONE, B.INPUT_DEVICE), "init")
    B.check(B.decompress_initialize(rows, cols, 0.0, 0.0, q, uv, s, B.QUANT_NONE), "init")
    try:
        src, dst, host_dst = B.DeviceBuffer.from_array(b), B.DeviceBuffer(4 * n), B.DeviceBuffer(4 * n)
        host = B.compress(src)
        B.check(B.decompress_to_device(host, host_dst, n), "decompress")
        expect_host = host_dst.download(np.uint8, 4 * n).tobytes()
        src.upload(a)
        packed = B.device_compress(src)
        B.device_decompress(packed, dst, n)
        B.device_synchronize()
        expect = dst.download(np.uint8, 4 * n).tobytes()
        assert expect != expect_host
        for queued in (1, 40):
            for _ in range(queued):
                B.device_decompress(packed, dst, n)
            B.check(B.decompress_to_device(host, host_dst, n), "decompress")
            B.device_decompress(packed, dst, n)
            B.device_synchronize()
            assert host_dst.download(np.uint8, 4 * n).tobytes() == expect_host
            assert dst.download(np.uint8, 4 * n).tobytes() == expect
    finally:
        B.compress_release()
        B.decompress_release()

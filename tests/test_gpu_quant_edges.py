"""The encoder's fast and element-by-element forms (quant.hip) against the
oracle, bit for bit: block maxima of 1 so that values pass unscaled, with every
decision threshold, every edge of the code table's bins and their float
neighbours as values; the same under other scales; blocks with NaN, infinities,
zeros and subnormals between ordinary ones; lengths around a chunk of 8, a
block of 64 and a workgroup's tile, and one (2^25) that takes four chunks a
lane; an input that starts off 16 bytes."""
import ctypes

import numpy as np
import pytest

import bitsqz_amd as B
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def edge_values():
    base = np.concatenate([B.nf4_thresholds(), (np.arange(0, 257) / np.float32(128.0) - 1).astype(np.float32)])
    v = [base]
    for _ in range(3):
        v = [np.nextafter(v[0], np.float32(-4), dtype=np.float32)] + v + [np.nextafter(v[-1], np.float32(4), dtype=np.float32)]
    v = np.concatenate(v)
    v = v[np.abs(v) <= 1]
    v = v[: v.size // 63 * 63].reshape(-1, 63)
    return np.concatenate([np.ones((v.shape[0], 1), np.float32), v], axis=1).ravel()


def values(n, seed=0):
    """Edge values at scales 1, 2^-130 (1 / scale overflows once multiplied),
    2^100 and random, blocks with odd values among them, n in all."""
    e = edge_values()
    rng = np.random.default_rng(seed)
    x = np.concatenate([e, e * np.float32(2.0**-126), e * np.float32(2.0**100), e * np.float32(0.3),
                        rng.standard_normal(4096).astype(np.float32)])
    x = np.tile(x, -(-n // x.size))[:n].copy()
    for at, val in ((70, np.nan), (200, np.inf), (290, -np.inf), (333, -0.0), (400, 1e-42)):
        if at < n:
            x[at] = val
    x[640:704] = 0.0
    x[704:768] = 1e-44  # absmax below 2^-128: 1 / absmax is infinite
    return x


def check(x, method, got):
    q = O.quant_compress(x, method)
    scales, codes, dq = got
    assert scales.tobytes() == q.scales.tobytes()
    assert codes.tobytes() == q.codes.tobytes()
    if method == B.NF4_DQ:
        assert np.float32(dq).tobytes() == np.float32(q.dq).tobytes()


@pytest.mark.parametrize("method", [B.NF4, B.NF4_DQ])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 63, 65, 2047, 2049, 8191, 8193, 100003, (1 << 25) + 2049])
def test_encode_edges(method, n):
    x = values(n)
    if method == B.NF4_DQ:
        x = np.clip(x, -3e4, 3e4)  # one global scale: keep the small blocks above 0
    check(x, method, B.quant_compress(x, method))


@pytest.mark.parametrize("method", [B.NF4, B.NF4_DQ])
def test_encode_unaligned_input(method):
    x = values(10007)
    n, nb = x.size, (x.size + 63) // 64
    d = B.DeviceBuffer.from_array(np.concatenate([np.zeros(1, np.float32), x]))
    sf, su, dq, c = B.DeviceBuffer(4 * nb), B.DeviceBuffer(nb), B.DeviceBuffer(4), B.DeviceBuffer((n + 1) // 2)
    src = ctypes.c_void_p(d.ptr.value + 4)
    B.check(B.lib().bsq_quant_compress(src, n, method, sf.ptr, su.ptr, dq.ptr, c.ptr, None), "quant_compress")
    B.check(B.lib().bsq_stream_synchronize(None), "sync")
    scales = sf.download(np.float32, nb) if method == B.NF4 else su.download(np.uint8, nb)
    check(x, method, (scales, c.download(np.uint8, (n + 1) // 2), float(dq.download(np.float32, 1)[0])))

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


def below_two(rows, cols):
    """Rows whose blocks of 64 hold values up to the float below 2 at an NF4_DQ
    block scale of 1 (a scale code of 0 under the large value of row 0): the
    largest the code table takes, whose sum with the bin offset rounds up to
    the table's end.  Every third block also reaches 2, which the scan takes."""
    top = np.nextafter(np.float32(2.0), np.float32(0.0))
    v = np.array([top, -top, np.nextafter(top, np.float32(0.0)), 1.9375, 1.0, 0.5, -1.0, 0.0], np.float32)
    x = np.tile(v, rows * cols // 8).reshape(rows, cols)
    x[:, 64 * 2 + 5::192] = 2.0
    x[0, 0] = 4e6
    return x


@pytest.mark.parametrize("rows", [1, 33, 1 << 16])  # one chunk a lane, a tile's remainder, four chunks a lane
def test_encode_largest_table_value(rows):
    x = below_two(rows, 512).ravel()
    check(x, B.NF4_DQ, B.quant_compress(x, B.NF4_DQ))


@pytest.mark.parametrize("outlier", [0.0, 0.004])  # with the separation: its bitmap and row maxima
@pytest.mark.parametrize("cols", [512, 4096])
def test_fused_encode_largest_table_value(cols, outlier):
    rows = 36
    x = below_two(rows, cols)
    if outlier:
        x[:, : B.topk_num_columns(cols, outlier) + 1] = 5e6  # one a row stays and sets the global scale
    B.compress_release()
    B.check(B.compress_initialize(rows, cols, outlier, 0.01, -1, 1, B.QUANT_NONE, B.QUANT_NONE, B.NF4_DQ,
                                  B.INPUT_HOST), "init")
    try:
        data = B.compress(x)
    finally:
        B.compress_release()
    cfg = O.Config(rows, cols, outlier, 0.01, -1, 1, O.QUANT_NONE, O.QUANT_NONE, O.NF4_DQ)
    assert O.mask_pointer(data) == O.mask_pointer(O.compress(x, cfg).to_bytes())

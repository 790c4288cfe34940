"""The scalar E4M3 and E2M1 conversions of the legacy formats and of NF4_DQ's
block scales at the values where a code changes, bit for bit against the
oracle: every decision point (midpoints of neighbouring levels, the subnormal
and the saturation limits) with the floats on either side, zeros of both
signs, infinities, NaN and the smallest subnormals."""
import numpy as np
import pytest

import bitsqz_amd as B
from oracle import legacy as LG
from oracle import oracle as O
from test_gpu_legacy import mask_payload

pytestmark = pytest.mark.gpu


def around(values):
    v = np.asarray(values, dtype=np.float32)
    v = np.concatenate([v, np.nextafter(v, np.float32(np.inf)), np.nextafter(v, np.float32(-np.inf))])
    special = np.array([0.0, np.inf, np.nan, 1e-45, 3e38], dtype=np.float32)
    v = np.concatenate([v, special])
    return np.concatenate([v, -v])


def test_e4m3_decision_points():
    levels = np.abs(O.e4m3_decode_table()[:127].astype(np.float64))
    v = around(np.concatenate([levels, (levels[1:] + levels[:-1]) / 2, [448.0, 464.0, 480.0, 7.5 / 512, 8 / 512]]))
    assert B.e4m3_encode(v).tobytes() == O.e4m3_encode(v).tobytes()


@pytest.mark.parametrize("method", [LG.FP8, LG.FP4, LG.MXFP8, LG.MXFP4, LG.NVFP4])
@pytest.mark.parametrize("n", [8, 31, 32, 33, 1001])
def test_formats_at_decision_points(method, n):
    """Blocks whose largest magnitude is the format's own, so the scale is a
    power of two and the decision points reach the encoder as they are."""
    e4m3 = method in (LG.FP8, LG.MXFP8)
    top = 448.0 if e4m3 else 6.0
    levels = np.abs(O.e4m3_decode_table()[:127].astype(np.float64)) if e4m3 else np.array([0, 0.5, 1, 1.5, 2, 3, 4, 6])
    v = around(np.concatenate([levels, (levels[1:] + levels[:-1]) / 2]))
    v = v[~(np.isfinite(v) & (np.abs(v) > top))]
    x = np.random.default_rng(n).choice(v, size=n).astype(np.float32)
    x[::8] = top
    expect = LG.encode(method, x)
    assert mask_payload(method, B.legacy_encode_device(method, x)) == expect
    assert B.legacy_decode_device(method, expect, n).tobytes() == LG.decode(method, expect, n).tobytes()


@pytest.mark.parametrize("method", [LG.FP8, LG.FP4, LG.MXFP8, LG.MXFP4, LG.NVFP4])
def test_every_code_decodes(method):
    """All 256 code bytes at ordinary, subnormal and overflowing scales."""
    n = 512
    for scale in (1.0, 1e-38, 3e38):
        p = bytearray(LG.encode(method, np.full(n, scale, np.float32)))
        nib = method in (LG.FP4, LG.MXFP4, LG.NVFP4)
        codes = np.tile(np.arange(256, dtype=np.uint8), 1 if nib else 2).tobytes()
        p[-len(codes):] = codes
        assert B.legacy_decode_device(method, bytes(p), n).tobytes() == LG.decode(method, bytes(p), n).tobytes()

"""The reconstruction at low ranks (FP32 sums) and its hand-over to the two-piece
form, where a slice of 32 may be ragged.

Through bsq_reconstruct_lowrank against FP64: every depth of the FP32 kernel (16
to 128 in its steps) with ranks at its edges and off four, tiles of 64 cut in
both directions, matrices of a single row or column, and the ragged last slices
of the two-piece form without scratch.  Tolerance: an FP32 chain of k terms is
2^-24 sqrt(k) of the norms' product, 1.4e-6 at k = 600; 2e-6 of the result.

Through the ABI, bit for bit: packed factors decoded by the reconstruction, and
the subtraction from the residual (the error set), against the FP32 factors'
reconstruction of the same entry point."""
import numpy as np
import pytest

import bitsqz_amd as B
from _svdcase import abi_round_trip, check_sections, lowrank, outlier_columns

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 15, 16, 17, 32, 33, 48, 49, 63, 64, 65, 96, 97, 127, 128,
                               129, 131, 132, 156, 601])
@pytest.mark.parametrize("m,n", [(1, 70), (63, 3), (64, 64), (65, 129), (200, 61)])
def test_reconstruct_against_fp64(m, n, k):
    rng = np.random.default_rng(m * 1000 + n + k)
    U, S, V = (rng.standard_normal(s).astype(np.float32) for s in ((m, k), (k,), (n, k)))
    ref = (U * S).astype(np.float64) @ V.astype(np.float64).T
    assert np.linalg.norm(B.reconstruct(U, S, V) - ref) <= 2e-6 * np.linalg.norm(ref)


@pytest.mark.parametrize("k", [64, 65, 100, 128])  # both forms: 289 tiles of 128, more than there are CUs
def test_hand_over_by_size(k):
    m = n = 16 * 128 + 3
    rng = np.random.default_rng(k)
    U, S, V = (rng.standard_normal(s).astype(np.float32) for s in ((m, k), (k,), (n, k)))
    rows = [0, 1, 127, 128, 1000, m - 1]
    ref = (U[rows] * S).astype(np.float64) @ V.astype(np.float64).T
    got = B.reconstruct(U, S, V)[rows]
    assert np.linalg.norm(got - ref) <= 2e-6 * np.linalg.norm(ref)


@pytest.mark.parametrize("rows,cols,q,uv,s,ro,re", [
    (70, 131, 1, B.NF4, B.QUANT_NONE, 0.0, 0.05),
    (40, 44, 40, B.NF4, B.NF4_DQ, 0.0, 0.05),            # the packed sections outgrow the host decode's staging
    (66, 66, 24, B.NF4_DQ, B.NF4_DQ, 0.0, 0.05),         # and fit it but for their alignment
    (131, 70, 3, B.NF4_DQ, B.NF4, 0.02, 0.05),
    (129, 257, 8, B.NF4, B.NF4, 0.02, 0.03),
    (200, 300, 30, B.NF4_DQ, B.QUANT_NONE, 0.01, 0.03),
    (300, 200, 50, B.NF4, B.QUANT_NONE, 0.01, 0.03),
    (260, 323, 60, B.QUANT_NONE, B.QUANT_NONE, 0.0, 0.03),
    (260, 320, 96, B.NF4_DQ, B.NF4_DQ, 0.01, 0.0),
    (300, 301, 101, B.NF4, B.QUANT_NONE, 0.01, 0.02),
    (2603, 2600, 64, B.NF4, B.QUANT_NONE, 0.0, 0.004),   # factors decoded ahead of the kernel
    (2600, 2605, 63, B.NF4_DQ, B.QUANT_NONE, 0.0, 0.0),
    (300, 400, 129, B.NF4, B.QUANT_NONE, 0.01, 0.02),    # two pieces, ragged by one
    (400, 300, 150, B.QUANT_NONE, B.QUANT_NONE, 0.0, 0.02),
    (400, 300, 156, B.NF4_DQ, B.QUANT_NONE, 0.01, 0.02),
])
def test_packed_factors_bit_exact(rows, cols, q, uv, s, ro, re):
    x = outlier_columns(lowrank(rows, cols, min(160, rows, cols), 1.0, 0.01, seed=q + rows), 4, 40.0, seed=cols)
    data, out = abi_round_trip(x, ro, re, q, 1, uv, s)
    check_sections(x, data, out, ro, re, q, uv, s)
    src, dst = B.DeviceBuffer.from_array(x), B.DeviceBuffer(rows * cols * 4)
    packed = B.device_compress(src)
    B.device_decompress(packed, dst, rows * cols)
    B.device_synchronize()
    assert dst.download(np.float32, rows * cols).tobytes() == out.tobytes()
    B.compress_release()
    B.decompress_release()

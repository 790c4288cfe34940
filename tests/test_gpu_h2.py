"""The range finder's products with A as two f16 pieces (gemm_h2.hip), through
bsq_svd_lowrank with the built-in sketch (a caller's sketch takes the FP32
product), against the FP64 oracle given the same sketch.

Sizes sit at the edges of the kernel's 128 x 128 tiles, its pairs of 32-deep
slices and its 64-column operand planes (K padded with zeros; a last group of
fewer than eight k lies turned in the planes of products with A), both
orientations, rows of a length that is no multiple of four
(unaligned row starts), and matrices whose rows differ in scale by 2^28, with
zero rows among them.

Tolerance: each product carries the rounding of FP32 sums of K <= 1300 terms,
2^-24 sqrt(K) = 2e-6 of the result, and up to 2 niter + 2 products follow one
another; 2e-5 covers them with the orthonormalisations between."""
import numpy as np
import pytest

import bitsqz_amd as B
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TOL = 2e-5


def low_rank(m, n, r, rng):
    a = rng.standard_normal((m, r)) * np.arange(1, r + 1) ** -0.7
    return (a @ rng.standard_normal((r, n)) + 1e-3 * rng.standard_normal((m, n))).astype(np.float32)


def svd_and_oracle(A, q, it):
    m, n = A.shape
    k = max(1, min(q, m, n))
    U, S, V = B.svd_lowrank(A, q, it)
    R = B.gaussian(min(m, n) * k, 1241).reshape(min(m, n), k)
    return O.reconstruct(U, S, V), O.reconstruct(*O.svd_lowrank(A, q, it, R))


@pytest.mark.parametrize("m,n,q,it", [
    (64, 64, 8, 1),      # (the FP32 products, which matrices as small as this keep)
    (368, 240, 32, 1), (240, 384, 32, 1), (240, 256, 33, 2),  # either side of their limits
    (64, 64, 7, 1),      # one pair of slices, a single partial tile
    (127, 65, 1, 2),     # K remainder 1 and 63, one column
    (129, 190, 63, 1), (190, 129, 64, 1), (257, 1283, 65, 2), (1283, 257, 129, 1),
    (1024, 320, 128, 0), (320, 1024, 256, 2), (700, 703, 300, 1),
])
def test_products_at_tile_edges(m, n, q, it):
    A = low_rank(m, n, min(m, n, 96), np.random.default_rng(m * 7 + n))
    got, ref = svd_and_oracle(A, q, it)
    assert np.linalg.norm(got - ref) <= TOL * np.linalg.norm(ref)


@pytest.mark.parametrize("sketch", [False, True])
@pytest.mark.parametrize("q", [33, 257])  # planes from the orthonormalisation, and split from FP32 bases
@pytest.mark.parametrize("m,n", [(513, 522), (523, 516), (517, 518), (519, 576), (584, 520)])
def test_last_group_of_k(m, n, q, sketch):
    """Every remainder of K by eight, in both products."""
    A = low_rank(m, n, 96, np.random.default_rng(m + 3 * n))
    if not sketch:
        got, ref = svd_and_oracle(A, q, 1)
    else:
        R = np.random.default_rng(q).standard_normal((min(m, n), q)).astype(np.float32)
        got, ref = O.reconstruct(*B.svd_lowrank(A, q, 1, R)), O.reconstruct(*O.svd_lowrank(A, q, 1, R))
    assert np.linalg.norm(got - ref) <= TOL * np.linalg.norm(ref)


@pytest.mark.parametrize("m,n", [(300, 517), (517, 300)])
def test_rows_of_very_different_scale(m, n):
    """A rank-8 matrix (recovered exactly by q = 16) with row scales 2^-14 ..
    2^14 and a few zero rows: every row comes back to its own scale's
    accuracy, since each row is scaled by itself."""
    rng = np.random.default_rng(n)
    A = (rng.standard_normal((m, 8)) @ rng.standard_normal((8, n))).astype(np.float32)
    A = np.ldexp(A, rng.integers(-14, 15, size=(m, 1))).astype(np.float32)
    A[::37] = 0.0
    U, S, V = B.svd_lowrank(A, 16, 1)
    err = np.linalg.norm(O.reconstruct(U, S, V) - A, axis=1)
    assert np.all(err <= TOL * np.linalg.norm(A, axis=1))

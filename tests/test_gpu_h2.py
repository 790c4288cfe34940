"""The range finder's products with A as two f16 pieces (gemm_h2.hip), through
bsq_svd_lowrank with the built-in sketch (a caller's sketch takes the FP32
product), against the FP64 oracle given the same sketch.

Sizes sit at the edges of the kernel's 128 x 128 tiles, its pairs of 32-deep
slices and its 64-column operand planes (K padded with zeros; a last group of
fewer than eight k lies turned in the planes of products with A), both
orientations, rows of a length that is no multiple of four
(unaligned row starts), and matrices whose rows differ in scale by 2^28, with
zero rows among them.

Tolerance: FP32 sums of K <= 1300 terms round by 2^-24 sqrt(K) = 2e-6 of the
result; the two-piece products with their sums came to 1.1e-7 .. 4.8e-7 of it
over these sizes, orthonormalisations and all, and 2e-6 is four times that.  That
they are no further off than FP32 sums of the same products is held by the last
two tests (0.35 to 0.56 of a plain chain's error when they were written)."""
import numpy as np
import pytest

import bitsqz_amd as B
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TOL = 2e-6


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


def chain(A, Bm):
    """A Bm with every sum a chain of FP32 additions in the order of k."""
    out = np.zeros((A.shape[0], Bm.shape[1]), np.float32)
    for k in range(A.shape[1]):
        out += A[:, k:k + 1] * Bm[k]
    return out


def fp32_chain_svd(A, R, it):
    """The randomised SVD with its products with A as FP32 chains and the rest in 64 bits."""
    tr = A.shape[0] < A.shape[1]
    Aw = np.ascontiguousarray(A.T if tr else A)
    At = np.ascontiguousarray(Aw.T)
    orth = lambda X: np.linalg.qr(X.astype(np.float64))[0].astype(np.float32)  # noqa: E731
    Q = orth(chain(Aw, R))
    for _ in range(it):
        Q = orth(chain(Aw, orth(chain(At, Q))))
    Y = chain(At, Q).astype(np.float64)
    low = Q.astype(np.float64) @ Y.T
    return low.T if tr else low


@pytest.mark.parametrize("columns", [0, 8])  # columns scaled by 50, as activations have them
@pytest.mark.parametrize("m,n,q", [(600, 520, 16), (520, 1000, 40), (1000, 700, 100)])
def test_error_no_larger_than_fp32_sums(m, n, q, columns):
    """The split's own error and the matrix instructions' sums together stay
    below the rounding of FP32 sums of the same products."""
    rng = np.random.default_rng(q + columns)
    A = low_rank(m, n, 200, rng)
    A[:, rng.permutation(n)[:columns]] *= 50
    got, ref = svd_and_oracle(A, q, 2)
    R = B.gaussian(min(m, n) * q, 1241).reshape(min(m, n), q)
    fp32 = np.linalg.norm(fp32_chain_svd(A, R, 2) - ref)
    assert np.linalg.norm(got - ref) <= fp32


@pytest.mark.parametrize("k", [136, 256, 1030])
@pytest.mark.parametrize("kind", ["normal", "lognormal", "one_signed", "decaying", "outlier"])
def test_reconstruction_error_no_larger_than_fp32_sums(k, kind):
    """The same through bsq_reconstruct_lowrank (one product, two pieces above rank 128)."""
    rng = np.random.default_rng(k)
    U, V = rng.standard_normal((300, k)), rng.standard_normal((260, k))
    S = np.ones(k)
    if kind == "lognormal":
        U, V = U * np.exp(rng.standard_normal(U.shape)), V * np.exp(rng.standard_normal(V.shape))
    elif kind == "one_signed":
        U, V = np.abs(U), np.abs(V)
    elif kind == "decaying":
        S = np.arange(1, k + 1) ** -1.0
    elif kind == "outlier":
        U[:, 5] *= 50
    U, S, V = U.astype(np.float32), S.astype(np.float32), V.astype(np.float32)
    US = U * S
    ref = US.astype(np.float64) @ V.astype(np.float64).T
    fp32 = np.linalg.norm(chain(US, np.ascontiguousarray(V.T)) - ref)
    assert np.linalg.norm(B.reconstruct(U, S, V) - ref) <= fp32

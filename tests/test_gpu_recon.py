"""bsq_reconstruct_lowrank (recon.hip) at the edges of its kernels: FP32 sums (at
these sizes ranks to 128), the two-piece form above in slices of 32 with every
kind of remainder, tiles of 64 and 128, rows of factors that start off 16 bytes,
and the values whose two-piece form needs care: infinities, NaN, zero rows and
rows of very different scale.

Tolerance: an entry is a sum of k products of FP32 values, each carried to
2^-22 of its row's scale at worst and summed in FP32: 2^-22 sqrt(k) of the
norms' product; 2e-6 of the whole result for these ranks."""
import numpy as np
import pytest

import bitsqz_amd as B

pytestmark = pytest.mark.gpu


def factors(m, n, k, seed):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((m, k)).astype(np.float32), rng.random(k).astype(np.float32),
            rng.standard_normal((n, k)).astype(np.float32))


def exact(U, S, V):
    with np.errstate(all="ignore"):
        return (U * S).astype(np.float64) @ V.astype(np.float64).T


@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (64, 64, 31), (65, 130, 17), (127, 129, 32), (129, 127, 33),
                                   (128, 128, 63), (200, 261, 64), (261, 200, 95), (129, 127, 129), (200, 261, 159), (261, 200, 160),
                                   (130, 259, 1030)])
def test_reconstruct_edges(m, n, k):
    U, S, V = factors(m, n, k, m + n + k)
    ref = exact(U, S, V)
    assert np.linalg.norm(B.reconstruct(U, S, V) - ref) <= 2e-6 * np.linalg.norm(ref)


@pytest.mark.parametrize("k", [20, 40, 130, 131, 256])
def test_reconstruct_non_finite_and_scales(k):
    U, S, V = factors(300, 200, k, k)
    U[7, 3], U[9, 5], U[20], V[30] = np.inf, np.nan, 0.0, 0.0
    V[11, 2], V[13, 1] = -np.inf, np.nan
    scale = np.ldexp(1.0, np.random.default_rng(k).integers(-40, 41, 300)).astype(np.float32)
    U *= scale[:, None]
    with np.errstate(all="ignore"):
        got, ref = B.reconstruct(U, S, V), exact(U, S, V).astype(np.float32)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    rows = [r for r in range(300) if r not in (7, 9)]  # every row to its own scale
    cols = [c for c in range(200) if c not in (11, 13)]
    d = (got - ref)[np.ix_(rows, cols)].astype(np.float64)
    assert np.all(np.linalg.norm(d, axis=1) <= 2e-6 * np.linalg.norm(ref[np.ix_(rows, cols)], axis=1))

"""The tridiagonalisation's hand-over above rank 256: the first k - 256 columns
by one launch each, the last 256 in the register kernel (sytrd.hip), through
bsq_svd_lowrank against the FP64 oracle with the same sketch.

Sizes: the smallest hand-over (one and two columns, either parity of the
double-buffered product), one in the middle, and the largest.  Tolerance: FP32
sums of up to 700 terms round by 2^-24 sqrt(700) = 1.6e-6 of the result; the
whole factorisation came to 4.3e-7 .. 6.7e-7 of it over these cases (S to 2.6e-7
at most), and 3e-6 is four times that."""
import numpy as np
import pytest

import bitsqz_amd as B
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rank", [96, 600])  # a singular Gram matrix, and a regular one
@pytest.mark.parametrize("q", [257, 258, 385, 511, 512])
def test_hand_over(q, rank):
    rng = np.random.default_rng(q + rank)
    a = rng.standard_normal((700, rank)) * np.arange(1, rank + 1) ** -0.7
    A = (a @ rng.standard_normal((rank, 600))).astype(np.float32)
    U, S, V = B.svd_lowrank(A, q, 1)
    R = B.gaussian(600 * q, 1241).reshape(600, q)
    Uo, So, Vo = O.svd_lowrank(A, q, 1, R)
    got, ref = O.reconstruct(U, S, V), O.reconstruct(Uo, So, Vo)
    assert np.linalg.norm(got - ref) <= 3e-6 * np.linalg.norm(ref)
    assert np.linalg.norm(S - So) <= 3e-6 * np.linalg.norm(So)

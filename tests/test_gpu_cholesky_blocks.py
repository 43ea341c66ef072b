"""The blocked Cholesky solve at the edges of its blocks (panels of 32, block
columns of 128, 64 x 64 tiles, and the tile order above 32 rows of tiles).
Tolerance: the normwise backward error of a Cholesky solve is at most about
4 n u (Higham, Accuracy and Stability, theorem 10.4), whatever the condition."""
import numpy as np
import pytest

import rbmongpu_amd as R

pytestmark = pytest.mark.gpu


def spd(n, seed, decades=0.0):
    r = np.random.default_rng(seed)
    B = r.normal(size=(n, n)) + 1j * r.normal(size=(n, n))
    B *= 10.0 ** (-decades * np.arange(n) / (2 * n))
    return B @ B.conj().T / n + 10.0 ** -decades * np.eye(n), r.normal(size=n) + 1j * r.normal(size=n)


@pytest.mark.parametrize("decades", [0.0, 8.0])
@pytest.mark.parametrize("n", [2, 63, 65, 96, 97, 127, 128, 130, 161, 192, 223, 256, 289, 384, 2177, 2240, 2305])
def test_backward_error(n, decades):
    print(f"[cholesky blocks] n={n} decades={decades}", flush=True)
    A, b = spd(n, n, decades)
    x = R.cholesky_solve(A, b)
    r = np.linalg.norm(A @ x - b) / (np.linalg.norm(A) * np.linalg.norm(x) + np.linalg.norm(b))
    assert r <= 4 * n * 2.0 ** -53


@pytest.mark.parametrize("k", [0, 5, 31, 32, 63, 64, 127, 128, 159, 160, 255, 256, 299])
def test_first_bad_pivot_is_reported(k):
    A, b = spd(300, 7)
    A[k, k] = -3.0
    with pytest.raises(ValueError, match=rf"pivot {k + 1}\)"):
        R.cholesky_solve(A, b)

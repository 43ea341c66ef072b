"""Cholesky solve where the last 32-column panel or the last 128-row block is
nearly empty: columns and rows past the matrix are left out of the steps.  FP64
end to end (1e-10 of the solution), and a pivot that is not positive in the last
row keeps its index."""
import numpy as np
import pytest

import rbmongpu_amd as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 7, 9, 30, 34, 63, 65, 95, 97, 130, 161, 193, 226])
def test_remainders(n):
    r = np.random.default_rng(n)
    B = r.normal(size=(n, n)) + 1j * r.normal(size=(n, n))
    A = B @ B.conj().T / n + 0.5 * np.eye(n)
    b = r.normal(size=n) + 1j * r.normal(size=n)
    ref = np.linalg.solve(A, b)
    assert np.max(np.abs(R.cholesky_solve(A, b) - ref)) <= 1e-10 * np.max(np.abs(ref))
    A[n - 1, n - 1] = -1.0
    with pytest.raises(ValueError, match=rf"pivot {n}\)"):
        R.cholesky_solve(A, b)

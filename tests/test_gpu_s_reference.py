"""get_S_matrix at the edges of its tiles (16 sign rows, 32 real columns, 4
row tiles a wavefront, 4-state steps), with a visible bias and in a sector,
against numpy in FP64 (the complex128 bar, 1e-10 of the largest entry)."""
import numpy as np
import pytest

import rbmongpu_amd as R
from oracle import oracle as O

pytestmark = pytest.mark.gpu


# sign rows 1 + N (N + 1) / 2: 16 at N = 5, 67 (5 tiles, 2 groups) at 11; real
# columns (M + 1)(M + 2): 30 at M = 4, 42 at 5
@pytest.mark.parametrize("N,M,with_a,sector", [(1, 1, False, None), (2, 4, True, None), (5, 5, False, None),
                                               (6, 4, False, 0), (11, 3, True, None), (9, 14, False, 1)])
def test_reference_s_matrix_tiles(N, M, with_a, sector):
    r = np.random.default_rng(10 * N + M)
    b = 0.3 * (r.normal(size=M) + 1j * r.normal(size=M))
    W = 0.3 * (r.normal(size=(N, M)) + 1j * r.normal(size=(N, M)))
    a = 0.1 * (r.normal(size=N) + 1j * r.normal(size=N)) if with_a else None
    psi = R.Psi(np.zeros(N), np.zeros(N), b, W, 1.0, False, True, a=a, precision=64)
    ex = R.ExactSummation(N, True)
    k = np.arange(2 ** N)
    s = ((k[:, None] >> np.arange(N)) & 1) * 2.0 - 1
    if sector is not None:
        ex.set_total_z_symmetry(sector)
        s = s[s.sum(1) == sector]
    T = O.tanh(b[None, :] + s @ W)
    rows = [np.zeros((len(s), 2 * N)), T, (s[:, :, None] * T[:, None, :]).reshape(len(s), -1)] + ([s] if with_a else [])
    Ok = np.concatenate(rows, axis=1).astype(complex)
    ref = Ok.T @ Ok.conj() / len(s)
    S = R.get_S_matrix(psi, ex)
    assert S.shape == ref.shape
    assert np.max(np.abs(S - ref)) <= 1e-10 * np.max(np.abs(ref))

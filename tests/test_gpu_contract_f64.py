"""The FP64 O_k contraction at the edges of its tiles (16 rows, 16 real columns,
5 row tiles a wavefront, 4-sample K steps) against numpy on the samples of the
call.  FP64 end to end: the complex128 bar, 1e-10 of the largest entry."""
import numpy as np
import pytest

import rbmongpu_amd as R
from oracle import oracle as O
from rbmongpu_amd import hamiltonians as HAM

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,M,chains,samples", [(3, 1, 1, 5), (15, 7, 33, 1), (16, 8, 50, 3), (79, 3, 41, 2), (80, 23, 64, 2),
                                                (128, 5, 37, 1)])
def test_contraction_shapes(N, M, chains, samples):
    r = np.random.default_rng(N)
    b = 0.1 * (r.normal(size=M) + 1j * r.normal(size=M))
    W = 0.1 * (r.normal(size=(N, M)) + 1j * r.normal(size=(N, M)))
    psi = R.Psi(np.zeros(N), np.zeros(N), b, W, 1.0, False, True, precision=64)
    mc = R.MonteCarloLoop(chains * samples, 1, 3, chains, True, seed=4)
    g, E = R.ExpectationValue(True).gradient(psi, R.Operator(*HAM.tfim_1d(N), True), mc)
    words, _, el = mc.last_samples()
    s = np.stack([(words[:, i >> 6] >> np.uint64(i & 63)) & np.uint64(1) for i in range(N)], axis=1).astype(float) * 2 - 1
    T = O.tanh(b[None, :] + s @ W)
    y = (2.0 / len(s)) * (el - el.mean())[:, None] * T.conj()
    ref = np.concatenate([y.sum(0), (s.T @ y).ravel()])
    assert abs(E - el.mean()) <= 1e-10 * abs(el.mean())
    assert np.max(np.abs(g[2 * N:] - ref)) <= 1e-10 * np.max(np.abs(y)) * len(s)

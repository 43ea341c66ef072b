"""A unit whose my_tanh overflows (FP32 past 250, FP64 past 1e19, where log psi is
still finite) spoils its own parameters' gradients and no others'.  The visible
biases' against numpy on the samples of the call, at the bar of their FP64 sums
(1e-10) and, with FP32 local energies, 1e-5."""
import numpy as np
import pytest

import rbmongpu_amd as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,b0,estimator,bar", [(64, 1e20, "hermitian", 1e-10), (64, 1e20, "E_k", 1e-10),
                                                        (32, 1e3, "E_k", 1e-5)])
@pytest.mark.parametrize("N,M", [(5, 3), (17, 9)])
def test_other_parameters_stay_finite(N, M, precision, b0, estimator, bar):
    r = np.random.default_rng(N)
    b = 0.1 * (r.normal(size=M) + 1j * r.normal(size=M))
    W = 0.1 * (r.normal(size=(N, M)) + 1j * r.normal(size=(N, M)))
    b[0], W[:, 0] = b0, 0
    a = (0.3 * r.normal(size=N)).astype(complex)
    psi = R.Psi(np.zeros(N), np.zeros(N), b, W, 1.0, False, True, a=a, precision=precision)
    # a chain of sigma^z sigma^z and a field: a diagonal operator forms no ratios of psi
    c = np.concatenate([r.normal(size=N - 1), r.normal(size=N)]).astype(complex)
    types = np.zeros((2 * N - 1, 3), np.int32)
    idx = -np.ones((2 * N - 1, 3), np.int32)
    types[:N - 1, :2], idx[:N - 1, 0], idx[:N - 1, 1] = 3, np.arange(N - 1), np.arange(1, N)
    types[N - 1:, 0], idx[N - 1:, 0] = 3, np.arange(N)
    mc = R.MonteCarloLoop(600, 1, 3, 200, True, seed=4)
    g, E = R.ExpectationValue(True).gradient(psi, R.Operator(c, types, idx, True), mc, estimator=estimator)
    words, _, _ = mc.last_samples()
    s = ((words[:, :1] >> np.arange(N, dtype=np.uint64)) & np.uint64(1)).astype(float) * 2 - 1
    e = (s[:, :-1] * s[:, 1:]) @ c[:N - 1].real + s @ c[N - 1:].real
    ref = (2.0 / len(s)) * (s * (e - e.mean())[:, None]).sum(0)
    assert abs(E - e.mean()) <= bar * np.abs(c).sum()
    assert np.all(np.abs(g[-N:] - ref) <= bar * 2 * np.abs(c).sum())
    assert np.all(np.isfinite(g[2 * N + 1:2 * N + M]))

"""Which states of 2048 parameters and more keep the pairs: a unit that follows
one spin leaves little variance in O_(i,j) = s_i T_j, also where the spin is
polarised, and goes to the Gram product without the moments being formed."""
import numpy as np
import pytest

import rbmongpu_amd as R
from oracle import oracle as O

pytestmark = pytest.mark.gpu
N = M = 45


def s_and_gram_launches(a, W, precision):
    psi = R.Psi(np.zeros(N), np.zeros(N), np.zeros(M, complex), W, 1.0, False, True, a=a, precision=precision)
    mc = R.MonteCarloLoop(4000, 1, 5, 2000, True, seed=2)
    R.timing_enable(True)
    R.timing_reset()
    S = R.get_S_matrix_centred(psi, mc)
    launches = R.timing_query("s_gram")[1]
    R.timing_enable(False)
    words, _, _ = mc.last_samples()
    s = np.stack([(words[:, 0] >> np.uint64(i)) & np.uint64(1) for i in range(N)], axis=1).astype(float) * 2 - 1
    T = O.tanh(s @ W)
    Ok = np.concatenate([T, (s[:, :, None] * T[:, None, :]).reshape(len(s), -1)] + ([s.astype(complex)] if a is not None else []), 1)
    c = Ok - Ok.mean(0)
    return S, c.conj().T @ c / len(s), launches


@pytest.mark.parametrize("pol,spread,precision", [(0.97, 1e-4, 64), (-0.9, 1e-4, 64), (0.0, 1e-3, 32)])
def test_units_that_follow_one_spin(pol, spread, precision):
    r = np.random.default_rng(4)
    a = np.full(N, 0.5 * np.arctanh(pol), complex)
    W = 0.4 * np.eye(N) + spread * (r.normal(size=(N, M)) + 1j * r.normal(size=(N, M)))
    if precision == 32:
        W = W.astype(np.complex64).astype(complex)
    S, ref, launches = s_and_gram_launches(a, W, precision)
    k = M + np.arange(N) * M + np.arange(N)   # W_ii
    print(f"W_ii {np.max(np.abs(S[k, k] - ref[k, k]) / ref[k, k].real):.1e}", flush=True)
    assert launches == 1
    # (without the visible biases' own variances: sums of two equal squares over
    # and over, whose FP32 rounding in the Gram product always goes one way)
    e = np.abs(S - ref)
    v = np.arange(M + N * M, len(S))
    e[v, v] = 0
    assert np.max(e) <= 1e-5 * np.max(np.abs(ref))
    # centred rows in FP32: 6e-8 of |T| against a spread of at least 1e-4 |T|
    assert np.all(np.abs(S[k, k] - ref[k, k]) <= 1e-3 * np.abs(ref[k, k]))


@pytest.mark.parametrize("with_a", [False, True])
def test_constant_units_keep_the_pairs(with_a):
    """Units without weights have no spread: S has nothing to lose there."""
    r = np.random.default_rng(5)
    W = (0.1 * (r.normal(size=(N, M)) + 1j * r.normal(size=(N, M)))).astype(np.complex64).astype(complex)
    W[:, ::7] = 0
    a = np.full(N, 0.3, complex) if with_a else None
    S, ref, launches = s_and_gram_launches(a, W, 32)
    assert launches == 1
    assert np.max(np.abs(S - ref)) <= 1e-6 * np.max(np.abs(ref))   # the Gram product leaves 2.5e-6

"""The centred S-matrix from pairs of spins and units, at the edges of its
tiles (16 sign rows, 48 real columns, 32-sample blocks, 4096-sample flushes)
and one model that it leaves to the Gram product, against FP64.  The bar is the
complex64 one: 1e-5 of the largest entry."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def centred(b, W, a, s, w):
    from oracle import oracle as O
    T = O.tanh(b[None, :] + s @ W)
    Ok = np.concatenate([T, (s[:, :, None] * T[:, None, :]).reshape(len(s), -1)] + ([s.astype(complex)] if a is not None else []), 1)
    w = w / w.sum()
    c = (Ok - (w[:, None] * Ok).sum(0)) * np.sqrt(w)[:, None]
    return c.conj().T @ c


def model(N, M, sigma, precision, with_a, seed=0):
    import rbmongpu_amd as R
    r = np.random.default_rng(seed + 100 * N + M)
    b = sigma * (r.normal(size=M) + 1j * r.normal(size=M))
    W = sigma * (r.normal(size=(N, M)) + 1j * r.normal(size=(N, M)))
    a = 0.1 * (r.normal(size=N) + 1j * r.normal(size=N)) if with_a else None
    if precision == 32:
        b, W = b.astype(np.complex64).astype(complex), W.astype(np.complex64).astype(complex)
    return b, W, a, R.Psi(np.zeros(N), np.zeros(N), b, W, 1.0, False, True, a=a, precision=precision)


def spins_of(words, N):
    return np.stack([(words[:, i >> 6] >> np.uint64(i & 63)) & np.uint64(1) for i in range(N)], axis=1).astype(float) * 2 - 1


# 2048 parameters and more.  9 spins: 3 row tiles, 43 056 columns; 16: visible
# bias and complex128 records
@pytest.mark.parametrize("N,M,precision,with_a", [(9, 205, 32, False), (12, 170, 64, True)])
def test_pairs_exact(N, M, precision, with_a):
    import rbmongpu_amd as R
    from oracle import oracle as O
    b, W, a, psi = model(N, M, 0.05, precision, with_a)
    ex = R.ExactSummation(N, True)
    psi.normalize(ex)
    S = R.get_S_matrix_centred(psi, ex)
    words = np.zeros((2 ** N, 2), np.uint64)
    words[:, 0] = np.arange(2 ** N)
    s = spins_of(words, N)
    lp = O.log_psi(O.RBM(b, W), words) + (s @ a if with_a else 0)
    ref = centred(b, W, a, s, np.exp(2 * (lp.real - lp.real.max())))
    assert np.array_equal(S, S.conj().T)
    assert np.max(np.abs(S - ref)) <= 1e-5 * np.max(np.abs(ref))


# 127 spins: 43 row groups; 40 and 50: one sample, ragged blocks; 22: several
# flushes in one split
@pytest.mark.parametrize("N,M,chains,samples", [(127, 16, 131, 1), (40, 50, 1, 1), (22, 90, 97, 3), (22, 90, 4100, 2)])
def test_pairs_monte_carlo(N, M, chains, samples):
    import rbmongpu_amd as R
    b, W, a, psi = model(N, M, 0.05, 32, N == 40)
    mc = R.MonteCarloLoop(chains * samples, 1, 5, chains, True, seed=2)
    S = R.get_S_matrix_centred(psi, mc)
    words, _, _ = mc.last_samples()
    ref = centred(b, W, a, spins_of(words, N), np.ones(len(words)))
    scale = np.max(np.abs(ref)) if len(words) > 1 else 1.0   # one sample: S = 0
    assert np.max(np.abs(S - ref)) <= 1e-5 * scale


def test_units_that_follow_one_spin_keep_their_accuracy():
    """W close to a diagonal: O_(i,i) hardly varies, and its small variance
    must come from the centred rows."""
    import rbmongpu_amd as R
    N = M = 45
    r = np.random.default_rng(3)
    W = (0.4 * np.eye(N) + 1e-3 * (r.normal(size=(N, M)) + 1j * r.normal(size=(N, M)))).astype(np.complex64).astype(complex)
    b = np.zeros(M, complex)
    psi = R.Psi(np.zeros(N), np.zeros(N), b, W, 1.0, False, True)
    mc = R.MonteCarloLoop(600, 1, 5, 200, True, seed=2)
    S = R.get_S_matrix_centred(psi, mc)
    words, _, _ = mc.last_samples()
    ref = centred(b, W, None, spins_of(words, N), np.ones(len(words)))
    k = M + np.arange(N) * M + np.arange(N)   # W_ii
    # centred rows in FP32: rounding 6e-8 of |T| against a spread of ~1e-3 |T|
    assert np.max(np.abs(S - ref)) <= 1e-5 * np.max(np.abs(ref))
    assert np.all(np.abs(S[k, k] - ref[k, k]) <= 1e-3 * np.abs(ref[k, k]))

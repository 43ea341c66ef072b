"""The centred S-matrix of ensembles whose weights are not all 1 (exact sums,
runs of a learned chain) where its entries are small differences of large
moments: polarised spins, units far from zero, a wavefunction that is not
normalised.  At least 2048 parameters, against FP64.

Tolerances: 1e-5 of the largest entry (the complex64 bar).  An entry is a sum
over the samples of products whose absolute values add up to at most
sqrt(S_kk S_ll); FP32 sums of 4096 samples are 384 rounded additions of a
running sum (three products per 32 samples), 2^-23 each, 4.6e-5: 1e-4 of
sqrt(S_kk S_ll) with the rounding of the factors."""
import numpy as np
import pytest

import rbmongpu_amd as R
from oracle import oracle as O
from rbmongpu_amd import hamiltonians as H

pytestmark = pytest.mark.gpu
N, M = 12, 170


def model(pol, b0, spread, precision, seed):
    """|psi|^2 close to a product with <s_i> = pol, biases around b0."""
    r = np.random.default_rng(seed)
    b = b0 + 0.1 * (r.normal(size=M) + 1j * r.normal(size=M))
    W = spread * (r.normal(size=(N, M)) + 1j * r.normal(size=(N, M)))
    a = np.full(N, 0.5 * np.arctanh(pol), complex)
    if precision == 32:
        a, b, W = (np.asarray(x, np.complex64).astype(complex) for x in (a, b, W))
    return a, b, W, R.Psi(np.zeros(N), np.zeros(N), b, W, 1.0, False, True, a=a, precision=precision)


def spins_of(words):
    return ((words[:, :1] >> np.arange(N, dtype=np.uint64)) & np.uint64(1)).astype(float) * 2 - 1


def basis():
    words = np.zeros((2 ** N, 2), np.uint64)
    words[:, 0] = np.arange(2 ** N)
    return words, spins_of(words)


def reference(b, W, s, w, n):
    """(1 / n) sum w (O_k - o_k)^* (O_l - o_l) with o = (1 / n) sum w O."""
    T = O.tanh(b[None, :] + s @ W)
    Ok = np.concatenate([T, (s[:, :, None] * T[:, None, :]).reshape(len(s), -1), s.astype(complex)], axis=1)
    c = (Ok - (w[:, None] * Ok).sum(0) / n) * np.sqrt(w)[:, None]
    return c.conj().T @ c / n


def check(S, ref):
    d = np.sqrt(np.diag(ref).real)
    k = d > 1e-12 * d.max()
    print(f"of the largest {np.abs(S - ref).max() / np.abs(ref).max():.1e}, scaled "
          f"{(np.abs(S - ref)[np.ix_(k, k)] / np.outer(d[k], d[k])).max():.1e}", flush=True)
    assert np.array_equal(S, S.conj().T)
    assert np.abs(S - ref).max() <= 1e-5 * np.abs(ref).max()
    assert np.all(np.abs(S - ref)[np.ix_(k, k)] <= 1e-4 * np.outer(d[k], d[k]))


@pytest.mark.parametrize("pol,b0,spread,precision", [(0.0, 0.5, 0.01, 64), (0.0, 0.5, 0.01, 32), (0.97, 0.5, 0.05, 64),
                                                     (0.999, 0.5, 0.05, 32), (0.9999, 0.5, 0.01, 64), (0.0, 3.0, 0.05, 64)])
def test_exact_sum(pol, b0, spread, precision):
    a, b, W, psi = model(pol, b0, spread, precision, seed=11)
    ex = R.ExactSummation(N, True)
    psi.normalize(ex)
    words, s = basis()
    lp = (O.log_psi(O.RBM(b, W), words) + s @ a).real
    w = np.exp(2 * (lp - lp.max()))
    check(R.get_S_matrix_centred(psi, ex), reference(b, W, s, w * (len(w) / w.sum()), len(w)))


@pytest.mark.parametrize("z", [4.0, 0.25])
def test_exact_sum_that_is_not_normalised(z):
    """sum w = z n: S keeps its definition and stays positive."""
    a, b, W, psi = model(0.3, 0.5, 0.05, 64, seed=12)
    ex = R.ExactSummation(N, True)
    psi.normalize(ex)
    psi.prefactor = psi.prefactor * np.sqrt(z)
    words, s = basis()
    lp = (O.log_psi(O.RBM(b, W), words) + s @ a).real
    w = np.exp(2 * (lp - lp.max()))
    S = R.get_S_matrix_centred(psi, ex)
    check(S, reference(b, W, s, w * (z * len(w) / w.sum()), len(w)))
    op = R.Operator(*H.tfim_1d(N, 1.0, 0.9), True)
    upd, _ = R.sr_update(psi, op, ex, 1e-2)
    g, _ = R.ExpectationValue(True).gradient(psi, op, ex)
    x, g = upd[2 * N:], g[2 * N:]
    assert np.linalg.norm(S @ x + 1e-2 * x - g) <= 1e-8 * np.linalg.norm(g)


@pytest.mark.parametrize("pol,proposed", [(0.0, 0.3), (0.97, 0.9), (0.999, 0.97)])
def test_runs_of_a_learned_chain(pol, proposed):
    a, b, W, psi = model(pol, 0.5, 0.01, 64, seed=13)
    hid = 32
    p = np.concatenate([np.zeros(2 * N * hid + hid), np.full(N, np.log((1 + proposed) / (1 - proposed)))]).astype(np.float32)
    mc = R.LearnedMonteCarloLoop(R.MADE(N, hid, params=p), 512 * 8, 10, 512, True, seed=3)
    S = R.get_S_matrix_centred(psi, mc)
    words, _, _ = mc.last_samples()
    assert mc.num_runs < 0.95 * len(words)   # some samples repeat
    check(S, reference(b, W, spins_of(words), np.ones(len(words)), len(words)))

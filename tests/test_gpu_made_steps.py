"""The training step of the autoregressive proposal at the edges of its tiles
(16 samples a wavefront, 64 x 64 gradient blocks, padded inputs 64 / 128,
hidden 64 ... 512, ragged batches and splits) against oracle/made.py in FP64.

Tolerances: every value is an FP32 sum of at most 128 + 512 + 128 products,
2^-24 each in the worst case, 4e-5 of the absolute sum; gradients in 2-norm to
1e-4 (losses are FP64 sums of values of that error, 1e-5)."""
import numpy as np
import pytest

from helpers import rel_err
from oracle import made as MD

import rbmongpu_amd as R

pytestmark = pytest.mark.gpu


def setup(N, H, n):
    r = np.random.default_rng(N + H + n)
    M1, M2 = MD.masks(N, H)
    p = MD.pack(0.4 * r.normal(size=(H, N)) * M1, 0.4 * r.normal(size=H), 0.4 * r.normal(size=(N, H)) * M2,
                0.4 * r.normal(size=N)).astype(np.float32)
    X = (r.random((n, N)) < 0.5).astype(np.uint64)
    return p, MD.words(X), X.astype(np.float64)


@pytest.mark.parametrize("N,H,n", [(1, 1, 1), (2, 64, 15), (63, 65, 17), (64, 128, 64), (65, 192, 65), (128, 256, 4097),
                                   (100, 320, 130), (106, 384, 16), (91, 448, 1000), (80, 512, 129), (64, 512, 70000)])
def test_gradient_shapes(N, H, n):
    print(f"[made step] N={N} H={H} n={n}", flush=True)
    p, words, X = setup(N, H, n)
    # bits past N are not inputs
    if N < 64:
        words = words | np.array([np.uint64(1) << np.uint64(63), np.uint64(5)], dtype=np.uint64)
    loss, g = R.MADE(N, H, params=p).loss_and_gradient(words)
    q = p.astype(np.float64)
    ref = MD.loss(q, X, N, H)
    assert abs(loss - ref) <= 1e-5 * abs(ref)
    # the derivative of the ReLU is undetermined where FP32 cannot tell an
    # activation's sign: the W1 row and b1 of such a hidden unit are left out
    W1, b1, _, _ = MD.unpack(q, N, H)
    firm = np.abs(X @ W1.T + b1).min(axis=0) > 1e-6
    assert firm.sum() >= 0.9 * H
    sel = MD.pack(np.repeat(firm[:, None], N, 1), firm, np.ones((N, H)), np.ones(N)) > 0
    assert rel_err(g[sel], MD.grad(q, X, N, H)[sel]) <= 1e-4


@pytest.mark.parametrize("n,batch", [(1000, 100), (333, 400), (5, 1)])
def test_minibatch_rows_are_the_philox_draw(n, batch):
    N, H, seed = 70, 96, 0x1234567890
    p, words, X = setup(N, H, n)
    md = R.MADE(N, H, params=p)
    losses = md.train(words, 2, batch=batch, lr=0.0, seed=seed)
    for t in range(2):
        u = MD.philox_np(t, np.arange(batch), 0, 4, seed & 0xFFFFFFFF, seed >> 32)[0].astype(np.float64)
        rows = np.minimum(((u + 0.5) / 2.0 ** 32 * n).astype(np.int64), n - 1)
        ref = MD.loss(p.astype(np.float64), X[rows], N, H)
        assert abs(losses[t] - ref) <= 1e-5 * abs(ref)

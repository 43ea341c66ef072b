"""Calls whose copies end at the edges of the staged copies' kernel (16-byte
words, 256 of them a workgroup, 1024 workgroups) and beyond the staged size:
the same configurations in one call and in pieces give the same bytes."""
import numpy as np
import pytest

import rbmongpu_amd as R
from rbmongpu_amd import hamiltonians as HAM

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 256, 257, 1024, 1025, 262143, 262144, 262145, 300001])
def test_pieces_agree(n):
    print(f"[copies] n={n}", flush=True)
    N, M = 70, 9
    r = np.random.default_rng(n)
    W = 0.1 * (r.normal(size=(N, M)) + 1j * r.normal(size=(N, M)))
    b = 0.1 * (r.normal(size=M) + 1j * r.normal(size=M))
    psi = R.Psi(np.zeros(N), np.zeros(N), b, W, 1.0, False, True, precision=32)
    words = r.integers(0, 2 ** 63, size=(n, 2), dtype=np.uint64)
    words[:, 1] &= np.uint64(63)
    whole = R.log_psi_batch(psi, words)
    cut = max(1, min(n - 1, 130)) if n > 1 else 1
    parts = [R.log_psi_batch(psi, words[:cut])] + ([R.log_psi_batch(psi, words[cut:])] if n > cut else [])
    assert np.array_equal(whole, np.concatenate(parts))
    op = R.Operator(*HAM.tfim_1d(N), True)
    k = min(n, 300)
    assert np.array_equal(R.local_energy_batch(psi, op, words[-k:]), R.local_energy_batch(psi, op, words)[-k:])

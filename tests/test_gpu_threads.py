"""Calls from several host threads, each with its own handles: the compute
calls of a device run one at a time, so every thread gets the results that it
gets alone, bit for bit."""
import threading

import numpy as np
import pytest

import rbmongpu_amd as R
from rbmongpu_amd import hamiltonians as HAM

pytestmark = pytest.mark.gpu


def test_threads_with_their_own_handles():
    def work(k, out):
        N, M = 6 + k, 10 + 3 * k
        r = np.random.default_rng(k)
        W = 0.1 * (r.normal(size=(N, M)) + 1j * r.normal(size=(N, M)))
        psi = R.Psi(np.zeros(N), np.zeros(N), np.zeros(M, complex), W, 1.0, False, True, precision=64 if k % 2 else 32)
        op, ex = R.Operator(*HAM.tfim_1d(N), True), R.ExactSummation(N, True)
        ev = R.ExpectationValue(True)
        for _ in range(20):
            p = psi.params
            psi.params = p
            g, E = ev.gradient(psi, op, ex)
        out[k] = (g, E, psi.vector)

    alone, together = {}, {}
    for k in range(4):
        work(k, alone)
    threads = [threading.Thread(target=work, args=(k, together)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=60)
    for k in range(4):
        for a, b in zip(alone[k], together[k]):
            assert np.array_equal(a, b)

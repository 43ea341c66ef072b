"""PsiDeep gradients on the exact sum at the edges of the row sums (256 columns a
workgroup, 64 samples and 8 rows a step) and of the 16-lane rows, against the
FP64 oracle.  Tolerances as for the other PsiDeep gradients: 1e-10 for
complex128 kernels, 1e-5 for complex64."""
import numpy as np
import pytest

from helpers import O, deep_layers, rel_err

import rbmongpu_amd as R
from rbmongpu_amd import hamiltonians as HAM

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ti", [False, True])
@pytest.mark.parametrize("precision,tol", [(64, 1e-10), (32, 1e-5)])
@pytest.mark.parametrize("N,M,C,K", [(3, [3], [2], 12), (5, [17], [5], 119), (6, [16, 23], [2, 7], 255),
                                     (7, [12, 14], [4, 12], 256), (4, [16, 19], [2, 9], 257), (9, [32, 35], [3, 9], 513)])
def test_gradient_rows(N, M, C, K, precision, tol, ti):
    print(f"[deep rows] N={N} M={M} C={C} precision={precision} ti={ti}", flush=True)
    biases, conns, weights, final = deep_layers(N, M, C, seed=K, scale=0.2)
    psi = R.PsiDeep(np.zeros(N), np.zeros(N), list(biases), [np.asarray(c, np.uint32) for c in conns], list(weights),
                    np.asarray(final, complex), 1.0, False, True, precision=precision, ref_compat_final=False)
    psi.translational_invariance = ti
    assert psi.num_params - 2 * N == K
    ref = O.Deep(N, biases, conns, weights, final, translational_invariance=ti, ref_compat_final=False)
    tab = HAM.tfim_1d(N)
    g, E = R.ExpectationValue(True).gradient(psi, R.Operator(*tab, True), R.ExactSummation(N, True))
    gr, Er = O.gradient(ref, O.Operator(*tab), O.Exact(N), mode=0)
    assert abs(E - Er) <= tol * abs(Er)
    assert rel_err(g, gr) <= tol

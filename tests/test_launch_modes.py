"""Launches of the scalar sums and the coefficients refuse modes and missing
operands that their kernels have no branch for, on the host: no GPU is needed,
and none is touched (an accepted launch would report the missing device)."""
import ctypes as C
import os

import pytest

import rbmongpu_amd as R

INVALID_VALUE = 1   # hipErrorInvalidValue


class CoefArgs(C.Structure):   # rbm_kernels.hpp
    _fields_ = [("n", C.c_int64), ("mode", C.c_int), ("exact", C.c_int), ("mult", C.c_void_p), ("is_unitary", C.c_int),
                ("num_configs", C.c_double), ("log_prefactor", C.c_double), ("lp", C.c_void_p), ("el", C.c_void_p),
                ("lp2", C.c_void_p), ("el2", C.c_void_p), ("alpha", C.c_double * 2), ("e_mean", C.c_double * 2),
                ("coef", C.c_void_p), ("sums", C.c_void_p), ("n_sums", C.c_int), ("n_steps", C.c_double)]


LIB = C.CDLL(os.path.join(os.path.dirname(R.__file__), "librbmhip.so"))


def coef(**kw):
    return LIB["_ZN6rbmhip11launch_coefERKNS_8CoefArgsEP12ihipStream_t"](C.byref(CoefArgs(n=1, n_steps=1.0, **kw)), None)


def sums(**kw):
    return LIB["_ZN6rbmhip18launch_scalar_sumsERKNS_8CoefArgsEiPdP12ihipStream_t"](C.byref(CoefArgs(n=1, **kw)), 1, None, None)


@pytest.mark.parametrize("mode", [-1, 0, 1, 6, 7, 8, 9])
def test_coefficients_of_other_modes(mode):
    assert coef(mode=mode, coef=16, sums=16, n_sums=1, lp2=16) == INVALID_VALUE


@pytest.mark.parametrize("kw", [dict(mode=4), dict(mode=5), dict(mode=2, sums=16, n_sums=1),
                                dict(mode=2, coef=16), dict(mode=2, coef=16, sums=16, n_sums=0),
                                dict(mode=2, coef=16, sums=16, n_sums=1025), dict(mode=3, coef=16, sums=16, n_sums=1)])
def test_coefficients_without_their_operands(kw):
    assert coef(**kw) == INVALID_VALUE


@pytest.mark.parametrize("kw", [dict(mode=m, lp2=16, el2=16) for m in (-1, 2, 3, 4, 5, 9)] +
                         [dict(mode=1), dict(mode=8), dict(mode=7, el2=16), dict(mode=7, lp2=16)])
def test_scalar_sums_without_a_branch(kw):
    assert sums(**kw) == INVALID_VALUE

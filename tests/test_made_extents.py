"""The training step's check of its launches against its buffers, without a GPU:
the plan passes at every shape that is accepted, and each buffer one element
short is reported."""
import ctypes as C
import os

import pytest

import rbmongpu_amd as R

SIZES = ["spins", "params", "packed", "h", "da", "dl", "xbits", "bias", "loss", "wgrad"]


class Plan(C.Structure):   # capi.cpp, MadeStepPlan
    _fields_ = [(k, C.c_int) for k in ("N", "H", "Np", "Hp", "B", "Bp", "tiles", "splits")] + \
               [(k, C.c_int64) for k in ("n", "off_b1", "off_W2", "off_b2", "padded", *SIZES)]


LIB = C.CDLL(os.path.join(os.path.dirname(R.__file__), "librbmhip.so"))
make = LIB["_ZN6rbmhip9made_planEiiliPNS_12MadeStepPlanE"]
make.argtypes = [C.c_int, C.c_int, C.c_int64, C.c_int, C.POINTER(Plan)]
make.restype = None
fault = LIB["_ZN6rbmhip17made_extent_faultERKNS_12MadeStepPlanE"]
fault.argtypes, fault.restype = [C.POINTER(Plan)], C.c_char_p


def plan(N, H, n, batch):
    p = Plan()
    make(N, H, n, batch, C.byref(p))
    assert (p.N, p.H, p.n, p.B) == (N, H, n, batch) and p.Np % 64 == 0 and p.tiles * 16 == p.Bp
    return p


@pytest.mark.parametrize("N,H,n,batch", [(1, 1, 1, 1), (64, 64, 64, 64), (65, 65, 65, 65), (100, 256, 1_007_616, 16384),
                                         (80, 512, 5, 400), (128, 256, 1 << 24, 1 << 24), (64, 512, 70000, 1 << 20)])
def test_one_element_short(N, H, n, batch):
    assert fault(C.byref(plan(N, H, n, batch))) is None
    for k in SIZES:
        p = plan(N, H, n, batch)
        # (weight partials are read and written up to their last weight, the biases behind it are not there)
        setattr(p, k, p.off_W2 + p.Np * p.Hp + (p.splits - 1) * p.padded - 1 if k == "wgrad" else getattr(p, k) - 1)
        assert fault(C.byref(p)) is not None, k


def test_offsets_that_overlap():
    for k in ("off_W2", "off_b2"):
        p = plan(100, 256, 1000, 1000)
        setattr(p, k, getattr(p, k) - 1)
        assert fault(C.byref(p)) is not None, k

"""The square root of the GPU pair force (ctc_amd/csrc/udx_dev.h sqrt_rn: x
times an estimate of 1 / sqrt(x), corrected once by its residual) in the
formula's own arithmetic, over every float of the range the force evaluates it
on: r = sqrt(r2) with r2 in [1e-6, 1), and the w_R roots of 1 - r in
[2^-24, 1].  From the float nearest to 1 / sqrt(x) the root is correctly rounded
everywhere.  From an estimate one float away a few dozen roots of the 2e8 are
not, so the formula alone does not settle it: the hardware's own estimates are
checked, every float of the range, by the device self-check
(test_gpu_arith.py)."""
import ctypes as C

import numpy as np
import pytest

import oracle as O

LO = float(np.ldexp(np.float32(1), -24))


def _verify(lo, hi, ulp, corrected=1):
    f = O.lib().orc_verify_sqrt_rn
    f.restype = C.c_long
    f.argtypes = [C.c_float, C.c_float, C.c_int, C.c_int, C.c_int]
    return f(lo, hi, 8, ulp, corrected)


def test_sqrt_from_the_nearest_estimate():
    assert _verify(LO, 1.0, 0) == 0


@pytest.mark.parametrize("ulp", [-1, 1])
def test_sqrt_from_a_neighbouring_estimate(ulp):
    """why the device check is needed: not zero, and no more than 2 in 1e7"""
    bad = _verify(LO, 1.0, ulp)
    assert 0 < bad <= 40


def test_verifier_catches_uncorrected_roots():
    """control: the uncorrected product is off for a large share of the range"""
    lo, hi = np.float32(0.25), np.float32(0.5)
    nfloat = int(hi.view(np.uint32)) - int(lo.view(np.uint32)) + 1
    assert _verify(lo, hi, 0, corrected=0) > nfloat // 20

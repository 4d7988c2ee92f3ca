"""The FP64 pair kernel's own 1/sqrt, 1/x and exp against 64-bit-mantissa
results, in units of the last place of the exact result."""
import ctypes as C
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "libpairfunctions.so")


def _apply(which, x):
    lib = C.CDLL(LIB)
    dp = C.POINTER(C.c_double)
    lib.pair_function.argtypes = [C.c_int, C.c_int, dp, dp]
    y = np.zeros_like(x)
    assert lib.pair_function(which, len(x), x.ctypes.data_as(dp), y.ctypes.data_as(dp)) == 0
    return y


# the last step of 1/sqrt and 1/x rounds once (half a unit) after terms of a
# thousandth of one; the series of exp rounds in its last additions too
@pytest.mark.parametrize("which,bound", [(0, 0.501), (1, 0.501), (2, 0.9)])
def test_error_in_units_of_the_last_place(which, bound):
    rng = np.random.default_rng(which)
    x = np.exp2(rng.uniform(-8, 8, 1 << 20))
    x[:4] = 2.0 ** -8, 2.0 ** 8, 1.0, 3.0
    if which == 2:
        x = -x
        x[4:6] = 0.0, -700.0
    y = _apply(which, x)
    with np.errstate(all="ignore"):
        exact = (1 / np.sqrt(x.astype(np.longdouble)), 1 / x.astype(np.longdouble), np.exp(x.astype(np.longdouble)))[which]
    err = np.abs((y.astype(np.longdouble) - exact) / np.spacing(exact.astype(np.float64)))
    print(f"function {which}: largest error {float(err.max()):.4f} units of the last place", flush=True)
    assert np.finfo(np.longdouble).nmant >= 63 and float(err.max()) <= bound


def test_limits():
    assert _apply(0, np.array([0.0]))[0] == np.inf  # coincident atoms
    assert np.array_equal(_apply(2, np.array([-746.0, -14400.0])), [0.0, 0.0])

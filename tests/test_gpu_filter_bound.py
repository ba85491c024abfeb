"""GPU: the error bound behind the filtered simulation kernel.  Its tests of
times are right because a single-precision normal pair is within 7e-6 (the
kernels' kPairErr) of the 64-bit one, for every block whose first word the
filter accepts.  The pair is a radius, which depends on the block's first two
words, times the sine and cosine of an angle, which depends on the other two:
both are evaluated over all 2^32 values of the leading word."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_pair_error_over_all_words(procell_lib):
    f = procell_lib.lib().procell_debug_pair_bounds
    f.argtypes = [ctypes.c_int32, ctypes.POINTER(ctypes.c_double)]
    out = np.zeros(4)
    assert f(0, out.ctypes.data_as(ctypes.POINTER(ctypes.c_double))) == procell_lib.OK
    radius, radius_low, sincos, pair = out
    print("radius", radius, "radius where u <= 1/2", radius_low, "sine, cosine", sincos, "pair", pair, flush=True)
    # single precision cannot be better than these: the sweep did run
    assert radius > 1e-6 and radius_low > 1e-6 and sincos > 3e-8
    assert radius <= 5.5e-6 and radius_low <= 3.7e-6 and sincos <= 2.8e-7
    assert pair <= 7.0e-6

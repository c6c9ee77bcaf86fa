"""The quick phase of the correctly rounded acos and sincos
(gpluto_dev_amd/csrc/crmath.hpp) against its double-double forms, on the host:
the same results, the quick sums within half of the error bound that the
rounding test takes (derived from the rounding errors of each term; half is the
margin asked for here), and both branches of the test taken."""
import ctypes
import math

import pytest

from test_crmath import ACOS_NEAR_ONE, ACOS_UNIFORM, SINCOS_CUBIC, SINCOS_UNIFORM, THREADS, lib  # noqa: F401


@pytest.mark.parametrize("mode,n,lo,hi", [
    (ACOS_UNIFORM, 4 * 10 ** 6, -1.0, 1.0),
    (ACOS_UNIFORM, 10 ** 6, 0.5 - 2.0 ** -30, 0.5 + 2.0 ** -30),      # the two forms meet
    (ACOS_UNIFORM, 10 ** 6, -0.5 - 2.0 ** -30, -0.5 + 2.0 ** -30),
    (ACOS_UNIFORM, 10 ** 6, -(2.0 ** -40), 2.0 ** -40),               # cos theta = 0
    (ACOS_NEAR_ONE, 4 * 10 ** 6, 0.0, 0.0),
    (SINCOS_CUBIC, 4 * 10 ** 6, 0.0, 0.0),
    (SINCOS_UNIFORM, 4 * 10 ** 6, 0.0, 2.19),
    (SINCOS_UNIFORM, 10 ** 6, 0.0, 2.0 ** -7),                        # the table's first entry
    (SINCOS_UNIFORM, 10 ** 6, 0.0, 1e-290),
    (SINCOS_UNIFORM, 10 ** 6, math.pi / 2 - 2.0 ** -30, math.pi / 2 + 2.0 ** -30),
])
def test_quick_phase_gives_the_double_double_results(lib, mode, n, lo, hi):  # noqa: F811
    lib.crm_quick.restype = ctypes.c_longlong
    lib.crm_quick.argtypes = [ctypes.c_int, ctypes.c_longlong, ctypes.c_ulonglong, ctypes.c_double,
                              ctypes.c_double, ctypes.c_int, ctypes.POINTER(ctypes.c_double)]
    out = (ctypes.c_double * 2)()
    assert lib.crm_quick(mode, n, 5, lo, hi, THREADS, out) == 0
    assert out[0] < 0.5, out[0]
    if mode in (ACOS_UNIFORM, ACOS_NEAR_ONE) and hi - lo in (2.0, 0.0):
        assert 0 < out[1] < 1e-3 * n, out[1]

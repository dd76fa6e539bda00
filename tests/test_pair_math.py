"""The pair kernels' arithmetic (physica_amd/csrc/device_math.hpp) against the
same expressions with the compiler's square root and division, for every float
squared distance from 2^-90 h^2 to just past the support, and for 0. The
support radii include the ends of both ranges whose quotients skip the
compiler's scaling, and radii beyond them."""
import ctypes

import numpy as np
import pytest

from physica_amd import build

pytestmark = pytest.mark.gpu


def _bits(x) -> int:
    return int(np.array([x], dtype=np.float32).view(np.uint32)[0])


# the ends of the ranges whose quotients skip the compiler's scaling (PBF's
# kernels, the cubic kernel's gradient), and the radii just outside them
ENDS = [2.0**-11, 2.0**8, 2.0**-20, 2.0**16]
OUTSIDE = [float(np.nextafter(np.float32(end), np.float32(0.0 if end < 1.0 else np.inf))) for end in ENDS]


@pytest.mark.parametrize("h", [0.02, 0.04, 0.1, 1.0 / 30.0, 1.0e-4, 700.0, 1.3e-6, 6.1e4, 1.0e6] + ENDS + OUTSIDE)
def test_pair_functions_equal_their_expressions(gpu_device, h):
    lib = ctypes.CDLL(str(build.PAIR_MATH_CHECK))
    lib.phx_test_pair_math.argtypes = [ctypes.c_float, ctypes.c_uint32, ctypes.c_uint32,
                                       ctypes.POINTER(ctypes.c_ulonglong)]
    h = float(np.float32(h))
    wrong = (ctypes.c_ulonglong * 4)()
    for first, count in ((_bits(2.0**-90 * h * h), _bits(1.01 * h * h) - _bits(2.0**-90 * h * h)), (0, 1)):
        assert lib.phx_test_pair_math(h, first, count, wrong) == 0
        assert list(wrong) == [0, 0, 0, 0], (h, first)


@pytest.mark.parametrize("rest", [1000.0, 1.0, 0.37, 2.0**-60, 2.0**60, 1.0e-30, 1.0e25, 0.0, float("inf")])
def test_mass_over_rest_density_equals_the_division(gpu_device, rest):
    """For every non-negative float mass: 0, subnormal, of any size, infinite."""
    lib = ctypes.CDLL(str(build.PAIR_MATH_CHECK))
    lib.phx_test_over_rest.argtypes = [ctypes.c_float, ctypes.c_uint32, ctypes.c_uint32,
                                       ctypes.POINTER(ctypes.c_ulonglong)]
    wrong = ctypes.c_ulonglong()
    assert lib.phx_test_over_rest(rest, 0, _bits(np.inf) + 1, ctypes.byref(wrong)) == 0
    assert wrong.value == 0

"""The short divisions and square roots of st_math.h on the GPU against the
correctly rounded ones (numpy's on the host)."""
import ctypes
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DIV_BY, DIV_SQRT = 0, 1


@pytest.fixture(scope="module")
def lib(device):
    return ctypes.CDLL(os.path.join(os.path.dirname(__file__), "native", "_build", "libmath_check.so"))


def _div(lib, kind, x, n):
    x, n = (np.ascontiguousarray(v, np.float64) for v in (x, n))
    q = np.empty_like(x)
    assert lib.mc_div(kind, *(v.ctypes.data_as(ctypes.c_void_p) for v in (x, n, q)), x.size) == 0
    return q


def _same(a, b):
    """Equal, signs of zeros and places of NaN included."""
    return np.array_equal(a, b, equal_nan=True) and np.array_equal(np.signbit(a), np.signbit(b))


SPECIAL = np.array([0.0, -0.0, np.inf, -np.inf, 1.0, -1.0, 3e38, 1e-45])


@pytest.mark.parametrize("n", [1.0, 3.0, 65536.0, 147455.0])
def test_division_of_special_values(lib, n):
    assert _same(_div(lib, DIV_BY, SPECIAL, np.full_like(SPECIAL, n)), SPECIAL / n)


@pytest.mark.parametrize("a", [4.0, 1e-280, 1e280, 1e-300, 0.0, np.inf, 2.0])
def test_division_of_special_values_by_a_root(lib, a):
    with np.errstate(all="ignore"):
        want = SPECIAL / np.sqrt(a)
    assert _same(_div(lib, DIV_SQRT, SPECIAL, np.full_like(SPECIAL, a)), want)

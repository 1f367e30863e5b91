"""The short divisions and square roots of st_math.h on the GPU against the
correctly rounded ones (numpy's on the host), and the Gaussian fit's sums
and 3 x 3 solve against their plain forms."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DIV_BY, DIV_SQRT = 0, 1


@pytest.fixture(scope="module")
def lib(device):
    native = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native")
    so = os.path.join(native, "_build", "libmath_check.so")
    if not os.path.exists(so):  # build() makes it
        subprocess.run(["make", "-s", "-C", native], check=True)
    return ctypes.CDLL(so)


def _div(lib, kind, x, n):
    x, n = (np.ascontiguousarray(v, np.float64) for v in (x, n))
    q = np.empty_like(x)
    assert lib.mc_div(kind, *(v.ctypes.data_as(ctypes.c_void_p) for v in (x, n, q)), x.size) == 0
    return q


def _ncc(lib, v):
    v = np.ascontiguousarray(v, np.float64)
    out = np.empty(len(v))
    assert lib.mc_ncc(*(x.ctypes.data_as(ctypes.c_void_p) for x in (v, out)), len(v)) == 0
    return out


def _ncc_plain(v):
    c, mean, var, s1, s2, n = v.T
    m = s1 / n
    return (c - mean * m) / np.sqrt(var * (s2 / (n - 1) - m * m))


def test_correlation_of_special_values(lib):
    """Sums, means and variances that are zero, infinite, NaN or near the ends of
    the range: the plain quotients' values, infinities among them."""
    x = [0.0, 3.0, -2.5, 1e-140, 1e150, 1e300, np.inf, -np.inf, np.nan]
    v = np.stack(np.meshgrid(x, x, x, x, x, [65536.0, 97 * 31.0], indexing="ij"), -1).reshape(-1, 6)
    with np.errstate(all="ignore"):
        want = _ncc_plain(v)
    got = _ncc(lib, v)
    assert np.array_equal(got, want, equal_nan=True), v[~((got == want) | (np.isnan(got) & np.isnan(want)))][:5]
    assert np.isinf(want).any() and np.isnan(want).any()


def test_correlation_is_the_plain_one(lib):
    rng = np.random.default_rng(7)
    n = np.floor(rng.uniform(3, 200, 1 << 20)) * np.floor(rng.uniform(3, 200, 1 << 20))
    mean = rng.uniform(0, 3, n.size) * 10.0 ** rng.uniform(-6, 6, n.size)
    v = np.stack([mean * mean * rng.uniform(0, 2, n.size), mean, mean**2 * rng.uniform(0.01, 1, n.size), n * mean,
                  n * mean**2 * rng.uniform(1.01, 2, n.size), n], 1)
    assert np.count_nonzero(_ncc(lib, v) != _ncc_plain(v)) == 0


def _hard_quotients(rng, n):
    """(x, g), g of 53 bits, with x / g beside the midpoint of two doubles by
    1 / (2 g) of their distance or 3 times that: x 2^54 = g m - c for an odd m
    of 54 bits, the midpoint in units of 2^-54, and c = +-1, +-3."""
    xs, gs = [], []
    while len(xs) < n:
        g, c = int(rng.integers(2**52, 2**53)) | 1, int(rng.choice([-3, -1, 1, 3]))
        m = c * pow(g, -1, 2**54) % 2**54
        if m >= 2**53:
            xs.append((g * m - c) >> 54)
            gs.append(g)
    return np.array(xs, np.float64), np.array(gs, np.float64)


def _hard_roots(rng, n):
    """Doubles a whose root lies beside the midpoint of two doubles by c / (2 m):
    a 2^55 = m^2 - c for an odd m of 54 bits and small c = 1 (mod 8), m from the
    roots of c modulo powers of two."""
    out = []
    while len(out) < n:
        c, m = 8 * int(rng.integers(-8, 9)) + 1, 2 * int(rng.integers(0, 4)) + 1
        for k in range(3, 56):  # m^2 = c (mod 2^k) -> (mod 2^(k + 1))
            if (m * m - c) >> k & 1:
                m += 1 << (k - 1)
        m = m % 2**55 if rng.integers(2) else -m % 2**55
        if 2**53 <= m < 2**54:
            assert (m * m - c) % 2**55 == 0
            out.append((m * m - c) >> 55)
    return np.array(out, np.float64) * 2.0**55


def test_quotient_by_a_root_is_rounded(lib):
    """The hardest quotients: the root of g^2 is g, its reciprocal has to be the
    rounded one for the last residual to fall on the right side.  The hardest
    roots, of 200 x each."""
    rng = np.random.default_rng(1)
    a = np.repeat(_hard_roots(rng, 2000), 200)
    x = rng.standard_normal(a.size)
    assert np.count_nonzero(_div(lib, DIV_SQRT, x, a) != x / np.sqrt(a)) == 0
    x, g = _hard_quotients(rng, 20000)
    a = g * g
    assert (np.sqrt(a) == g).all()
    assert np.count_nonzero(_div(lib, DIV_SQRT, x, a) != x / g) == 0
    x, a = rng.standard_normal(1 << 20), np.exp(rng.uniform(-600, 600, 1 << 20))
    assert np.count_nonzero(_div(lib, DIV_SQRT, x, a) != x / np.sqrt(a)) == 0


def test_division_is_rounded(lib):
    """Whole divisors up to the lags of a window (2048^2), and every mantissa."""
    rng = np.random.default_rng(2)
    x, n = rng.standard_normal(1 << 20) * 1e6, np.floor(np.exp(rng.uniform(0, np.log(2**22), 1 << 20)))
    assert np.count_nonzero(_div(lib, DIV_BY, x, n) != x / n) == 0
    n = np.arange(1.0, 2**16)
    x = np.nextafter(n * rng.integers(1, 2**30, n.size), rng.choice([-np.inf, np.inf], n.size))
    assert np.count_nonzero(_div(lib, DIV_BY, x, n) != x / n) == 0


def _lm_coef(lib, y, a):
    y, a = (np.ascontiguousarray(v, np.float32) for v in (y, a))
    out = np.empty((2, len(a), 13), np.float32)
    assert lib.mc_lm_coef(*(v.ctypes.data_as(ctypes.c_void_p) for v in (y, a, out)), len(a)) == 0
    return out


def test_fit_sums_equal_their_plain_form(lib):
    """Amplitude, centre and width over and far beyond what a fit meets; the
    reciprocals give the very quotients."""
    rng = np.random.default_rng(3)
    n = 1 << 18
    a = np.stack([rng.uniform(-2, 3, n), rng.uniform(-8, 26, n), np.exp(rng.uniform(-3, 4, n)) * rng.choice([-1, 1], n)], 1)
    a[n // 2:] *= 10.0 ** rng.uniform(-6, 6, (n - n // 2, 3))
    short, plain = _lm_coef(lib, rng.uniform(0, 1, (n, 18)), a)
    assert np.array_equal(short, plain, equal_nan=True)


def test_fit_sums_of_special_parameters(lib):
    """Widths and centres that are zero, infinite, NaN, or whose squares and
    cubes leave the floats' range: what the plain quotients give."""
    v = np.array([0.0, 1.0, -3.0, 8.5, 1e-22, 1e-15, 1e-13, 1e13, 1e19, 3e19, 3.4e38, np.inf, -np.inf, np.nan])
    a = np.stack(np.meshgrid([1.0, 0.0, 1e30, np.inf], v, v, indexing="ij"), -1).reshape(-1, 3)
    short, plain = _lm_coef(lib, np.random.default_rng(4).uniform(0, 1, (len(a), 18)), a)
    bad = ~((short == plain) | (np.isnan(short) & np.isnan(plain))).all(1)
    assert not bad.any(), a[bad]


def test_every_square_root_of_the_short_form(lib):
    """All floats from 2^-96 to the largest, against the rounded FP64 root."""
    bad = ctypes.c_ulonglong(1)
    assert lib.mc_sqrt(0x0F800000, 0x7F800000, ctypes.byref(bad)) == 0
    assert bad.value == 0


def test_range_test_of_the_short_square_root(lib):
    """One value of a wave outside [2^-96, FLT_MAX], in either register and any
    lane, sends the whole wave to the full form; values at the ends do not."""
    inside = np.array([2.0**-96, 1.0, np.finfo(np.float32).max], np.float32)
    outside = np.array([0.0, 1e-45, np.nextafter(np.float32(2.0**-96), np.float32(0)), np.inf, np.nan], np.float32)
    x = np.random.default_rng(5).choice(inside, (2 * 64 * len(outside) + 2, 64, 2))
    for k, v in enumerate(outside):
        for lane in range(64):
            for reg in range(2):
                x[(k * 64 + lane) * 2 + reg, lane, reg] = v
    r = np.empty(x.shape[:2], np.int32)
    assert lib.mc_needs_full(*(v.ctypes.data_as(ctypes.c_void_p) for v in (x, r)), len(x)) == 0
    assert (r[:-2] != 0).all() and (r[-2:] == 0).all()


def test_solve3_equals_its_plain_form(lib):
    """Random systems, symmetric ones as the fit's, ties of the pivots, singular
    ones, infinities and NaN."""
    rng = np.random.default_rng(6)
    n = 1 << 16
    a = rng.standard_normal((4, n, 12)) * 10.0 ** rng.uniform(-4, 4, (4, n, 12))
    a[1, :, 3], a[1, :, 6], a[1, :, 7] = a[1, :, 1], a[1, :, 2], a[1, :, 5]
    a[2] = rng.integers(-2, 3, (n, 12))
    a[3] = rng.choice([0.0, 1.0, -1.0, 1e30, 1e-40, np.inf, np.nan], (n, 12), p=[.2, .3, .2, .1, .1, .05, .05])
    a = np.ascontiguousarray(a.reshape(-1, 12), np.float32)
    out = np.empty((2, len(a), 4), np.float32)
    assert lib.mc_solve3(*(v.ctypes.data_as(ctypes.c_void_p) for v in (a, out)), len(a)) == 0
    assert np.array_equal(out[0], out[1], equal_nan=True)
    assert 0.2 < out[0, 2 * n:3 * n, 0].mean() < 0.95

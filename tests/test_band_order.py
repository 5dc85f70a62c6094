"""The number of points of the radial bands (band_order of hbem_radial.hip),
checked on the CPU with scipy's Bessel functions: the polynomial interpolant
at that many Chebyshev points reproduces the radial functions of the operators
on the band for every kappa up to the tier's edge.

Tolerance: the bound band_order meets (1e-16, or the separated-pair rules'
5e-14, relative to the largest value on the band) plus rounding: scipy's
functions are good to a few ulp and the Lebesgue constant of 200 Chebyshev
points is below 4.5, so 1e-14.  Points and arguments are held in extended
precision (a phase kappa r of 8000 rounded to 64 bits is off by 1e-12 already);
what scipy's functions do not see of an argument enters by their derivatives.
"""
import ctypes
import math
import os

import numpy as np
import pytest
import scipy.special as sp

LIB = os.path.join(os.path.dirname(__file__), "..", "helmholtzbem_amd", "libhbem.so")
EDGES = (0.625, 1.25, 2.5, 5.0, 10.0, 20.0)     # kappa times the largest panel diameter
RADIUS, WIDTH, STEP = 10.0, 4.0, 2.0            # near radius, interval width, band step in panel diameters


@pytest.fixture(scope="module")
def order():
    f = ctypes.CDLL(LIB)._ZN4hbem10band_orderEddddb
    f.restype = ctypes.c_int
    f.argtypes = [ctypes.c_double] * 4 + [ctypes.c_bool]
    return f


PI = 4 * np.arctan(np.longdouble(1))


def points(p):
    return np.cos((2 * np.arange(p, dtype=np.longdouble) + 1) * PI / (2 * p))


def hankel(x):
    """H0, H1 of the first kind at extended-precision arguments."""
    x0 = x.astype(float)
    d = x - x0
    h0, h1 = (sp.hankel1(n, x0).astype(np.clongdouble) for n in (0, 1))
    return h0 - d * h1, h1 + d * (h0 - h1 / x0)


def interpolate(p, values, s):
    """The interpolant through the p Chebyshev points at s (barycentric form)."""
    sj = points(p)
    w = (-1.0) ** np.arange(p) * np.sin((2 * np.arange(p, dtype=np.longdouble) + 1) * PI / (2 * p))
    d = s[:, None] - sj[None, :]
    hit = np.abs(d) < 1e-15
    d[hit] = 1.0
    c = w / d
    out = (c @ values) / c.sum(1)
    r, k = np.nonzero(hit)
    out[r] = values[k]
    return out


@pytest.mark.parametrize("edge", EDGES)
@pytest.mark.parametrize("band", [1, 2, 3, 6, 20, 200])
@pytest.mark.parametrize("tol", [1e-16, 5e-14])
def test_far_band(order, edge, band, tol):
    lo = RADIUS - WIDTH + (band - 1) * STEP
    a = 0.5 * (STEP + WIDTH)
    c = lo + a
    p = order(c, a, edge, tol, False)
    assert p > 0 and p % 4 == 0
    s = np.linspace(-1.0, 1.0, 401).astype(np.longdouble)
    for kap in (edge, 0.5 * edge):
        for f in (lambda r: hankel(kap * r)[0], lambda r: hankel(kap * r)[1] / r,
                  lambda r: hankel(kap * r)[1] * r, lambda r: hankel(kap * r)[0] * r * r):
            want = f(c + a * s)
            got = interpolate(p, f(c + a * points(p)), s)
            assert np.abs(got - want).max() <= (tol + 1e-14) * np.abs(want).max(), (edge, band, p)


def entire_parts(x):
    """J0, the entire part of Y0, J1 / x, the entire part of Y1 over x."""
    xs = np.where(x > 0, x, 1.0)
    xs = xs.astype(float)
    x = x.astype(float)
    l2 = 2.0 / math.pi * np.log(0.5 * xs)
    j0, j1 = sp.j0(x), sp.j1(xs) / xs
    c = sp.y0(xs) - l2 * sp.j0(xs)
    d = (sp.y1(xs) - l2 * sp.j1(xs) + 2.0 / (math.pi * xs)) / xs
    return j0, c, j1, d


@pytest.mark.parametrize("edge", EDGES)
def test_near_band(order, edge):
    p = order(0.0, RADIUS, edge, 1e-17, True)
    assert p > 0 and p % 4 == 0
    s = np.linspace(-0.999, 1.0, 401)
    for kap in (edge, 0.5 * edge):
        x = lambda t: kap * RADIUS * np.sqrt(0.5 * (t + 1.0))     # noqa: E731
        for got, want in zip(entire_parts(x(points(p))), entire_parts(x(s))):
            # the parts are formed from Y by subtracting logarithms of size up to ln(1 / x)
            # and, for Y1, 2 / (pi x^2)
            scale = 1.0 + 4.0 / x(s) ** 2
            assert (np.abs(interpolate(p, got, s) - want) / scale).max() <= 2e-14, (edge, p)


def test_too_wide_a_band_is_refused(order):
    assert order(9.0, 3.0, 1e4, 1e-16, False) == 0
    assert order(0.0, 10.0, 1e4, 1e-17, True) == 0

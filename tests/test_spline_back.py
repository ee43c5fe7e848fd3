"""The back substitution with reciprocals of the diagonal (csrc/tridiag.hpp)
against the one with divisions, bit for bit: ordinary values, groups of eight
rows with a value out of the reciprocals' range (zeros of either sign, tiny,
huge, infinite, not a number), every number of rows around the groups."""

import ctypes

import numpy as np
import pytest

from test_host_twin import P, _p, tw  # noqa: F401


def _pair(tw, n, d, du, dl, b):
    F = np.zeros((5, n))
    F[2], F[3], F[4] = d, du, dl
    out = np.zeros((3, n))
    tw.twin_dgtsv_back_pair.argtypes = [ctypes.c_int, P, P, P, P, P]
    tw.twin_dgtsv_back_pair.restype = None
    tw.twin_dgtsv_back_pair(n, _p(F), _p(b), _p(out[0]), _p(out[1]), _p(out[2]))
    return out


def _same(a, b):
    return np.array_equal(a.view(np.int64)[~np.isnan(a)], b.view(np.int64)[~np.isnan(b)]) and \
        np.array_equal(np.isnan(a), np.isnan(b))


@pytest.mark.parametrize("n", [3, 4, 10, 11, 18, 19, 120, 291])
def test_back_with_reciprocals(tw, n):  # noqa: F811
    rng = np.random.default_rng(n)
    for trial in range(200):
        d = rng.uniform(0.5, 4.0, n) * rng.choice([-1.0, 1.0], n) * 10.0 ** rng.uniform(-3, 6)
        du, dl = rng.normal(size=n) * np.abs(d) * 0.4, rng.normal(size=n) * np.abs(d) * 0.1
        b = rng.normal(size=n) * 10.0 ** rng.uniform(-20, 5)
        if trial % 4 == 1:
            b[rng.random(n) < 0.3] = rng.choice([0.0, -0.0, 5e-324, 1e-310, 1e-200, 1e200, 1e308])
        if trial % 4 == 2:
            du[:] = dl[:] = 0.0
            b[rng.random(n) < 0.3] = -0.0
        if trial % 8 == 3:
            d[rng.integers(n)] = rng.choice([1e-300, 1e300, 5e-324])
            b[rng.integers(n)] = rng.choice([np.inf, np.nan, 1.0])
        with np.errstate(all="ignore"):
            x_div, x_rec, _ = _pair(tw, n, d, du, dl, b)
        assert _same(x_div, x_rec), trial


def test_division_by_reciprocal(tw):  # noqa: F811
    """Quotients of random and of hard mantissas (all ones, just above one,
    products rounded to neighbours of exact quotients)."""
    rng = np.random.default_rng(7)
    n = 400000
    one = np.float64(1.0)
    d = rng.uniform(1.0, 2.0, n)
    a = rng.uniform(1.0, 2.0, n)
    d[:1000] = np.nextafter(2.0, 1.0) - rng.integers(0, 8, 1000) * 2.0 ** -52
    a[:500] = np.nextafter(one, 2.0) + rng.integers(0, 8, 500) * 2.0 ** -52
    k = slice(1000, 200000)   # a next to q d for a rounded q
    a[k] = rng.uniform(1.0, 2.0, 199000) * d[k]
    a[1000:100000] = np.nextafter(a[1000:100000], 4.0)
    a *= 2.0 ** rng.integers(-300, 300, n)
    d *= 2.0 ** rng.integers(-300, 300, n) * rng.choice([-1.0, 1.0], n)
    q = _pair(tw, n, d, np.zeros(n), np.zeros(n), a)[2]
    assert np.array_equal(q, a / d)

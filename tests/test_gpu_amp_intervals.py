"""GPU test of the knot interval of interp2D's points (found by halving, one lane
per coordinate): points on, just beside and between the knots, beyond both ends,
repeated inner knots, no inner knots, all degrees; the oracle's bits."""

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _knots(rng, inner, k):
    t = np.sort(rng.uniform(0.0, 1.0, inner))
    if inner > 4:
        t[2] = t[3]  # a repeated inner knot
    return np.concatenate([np.zeros(k + 1), t, np.ones(k + 1)])


def _points(rng, t, n):
    p = np.concatenate([t, np.nextafter(t, -1.0), np.nextafter(t, 2.0), [-0.5, 1.5],
                        rng.uniform(0.0, 1.0, n)])
    return p[rng.permutation(len(p))]


@pytest.mark.parametrize("kx,ky", [(1, 1), (2, 5), (3, 3), (4, 3), (5, 4)])
@pytest.mark.parametrize("nx,ny", [(0, 1), (1, 0), (5, 8), (33, 64)])
def test_interp2d_intervals(gpu, kx, ky, nx, ny):
    from fastemriwaveforms_amd import pyinterp
    rng = np.random.default_rng(100 * kx + nx)
    tx, ty = _knots(rng, nx, kx), _knots(rng, ny, ky)
    x, y = _points(rng, tx, 200), _points(rng, ty, 200)
    n = min(len(x), len(y))
    x, y = x[:n], y[:n]
    sets = 3
    c = rng.normal(size=(sets, (len(tx) - kx - 1) * (len(ty) - ky - 1)))
    ref = oracle.interp2d(tx, ty, c, x, y, kx, ky)
    z = np.zeros(sets * n)
    pyinterp.interp2D(z, tx, len(tx), ty, len(ty), c.flatten(), kx, ky, x, n, y, n, sets, c.shape[1])
    assert np.array_equal(z.reshape(sets, n), ref, equal_nan=True)

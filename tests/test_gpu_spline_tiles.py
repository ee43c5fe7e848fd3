"""GPU tests of the tiled spline evaluation (64 arrays x 64 points, from 2^19
values on): the reference's operations in its order, compared bit for bit."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _np_eval(t, c, x0, d):
    """The reference's evaluation (interpolatedmodesum.py:161-257): c is (4, arrays, L)."""
    L = len(t)
    j = np.searchsorted(t, x0, side="right") - 1
    j[x0 == t[-1]] = L - 2
    left, right = x0 < t[0], x0 > t[-1]
    j = np.clip(j, 0, L - 1)
    x = x0 - t[j]
    x2 = x * x
    y, c1, c2, c3 = (c[p][:, j] for p in range(4))
    if d == 0:
        v = y + c1 * x + c2 * x2 + c3 * (x * x2)
        v[:, left] = c[0][:, :1]
        v[:, right] = c[0][:, -1:]
        return v
    if d == 1:
        return c1 + 2 * c2 * x + 3 * c3 * x2
    if d == 2:
        return 2 * c2 + 6 * c3 * x
    return np.broadcast_to(6 * c3, (c.shape[1], len(x0)))


# sizes on both sides of the tile edges and of the 2^19 values where tiles start
@pytest.mark.parametrize("arrays,points,L", [(64, 8192, 5), (64, 8191, 5), (65, 8129, 40),
                                             (8200, 64, 7), (521, 1025, 150), (63, 9000, 20)])
def test_spline_eval_tiles(gpu, arrays, points, L):
    from fastemriwaveforms_amd.summation import CubicSplineInterpolant
    rng = np.random.default_rng(arrays + points)
    t = np.concatenate([[0.0], np.cumsum(rng.uniform(0.1, 1.0, L - 1))])
    y = rng.normal(size=(arrays, L))
    spl = CubicSplineInterpolant(t, y)
    c = np.stack([v.cpu().numpy() for v in (spl.y, spl.c1, spl.c2, spl.c3)])
    x = rng.uniform(t[0], t[-1], points)
    x[:L] = t   # knots, the last one included
    for d in range(4):
        got = spl(x, deriv_order=d).cpu().numpy()
        assert np.array_equal(got, _np_eval(t, c, x, d)), d
    x[rng.integers(L, points, 5)] = t[-1] + 1.0
    x[rng.integers(L, points, 5)] = t[0] - 1.0
    assert np.array_equal(spl(x).cpu().numpy(), _np_eval(t, c, x, 0))
    with pytest.raises(ValueError):
        spl(x, deriv_order=1)

"""GPU tests of the tiled spline evaluation at the edges of its rule (7 * 2^17 values,
or 2^19 from 1536 arrays on) and of its spread over the XCDs (tile counts below and
between multiples of eight, one group of arrays and several), bit for bit."""

import numpy as np
import pytest

from test_gpu_spline_tiles import _np_eval

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("arrays,points,L", [
    (64, 14335, 6), (64, 14336, 6),        # either side of 7 * 2^17
    (64, 64 * 225 + 1, 30),                # 226 tiles of one group, the last of one point
    (65, 14200, 30),                       # the second group holds one array
    (449, 2100, 12), (600, 1700, 12),      # 8 and 10 groups, odd tile counts
    (1535, 350, 9), (1536, 341, 9), (1536, 342, 9), (1600, 350, 9)])
def test_rule_edges(gpu, arrays, points, L):
    from fastemriwaveforms_amd.summation import CubicSplineInterpolant
    rng = np.random.default_rng(arrays + points)
    t = np.concatenate([[0.0], np.cumsum(rng.uniform(0.1, 1.0, L - 1))])
    spl = CubicSplineInterpolant(t, rng.normal(size=(arrays, L)))
    c = np.stack([v.cpu().numpy() for v in (spl.y, spl.c1, spl.c2, spl.c3)])
    x = rng.uniform(t[0], t[-1], points)
    x[:L] = t
    for d in (0, 2):
        assert np.array_equal(spl(x, deriv_order=d).cpu().numpy(), _np_eval(t, c, x, d)), d
    x = np.sort(x)
    x[-1] = t[-1] + 1.0
    assert np.array_equal(spl(x).cpu().numpy(), _np_eval(t, c, x, 0))

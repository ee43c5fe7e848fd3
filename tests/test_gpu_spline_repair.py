"""GPU test of the spline build's back substitution where only some of a block's
32 systems leave the reciprocals' range: those rows are written twice (quotients
by reciprocals, then by divisions), and the coefficients must come from the second
value in every column, the systems beside them keeping theirs.  Bit for bit."""

import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


def _columns(rng, nsys, length):
    """Ordinary systems with others among them: zero from some knot on, all zero
    (either sign), tiny and huge values."""
    y = rng.normal(size=(nsys, length))
    for s in range(nsys):
        cut = int(rng.integers(0, length))
        kind = s % 7
        if kind == 1:
            y[s, cut:] = 0.0
        elif kind == 2:
            y[s] = -0.0
        elif kind == 3:
            y[s, :cut] *= 1e-290
        elif kind == 4:
            y[s] *= 1e180
        elif kind == 5:
            y[s, cut:] = y[s, cut]
    return y[rng.permutation(nsys)]


@pytest.mark.parametrize("length", [4, 5, 10, 11, 12, 19, 20, 120, 290])
def test_some_columns_repaired(gpu, length):
    from fastemriwaveforms_amd._lib import lib
    from fastemriwaveforms_amd.pipeline import _stream
    dev = torch.device("cuda", 0)
    for nsys in (32, 45, 200):
        rng = np.random.default_rng(1000 * length + nsys)
        h = rng.uniform(0.2, 1.0, length - 1)
        h[rng.random(length - 1) < 0.2] *= 40.0  # uneven spacing: row interchanges
        t = np.concatenate([[0.0], np.cumsum(h)])
        y = _columns(rng, nsys, length)
        t_d, y_d = torch.from_numpy(t).to(dev), torch.from_numpy(y).to(dev)
        out = torch.full((4, nsys, length), 7.0, dtype=torch.float64, device=dev)
        scratch = torch.zeros(4 * length * nsys, dtype=torch.float64, device=dev)
        rc = lib().few_spline_build_async(y_d.data_ptr(), length, 1, t_d.data_ptr(), 0, 1,
                                          out.data_ptr(), nsys * length, length, 1, nsys, length,
                                          0, scratch.data_ptr(), _stream())
        assert rc == 0, lib().few_last_error()
        torch.cuda.synchronize()
        with np.errstate(all="ignore"):
            ref, _, info = oracle.interpolate_arrays(np.tile(t, (nsys, 1)), y)
        assert info == 0
        np.testing.assert_array_equal(out.cpu().numpy(), ref)

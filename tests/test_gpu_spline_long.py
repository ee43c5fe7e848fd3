"""GPU test of the spline build's LDS path at its largest lengths, bit for bit."""

import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("length", [152, 200, 289, 290, 291])
def test_spline_shared_knots_long(gpu, length):
    """Up to 290 knots the systems on shared knots are built in LDS, 291 with a
    lane per system: the oracle's bits on both sides."""
    from fastemriwaveforms_amd._lib import lib
    from fastemriwaveforms_amd.pipeline import _stream
    rng = np.random.default_rng(length)
    dev = torch.device("cuda", 0)
    for nsys in (1, 33, 70):
        h = rng.uniform(0.2, 1.0, length - 1)
        h[rng.random(length - 1) < 0.2] *= 40.0  # uneven spacing: row interchanges
        t = np.concatenate([[0.0], np.cumsum(h)]) * 1e4
        y = rng.normal(size=(nsys, length))
        t_d, y_d = torch.from_numpy(t).to(dev), torch.from_numpy(y).to(dev)
        out = torch.zeros((4, nsys, length), dtype=torch.float64, device=dev)
        scratch = torch.zeros(4 * length * nsys, dtype=torch.float64, device=dev)
        rc = lib().few_spline_build_async(y_d.data_ptr(), length, 1, t_d.data_ptr(), 0, 1,
                                          out.data_ptr(), nsys * length, length, 1, nsys, length,
                                          0, scratch.data_ptr(), _stream())
        assert rc == 0, lib().few_last_error()
        torch.cuda.synchronize()
        ref, _, info = oracle.interpolate_arrays(np.tile(t, (nsys, 1)), y)
        assert info == 0 and np.array_equal(out.cpu().numpy(), ref), nsys

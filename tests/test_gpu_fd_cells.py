"""The frequency-domain sum over cells (csrc/fd.hip): modes sharing (m, k, n) and
their bin ranges, modes that share the indices only, both tile sizes, many
segments, and the ungrouped form."""

import dataclasses

import numpy as np
import pytest

import oracle
from fastemriwaveforms_amd import synthetic
from helpers import fd_frequencies, oracle_fd, oracle_fd_inputs
from test_gpu_fd import FD_TOL, _grid, _rel_l2, _run_capi

pytestmark = pytest.mark.gpu


def _inp(K, T=0.01, L=25, seed=3, chirp="rising", phases="spline", few=True):
    inp = synthetic.make_input(T, 10.0, L, "m_nonneg_30", K, seed, chirp=chirp, phases=phases)
    if few:   # few distinct (m, n), in random order
        rng = np.random.default_rng(seed)
        inp = dataclasses.replace(inp, m=rng.integers(0, 4, K).astype(np.int32),
                                  n=rng.integers(-3, 4, K).astype(np.int32))
    return inp


@pytest.mark.parametrize("K,minus,phases", [(63, True, "spline"), (64, True, "spline"),
                                            (65, False, "spline"), (150, True, "dopr"),
                                            (300, True, "spline")])
def test_cells_vs_oracle(gpu, K, minus, phases):
    inp = _inp(K, phases=phases)
    freq = _grid(inp)
    ref, (start, end, zero) = oracle_fd(inp, freq, include_minus_m=minus)
    got = _run_capi(inp, freq, start, end, zero, minus)
    assert np.abs(ref).max() > 0
    assert _rel_l2(got, ref) < FD_TOL


def test_same_indices_other_ranges(gpu):
    """Modes with equal (m, k, n) but other bin ranges are not one cell."""
    inp = _inp(80)
    freq = _grid(inp)
    _, (start, end, zero) = oracle_fd(inp, freq)
    rng = np.random.default_rng(1)
    end = np.where(rng.random(end.shape) < 0.1, end - 3, end).astype(np.int32)
    interp, pcoef = oracle_fd_inputs(inp)
    ref = oracle.fd_waveform(interp, inp.t, pcoef, inp.m, inp.k, inp.n, inp.t, freq, start, end,
                             inp.ylms, zero)
    assert _rel_l2(_run_capi(inp, freq, start, end, zero), ref) < FD_TOL


def test_long_tiles(gpu):
    """More than 2^17 owner pairs: two owners per lane; and a zero bin off centre
    (bins without a mirror)."""
    inp = _inp(70, T=0.09, L=20)
    freq = _grid(inp)
    assert len(freq) // 2 >= 1 << 17
    ref, (start, end, zero) = oracle_fd(inp, freq)
    assert _rel_l2(_run_capi(inp, freq, start, end, zero), ref) < FD_TOL
    interp, pcoef = oracle_fd_inputs(inp)
    for z in (zero - 70001, zero + 70001):
        ref = oracle.fd_waveform(interp, inp.t, pcoef, inp.m, inp.k, inp.n, inp.t, freq, start,
                                 end, inp.ylms, z)
        assert _rel_l2(_run_capi(inp, freq, start, end, z), ref) < FD_TOL


@pytest.mark.parametrize("L", [66, 130, 1100])
def test_many_segments(gpu, L):
    """Segment counts around the wave and the index kernel's LDS chunk."""
    inp = _inp(6 if L > 1000 else 70, T=0.01, L=L, few=L < 1000)
    freq = _grid(inp)
    ref, (start, end, zero) = oracle_fd(inp, freq)
    assert _rel_l2(_run_capi(inp, freq, start, end, zero), ref) < FD_TOL


@pytest.mark.parametrize("n,pad,dt", [(1, 0, 3.0), (2, 1, 7.3), (315581, 0, 10.0), (315582, 1, 15.0)])
def test_frequency_grid_device(gpu, n, pad, dt):
    """The grid formed on the GPU holds numpy's values."""
    from fastemriwaveforms_amd import fdinterp
    np.testing.assert_array_equal(fdinterp.frequency_grid_device(n, pad, dt).cpu().numpy(),
                                  fdinterp.frequency_grid(n, pad, dt))

"""GPU test of the FP64 sum of few modes (a lane per sample, csrc/modesum_direct.hip):
against the oracle on both sides of the rule, around its tiles and intervals, added
to an output and written over it, with phases past the fast sincos' range, and bit for
bit the sum of the four-wave tiles at the samples both have."""

import dataclasses

import numpy as np
import pytest

import oracle
from helpers import oracle_waveform

pytestmark = pytest.mark.gpu

TOL = 1e-12   # the FP64 path's bar against the oracle (phase arguments are identical)


def _input(K, num, L=14, seed=1):
    """K modes, num samples, knots up to the last sample."""
    from fastemriwaveforms_amd import synthetic
    T = (num - 1) * 10.0 / synthetic.YRSID_SI * (1.0 + 1e-12)
    inp = synthetic.make_input(T, 10.0, L, "m_nonneg_30", K, seed + K, phases="dopr")
    return dataclasses.replace(inp, num_pts=num)


def _run(inp, overwrite=True):
    from fastemriwaveforms_amd.pipeline import ModeSumProblem
    p = ModeSumProblem(inp)
    p.build_splines()
    p.wave.fill_(2.0 - 3.0j)
    p.mode_sum("fp64", 3, overwrite)
    return p.wave.cpu().numpy()


@pytest.mark.parametrize("K", [1, 2, 3, 4, 5, 7, 8, 15, 16, 17])
@pytest.mark.parametrize("num", [300, 4095, 4097, 65535, 65536, 70001])
def test_few_modes(gpu, K, num):
    inp = _input(K, num)
    ref = oracle_waveform(inp)
    h = _run(inp)
    assert oracle.rel_l2(h, ref) <= TOL
    np.testing.assert_array_equal(_run(inp, overwrite=False), h + (2.0 - 3.0j))


@pytest.mark.parametrize("K", [1, 6, 16])
def test_same_bits_either_way(gpu, K):
    """Outputs on both sides of the rule (4096 samples per mode) hold the same samples."""
    inp = _input(K, 4096 * K + 700, L=20)
    h = _run(inp)
    for num in (4096 * K - 1, 4096 * K):
        np.testing.assert_array_equal(_run(dataclasses.replace(inp, num_pts=num))[:num], h[:num])


def test_past_the_knots_and_long_phases(gpu):
    inp = _input(3, 20000)
    dense = inp.dense.copy()
    dense[0, 3:5] += 3.0e8   # those intervals' phases take the library sincos
    inp = dataclasses.replace(inp, dense=dense, num_pts=21500)
    h, ref = _run(inp), oracle_waveform(inp)
    n = int(np.ceil(inp.t[-1] / inp.dt))
    assert np.all(h[n + 1:] == 0.0)
    assert oracle.rel_l2(h[:n], ref[:n]) <= TOL
    nan = inp.dense.copy()
    nan[0, 2] = np.nan
    h = _run(dataclasses.replace(inp, dense=nan))
    edge = [int(np.ceil(t / inp.dt)) for t in inp.t[2:4]]
    assert np.all(np.isnan(h[edge[0]:edge[1]].real))
    np.testing.assert_array_equal(h[:edge[0]], _run(inp)[:edge[0]])


def test_batch(gpu):
    """A batch of sets on both sides of the rule: the single waveforms' samples."""
    from fastemriwaveforms_amd.pipeline import BatchProblem
    inputs = [_input(K, num, L=9 + K, seed=20) for K, num in
              ((1, 5000), (16, 66000), (17, 3000), (2, 100), (200, 900), (9, 255))]
    b = BatchProblem(inputs)
    b.run("fp64")
    for i, inp in enumerate(inputs):
        np.testing.assert_array_equal(b.waveform(i).cpu().numpy(), _run(inp))


@pytest.mark.parametrize("prepared,summed", [(3, 200), (200, 3), (16, 17), (5, 6)])
@pytest.mark.parametrize("num", [70001, 140000])
def test_sum_of_other_modes_than_prepared(gpu, prepared, summed, num):
    """The interval plan does not depend on the modes: a sum may follow the preparing
    call of another set, whichever way either runs, and another precision's stays
    refused."""
    from fastemriwaveforms_amd._lib import lib
    from fastemriwaveforms_amd.pipeline import ModeSumProblem, _stream
    a, b = _input(prepared, num), _input(summed, num)
    pa, pb = ModeSumProblem(a), ModeSumProblem(dataclasses.replace(b, t=a.t, dense=a.dense))
    pb.build_splines()

    def call(p, ws, precision, stage):
        return lib().few_get_waveform_plan_async(
            p.wave.data_ptr(), p.interp.data_ptr(), p.t.data_ptr(), p.pcoef.data_ptr(), None,
            p.m.data_ptr(), p.k.data_ptr(), p.n.data_ptr(), p.L, p.N, p.K, p.ylm.data_ptr(), p.dt,
            p.t.data_ptr(), precision, 0, stage, ws.data_ptr(), ws.numel(), _stream())

    want = pb.run("fp64").cpu().numpy()
    ws = pb.ws if pb.ws.numel() >= pa.ws.numel() else pa.ws
    pb.wave.fill_(5.0)
    assert call(pa, ws, 0, 1) == 0, lib().few_last_error()
    assert call(pb, ws, 0, 6) == 0, lib().few_last_error()
    np.testing.assert_array_equal(pb.wave.cpu().numpy(), want)
    pb.mode_sum("mixed16", 1)
    assert call(pb, pb.ws, 0, 6) != 0

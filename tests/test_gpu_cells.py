"""GPU parity of the FP64 sum over cells (csrc/cells.hip, csrc/modesum_direct.hip):
modes sharing (m, k, n) in any order and number, both tile sizes, the ungrouped
form, phases past the fast sincos' range."""

import dataclasses

import numpy as np
import pytest

import oracle
from helpers import oracle_waveform

pytestmark = pytest.mark.gpu

TOL = 1e-12   # the FP64 path's bar against the oracle (phase arguments are identical)


def _input(K, seed, T=0.002, dt=10.0, L=9, kind="m_nonneg_30"):
    """K modes in random order; small sets repeat a few (m, k, n) many times."""
    from fastemriwaveforms_amd import synthetic
    inp = synthetic.make_input(T, dt, L, kind, max(K, 1), seed, phases="dopr")
    rng = np.random.default_rng(seed)
    o = rng.permutation(inp.K)
    ylm = np.concatenate([inp.ylms[:inp.K][o], inp.ylms[inp.K:][o]])
    return dataclasses.replace(inp, teuk=np.ascontiguousarray(inp.teuk[:, o]), ylms=ylm,
                               l=inp.l[o], m=inp.m[o], k=inp.k[o], n=inp.n[o])


def _run(inp):
    from fastemriwaveforms_amd.pipeline import ModeSumProblem
    return ModeSumProblem(inp).run("fp64").cpu().numpy()


@pytest.mark.parametrize("K", [1, 2, 63, 64, 65, 255, 256, 257, 1000, 2047, 2049, 3843])
def test_mode_counts(gpu, K):
    inp = _input(K, 100 + K)
    assert oracle.rel_l2(_run(inp), oracle_waveform(inp)) <= TOL


@pytest.mark.parametrize("case", ["one_cell", "no_cell", "polar", "signs"])
def test_groupings(gpu, case):
    inp = _input(300, 7, kind="k1_20" if case == "polar" else "m_nonneg_30")
    if case == "one_cell":
        inp = dataclasses.replace(inp, m=np.full_like(inp.m, 2), n=np.full_like(inp.n, -3))
    if case == "no_cell":   # every mode its own (m, k, n)
        inp = dataclasses.replace(inp, m=(np.arange(300) % 11).astype(np.int32),
                                  n=(np.arange(300) // 11 - 10).astype(np.int32))
    if case == "signs":     # (m, n) and (-m, -n) are different cells, m = 0 has no -m term
        s = np.where(np.arange(300) % 2, 1, -1).astype(np.int32)
        inp = dataclasses.replace(inp, m=(inp.m % 3) * s, n=(inp.n % 4) * s)
    assert oracle.rel_l2(_run(inp), oracle_waveform(inp)) <= TOL


def test_ungrouped_workspace(gpu):
    """A workspace with room for the interval plan only runs one cell per mode;
    grouped and ungrouped sums differ by rounding (each within TOL of the oracle)."""
    from fastemriwaveforms_amd._lib import check, lib
    from fastemriwaveforms_amd.pipeline import ModeSumProblem, _stream
    import torch
    inp = _input(500, 3)
    p = ModeSumProblem(inp)
    grouped = p.run("fp64").clone()
    small = int(lib().few_plan_workspace_bytes(None, p.L, p.N, 0))
    assert small < p.plan.workspace_bytes(p.L, p.N, "fp64")
    p.wave.fill_(7.0)
    check(lib().few_get_waveform_plan_async(
        p.wave.data_ptr(), p.interp.data_ptr(), p.t.data_ptr(), p.pcoef.data_ptr(), p.plan.handle,
        p.m.data_ptr(), p.k.data_ptr(), p.n.data_ptr(), p.L, p.N, p.K, p.ylm.data_ptr(), p.dt,
        p.t.data_ptr(), 0, 0, 7, p.ws.data_ptr(), small, _stream()), "get_waveform")
    ref = oracle_waveform(inp)
    assert oracle.rel_l2(p.wave.cpu().numpy(), ref) <= TOL
    assert oracle.rel_l2(grouped.cpu().numpy(), ref) <= TOL
    assert float((p.wave - grouped).abs().max()) <= TOL * float(grouped.abs().max())
    torch.cuda.synchronize()


def test_tile_sizes_same_bits(gpu):
    """Outputs on both sides of the tile rule (2^17 samples) hold the same samples."""
    from fastemriwaveforms_amd import synthetic
    base = synthetic.make_input(0.05, 10.0, 12, "m_nonneg_30", 90, 11)
    runs = [_run(dataclasses.replace(base, num_pts=n)) for n in (131071, 131072, 131329)]
    # the last interval's samples depend on the output length only through the
    # knots, which are the same
    for h in runs[1:]:
        np.testing.assert_array_equal(h[:131071], runs[0])


def test_overwrite_past_the_knots(gpu):
    """Overwriting sum: samples past the last interval read zero."""
    inp = _input(80, 5)
    h = _run(dataclasses.replace(inp, num_pts=inp.num_pts + 700))
    n = int(np.ceil(inp.t[-1] / inp.dt))
    ref = oracle_waveform(inp)
    assert np.all(h[n + 1:] == 0.0)
    assert oracle.rel_l2(h[:n], ref[:n]) <= TOL


def test_phases_beyond_the_fast_range(gpu):
    """Phases of 1e9 rad in some intervals: those tiles take the library sincos."""
    inp = _input(100, 9)
    dense = inp.dense.copy()
    dense[0, 3:5] += 3.0e8
    inp = dataclasses.replace(inp, dense=dense)
    h, ref = _run(inp), oracle_waveform(inp)
    assert oracle.rel_l2(h, ref) <= TOL


# ------------------------------------------------------------------ adjoint

def _adjoint(inp, g, ws_bytes=None):
    """(dL/d amplitude coefficients (4, L, 2K), dL/d phase coefficients (4, L, 3))"""
    import torch
    from fastemriwaveforms_amd._lib import check, lib
    from fastemriwaveforms_amd.pipeline import ModeSumProblem, _stream
    p = ModeSumProblem(inp)
    p.build_splines()
    need = int(lib().few_adjoint_workspace_bytes(p.L, p.N, p.K, 0))
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    gi = torch.full((4, p.L, 2 * p.K), 5.0, dtype=torch.float64, device="cuda")
    gp = torch.full((4, p.L, 3), 5.0, dtype=torch.float64, device="cuda")
    gd = torch.from_numpy(g).cuda()
    check(lib().few_waveform_adjoint_async(
        gd.data_ptr(), p.interp.data_ptr(), p.t.data_ptr(), p.pcoef.data_ptr(), p.m.data_ptr(),
        p.k.data_ptr(), p.n.data_ptr(), p.L, p.N, p.K, p.ylm.data_ptr(), p.dt, p.t.data_ptr(),
        gi.data_ptr(), gp.data_ptr(), 0, ws.data_ptr(), need if ws_bytes is None else ws_bytes(need, p),
        _stream()), "adjoint")
    return gi.cpu().numpy(), gp.cpu().numpy()


def _adjoint_ref(inp, g):
    from helpers import oracle_coefficients
    interp, pcoef = oracle_coefficients(inp)
    return oracle.waveform_adjoint(g, interp, inp.t, pcoef, inp.m, inp.k, inp.n, inp.L, inp.num_pts,
                                   inp.K, inp.ylms, inp.dt, inp.t)


def _close(got, ref):
    # per power: each is a sum of its own scale
    for p in range(4):
        assert oracle.rel_l2(got[0][p], ref[0][p]) <= TOL
        assert oracle.rel_l2(got[1][p], ref[1][p]) <= 10 * TOL   # cancelling sums over all modes


@pytest.mark.parametrize("K", [1, 63, 64, 65, 127, 128, 129, 400, 1500])
def test_adjoint_mode_counts(gpu, K):
    inp = _input(K, 500 + K, L=6)
    rng = np.random.default_rng(K)
    g = rng.normal(size=inp.num_pts) + 1j * rng.normal(size=inp.num_pts)
    _close(_adjoint(inp, g), _adjoint_ref(inp, g))


@pytest.mark.parametrize("samples", [1, 63, 64, 65, 255, 257, 2048, 2049, 4500])
def test_adjoint_interval_lengths(gpu, samples):
    """Intervals of every length around the 64-sample groups and the chunk."""
    inp = _input(70, 21, T=0.004, L=5)
    t = np.array([0.0, samples, samples + 700, samples + 701, 12000]) * inp.dt
    inp = dataclasses.replace(inp, t=t, num_pts=samples + 2000)
    rng = np.random.default_rng(samples)
    g = rng.normal(size=inp.num_pts) + 1j * rng.normal(size=inp.num_pts)
    _close(_adjoint(inp, g), _adjoint_ref(inp, g))


def test_adjoint_ungrouped_and_big_phases(gpu):
    inp = _input(90, 33, L=6)
    rng = np.random.default_rng(0)
    g = rng.normal(size=inp.num_pts) + 1j * rng.normal(size=inp.num_pts)
    ref = _adjoint_ref(inp, g)
    _close(_adjoint(inp, g), ref)
    # one byte short of the index's room: one cell per mode
    _close(_adjoint(inp, g, ws_bytes=lambda need, p: need - 1), ref)
    dense = inp.dense.copy()
    dense[0, 2:4] += 3.0e8
    inp = dataclasses.replace(inp, dense=dense)
    _close(_adjoint(inp, g), _adjoint_ref(inp, g))

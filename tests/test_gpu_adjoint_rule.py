"""GPU test of the FP64 adjoint on both sides of the rule that groups the modes into
cells (more than 256 workgroups with a cell per mode): against the oracle, with the
groupings, interval lengths and phases that matter there."""

import dataclasses

import numpy as np
import pytest

from test_gpu_cells import _adjoint, _adjoint_ref, _close, _input

pytestmark = pytest.mark.gpu


def _check(inp, seed, **kw):
    rng = np.random.default_rng(seed)
    g = rng.normal(size=inp.num_pts) + 1j * rng.normal(size=inp.num_pts)
    _close(_adjoint(inp, g, **kw), _adjoint_ref(inp, g))


def _blocks(inp):
    return ((inp.num_pts + 2047) // 2048 + inp.L) * ((inp.K + 127) // 128)


# knots so that the workgroups lie on either side of 256
@pytest.mark.parametrize("K,L,grouped", [(63, 300, True), (64, 252, False), (64, 253, True),
                                         (65, 270, True), (127, 260, True), (128, 260, True),
                                         (129, 120, False), (129, 130, True), (400, 70, True),
                                         (1500, 12, False), (1500, 40, True)])
def test_mode_counts(gpu, K, L, grouped):
    inp = _input(K, 40 + K, L=L)
    assert (_blocks(inp) > 256) == grouped
    _check(inp, K)


@pytest.mark.parametrize("case", ["one_cell", "no_cell", "polar", "short_workspace", "big_phases"])
def test_grouped(gpu, case):
    inp = _input(300, 8, L=120, kind="k1_20" if case == "polar" else "m_nonneg_30")
    assert _blocks(inp) > 256
    if case == "one_cell":
        inp = dataclasses.replace(inp, m=np.full_like(inp.m, 2), n=np.full_like(inp.n, -3))
    if case == "no_cell":
        inp = dataclasses.replace(inp, m=(np.arange(300) % 11).astype(np.int32),
                                  n=(np.arange(300) // 11 - 10).astype(np.int32))
    if case == "big_phases":
        dense = inp.dense.copy()
        dense[0, 50:55] += 3.0e8
        inp = dataclasses.replace(inp, dense=dense)
    kw = dict(ws_bytes=lambda need, p: need - 1) if case == "short_workspace" else {}
    _check(inp, 3, **kw)

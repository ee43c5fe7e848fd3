"""GPU test of the cell index where the rows of two modes differ but share the 32-bit
hash by which they are compared first: no mode is then grouped (csrc/cells.hip)."""

import numpy as np
import pytest

import oracle
from helpers import oracle_fd, oracle_fd_inputs
from test_gpu_fd import FD_TOL, _grid, _rel_l2, _run_capi
from test_gpu_fd_cells import _inp

pytestmark = pytest.mark.gpu


def _hashes(start, end):
    """cell_hash_kernel's hash of the rows (start, end), each (rows, segments)."""
    u = np.uint64
    v = (start.astype(np.uint32).astype(u) << u(32)) | end.astype(np.uint32).astype(u)
    with np.errstate(over="ignore"):
        v = v + u(0x9e3779b97f4a7c15) * np.arange(1, start.shape[1] + 1, dtype=u)
        v = (v ^ (v >> u(30))) * u(0xbf58476d1ce4e5b9)
        v = (v ^ (v >> u(27))) * u(0x94d049bb133111eb)
        h = (v ^ (v >> u(31))).sum(axis=1, dtype=u)
    return ((h ^ (h >> u(32))) & u(0xffffffff)).astype(np.uint32)


def _colliding(start, end):
    """Two different rows of bin ranges with one hash: variants of a mode's own row
    with the last bins of some segments left out."""
    wide = np.nonzero(end - start >= 4)[0][:9]
    assert len(wide) == 9
    digits = np.stack(np.unravel_index(np.arange(4 ** 9), (4,) * 9), axis=1)
    rows = np.repeat(end[None], len(digits), axis=0)
    rows[:, wide] -= digits
    h = _hashes(np.broadcast_to(start, rows.shape), rows)
    order = np.argsort(h, kind="stable")
    same = np.nonzero(h[order][1:] == h[order][:-1])[0]
    assert len(same) > 0
    a, b = rows[order[same[0]]], rows[order[same[0] + 1]]
    assert np.any(a != b)
    return a, b


def test_rows_with_one_hash(gpu):
    inp = _inp(90, T=0.02, L=40)
    freq = _grid(inp)
    _, (start, end, zero) = oracle_fd(inp, freq)
    # the (m, n) with the most modes among those that sweep bins in enough segments
    ok = (end - start >= 4).sum(axis=1) >= 9
    keys, count = np.unique(np.stack([inp.m[ok], inp.n[ok]]), axis=1, return_counts=True)
    assert count.max() >= 3
    key = keys[:, count.argmax()]
    q = np.nonzero(ok & (inp.m == key[0]) & (inp.n == key[1]))[0]
    a, b = _colliding(start[q[0]], end[q[0]])
    end = end.copy()
    end[q[0]], end[q[1]] = a, b
    interp, pcoef = oracle_fd_inputs(inp)
    ref = lambda e: oracle.fd_waveform(interp, inp.t, pcoef, inp.m, inp.k, inp.n, inp.t, freq, start,
                                       e, inp.ylms, zero)
    want = ref(end)
    merged = end.copy()
    merged[q[1]] = a   # what grouping the two would give
    assert _rel_l2(ref(merged), want) > 100 * FD_TOL
    assert _rel_l2(_run_capi(inp, freq, start, end, zero), want) < FD_TOL

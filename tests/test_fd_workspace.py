"""Workspace of the frequency-domain sum (few_fd_workspace_bytes): its bound, and
the sums in the smallest workspace they take and over several slabs of cells."""

import ctypes

import numpy as np
import pytest

from fastemriwaveforms_amd._lib import check, lib
from helpers import oracle_fd, oracle_fd_inputs
from test_gpu_fd import FD_TOL, _grid, _rel_l2, _run_capi
from test_gpu_fd_cells import _inp


def _asked(K, nseg):
    n = ctypes.c_size_t(0)
    check(lib().few_fd_workspace_bytes(K, nseg, ctypes.byref(n)), "fd workspace size")
    return n.value


def _least(K, nseg):
    """28 B per (mode, segment): a scan of 64-bit counts, and three ints and a count."""
    up = lambda b: (b + 255) // 256 * 256
    n = K * nseg
    return up(8 * (2 * n + 2 + (n + 1023) // 1024)) + up(4 * K) + 3 * up(4 * n)


@pytest.mark.parametrize("K,nseg", [(1, 1), (6, 29), (64, 1), (500, 99), (3843, 119), (3843, 1099),
                                    (12987, 199)])
def test_size_bounded(K, nseg):
    """The least the sums take, or the index and at most 64 MB of tables (one cell's
    at least), whatever the number of modes."""
    assert _least(K, nseg) <= _asked(K, nseg) <= _least(K, nseg) + (1 << 26) + 600 * nseg + 40 * K + 4096


def _run_with(inp, freq, start, end, zero, nbytes, minus=True, separate=False):
    import torch
    dev = torch.device("cuda", 0)
    interp, pcoef = oracle_fd_inputs(inp)
    d = lambda a, dt=torch.float64: torch.from_numpy(np.ascontiguousarray(a)).to(dev, dt)
    wave = torch.zeros((inp.K, len(freq)) if separate else len(freq), dtype=torch.complex128,
                       device=dev)
    x = [d(interp), d(inp.t), d(pcoef), d(inp.m, torch.int32), d(inp.k, torch.int32),
         d(inp.n, torch.int32), d(inp.t), d(freq), d(start, torch.int32), d(end, torch.int32),
         d(inp.ylms, torch.complex128)]
    ws = torch.full((nbytes + 4096,), 171, dtype=torch.uint8, device=dev)
    a = [v.data_ptr() for v in x]
    rc = lib().few_get_waveform_generic_fd_async(
        wave.data_ptr(), a[0], a[1], a[2], a[3], a[4], a[5], inp.K, inp.dt, a[6], inp.L, len(freq),
        a[7], a[8], a[9], inp.L - 1, a[10], zero, int(minus), int(separate), ws.data_ptr(), nbytes,
        int(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert bool((ws[nbytes:] == 171).all())  # nothing written past the workspace
    return rc, wave.cpu().numpy()


@pytest.mark.gpu
@pytest.mark.parametrize("K,L", [(1, 2), (6, 25), (63, 25), (64, 2), (64, 25), (150, 40)])
@pytest.mark.parametrize("separate", [False, True])
def test_least_workspace(gpu, K, L, separate):
    """The least workspace is accepted by either path; a byte less is refused."""
    inp = _inp(K, L=max(L, 4))
    nseg = inp.L - 1
    freq = _grid(inp)
    ref, (start, end, zero) = oracle_fd(inp, freq, include_minus_m=not separate,
                                        separate_modes=separate)
    least = _least(K, nseg)
    rc, got = _run_with(inp, freq, start, end, zero, least, not separate, separate)
    assert rc == 0, lib().few_last_error()
    assert np.abs(ref).max() > 0 and _rel_l2(got, ref) < FD_TOL
    rc, got = _run_with(inp, freq, start, end, zero, least - 1, not separate, separate)
    assert rc != 0 and not np.any(got)


@pytest.mark.gpu
@pytest.mark.parametrize("few", [False, True])
def test_slabs(gpu, few):
    """More modes than a slab of tables holds (190 cells of 1099 segments): the
    cells fill two slabs, or stay within the first."""
    inp = _inp(320, T=0.01, L=1100, few=few)
    cells = len(np.unique(np.stack([inp.m, inp.n]), axis=1).T)
    assert cells > 200 if not few else cells < 60
    freq = _grid(inp)
    ref, (start, end, zero) = oracle_fd(inp, freq)
    assert _rel_l2(_run_capi(inp, freq, start, end, zero), ref) < FD_TOL

"""The bin evaluation of the frequency-domain kernels (fd_bin_fast, csrc/fd.hip)
on the CPU, against the oracle and against the reference's operations.

fd_bin_fast takes the same roots, phase and stationary-phase factor as fd_bin
through fewer operations; both round, so they agree to the conditioning of the
root: 2 pi f t - phase is up to ~1e5 rad here, an ulp of the time (1.5e-11 of
the phase) is the unit of the difference, as between two libms."""

import ctypes

import numpy as np
import pytest

import oracle
from fastemriwaveforms_amd import synthetic
from helpers import oracle_fd, oracle_fd_inputs

P = ctypes.c_void_p
FD_TOL = 2e-11   # the bar of the GPU comparison


def _p(a):
    return ctypes.c_void_p(a.ctypes.data)


def _fast(twin, inp, freq, start, end, zero, minus):
    interp, pcoef = oracle_fd_inputs(inp)
    i32 = lambda a: np.ascontiguousarray(a, dtype=np.int32)
    m, k, n, s0, s1 = i32(inp.m), i32(inp.k), i32(inp.n), i32(start), i32(end)
    wave = np.zeros(len(freq), dtype=np.complex128)
    ylm = np.ascontiguousarray(inp.ylms)
    I = ctypes.c_int
    twin.twin_fd_waveform_fast.argtypes = [P] * 7 + [I, P, I, I, P, P, P, I, P, I, I]
    twin.twin_fd_waveform_fast(_p(wave), _p(interp), _p(inp.t), _p(pcoef), _p(m), _p(k), _p(n),
                               inp.K, _p(inp.t), inp.L, len(freq), _p(freq), _p(s0), _p(s1),
                               inp.L - 1, _p(ylm), zero, int(minus))
    return wave


@pytest.mark.parametrize("case", [dict(), dict(chirp="smooth", seed=5), dict(phases="dopr", seed=8),
                                  dict(mode="k1_20", phases="dopr", seed=9),
                                  dict(T=0.2, L=60, K=8, seed=21)])
@pytest.mark.parametrize("minus", [True, False])
def test_fast_vs_oracle(twin, case, minus):
    c = dict(T=0.05, L=40, K=16, seed=11, chirp="rising", mode="m_nonneg_30", phases="spline")
    c.update(case)
    inp = synthetic.make_input(c["T"], 10.0, c["L"], c["mode"], c["K"], c["seed"],
                               chirp=c["chirp"], phases=c["phases"])
    freq = oracle.fd_frequency_grid(inp.num_pts, 1 - inp.num_pts % 2, inp.dt)
    ref, (start, end, zero) = oracle_fd(inp, freq, include_minus_m=minus)
    got = _fast(twin, inp, freq, start, end, zero, minus)
    assert np.abs(ref).max() > 0
    err = float(np.linalg.norm(got - ref) / np.linalg.norm(ref))
    print(case, err)
    assert err < FD_TOL


def test_roots(twin):
    """Three real roots, one real root of either sign, and the degenerate cubics
    that give the reference no root inside any segment."""
    rng = np.random.default_rng(4)
    a = rng.normal(size=(400, 4)) * 10.0 ** rng.uniform(-2, 2, (400, 4))
    ref, out = np.zeros((400, 3)), np.zeros((400, 3))
    twin.twin_fd_cube_roots.argtypes = twin.twin_fd_roots.argtypes = [P, ctypes.c_long, P]
    twin.twin_fd_cube_roots(_p(a), 400, _p(ref))
    twin.twin_fd_roots(_p(a), 400, _p(out))
    # the same operations but for the sincos of a third of the argument (an ulp)
    size = np.abs(ref).max(axis=1) + np.abs(a[:, 1] / (3 * a[:, 0]))
    assert np.all(np.abs(out - ref) <= 1e-15 * size[:, None])
    same = np.mean(out == ref)
    print("identical roots", same)
    assert same > 0.95   # "98 % of them bit for bit" (csrc/fd.hip)
    three = np.isclose(ref[:, 1], ref[:, 2], rtol=1e-9)
    assert three.any() and (~three).any()
    bad = np.array([[0.0, 1.0, 2.0, 3.0], [0.0, -1.0, 2.0, 3.0], [1.0, 0.0, 0.0, 0.0],
                    [np.nan, 1.0, 1.0, 1.0], [1.0, 1.0, 1.0, np.nan], [0.0, 0.0, 1.0, 1.0]])
    ref, out = np.zeros((len(bad), 3)), np.zeros((len(bad), 3))
    twin.twin_fd_cube_roots(_p(bad), len(bad), _p(ref))
    twin.twin_fd_roots(_p(bad), len(bad), _p(out))
    assert not np.isfinite(ref).any() and not np.isfinite(out).any()


def test_amp(twin):
    """The stationary-phase factor on both sides of |x| = 7 and for both signs:
    a handful of rounded terms; exact zeros take the general form's result."""
    rng = np.random.default_rng(6)
    x = np.concatenate([np.linspace(-60, 60, 1201), 10.0 ** rng.uniform(-6, 12, 300),
                        -10.0 ** rng.uniform(-6, 12, 300)])
    x = x[np.abs(np.abs(x) - 7.0) > 1e-9]   # the series differ by ~1e-6 at the switch itself
    x = x[x != 0.0]
    fdot = np.sign(x) * 10.0 ** rng.uniform(-14, -8, len(x))
    fddot = np.sqrt(2 * np.pi * fdot ** 3 / (3 * x)) * rng.choice([-1.0, 1.0], len(x))
    fast, ref = np.zeros(len(x), np.complex128), np.zeros(len(x), np.complex128)
    twin.twin_fd_amp.argtypes = [P, P, ctypes.c_long, P, P]
    twin.twin_fd_amp(_p(fdot), _p(fddot), len(x), _p(fast), _p(ref))
    assert np.all(np.isfinite(ref))
    assert np.all(np.abs(fast - ref) <= 4e-15 * np.abs(ref))
    edge = np.array([0.0, 1e-12, -1e-12, np.nan, 1e-12, np.inf])
    edge2 = np.array([1e-20, 0.0, 0.0, 1e-20, np.nan, 1e-20])
    fast, ref = np.zeros(6, np.complex128), np.zeros(6, np.complex128)
    twin.twin_fd_amp(_p(edge), _p(edge2), 6, _p(fast), _p(ref))
    assert np.array_equal(fast, ref, equal_nan=True)

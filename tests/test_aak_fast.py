"""The AAK kernel's Bessel values (aak_bessel5, csrc/aak.hip) against the five
Miller recurrences they replace, on the CPU through the host twin."""

import ctypes

import numpy as np
import pytest

from helpers import aak_input, oracle_aak

P = ctypes.c_void_p


def _p(a):
    return ctypes.c_void_p(a.ctypes.data)


@pytest.mark.parametrize("nmodes", [30, 120])
def test_bessel5(twin, nmodes):
    """Every harmonic n and eccentricities from 1e-9 (the rescaled recurrences
    take over) to 0.95.  A recurrence of ~n + sqrt(40 n) fused steps grows by
    rounding at each: 2^-53 times the steps, of each value; orders above x have
    no sign changes, so the relative error is bounded the same way."""
    rng = np.random.default_rng(3)
    e = np.concatenate([10.0 ** rng.uniform(-9, -2, 40), rng.uniform(0.01, 0.95, 120), [0.5, 2 / 3]])
    n = np.repeat(np.arange(1, nmodes + 1), len(e))
    x = n * np.tile(e, nmodes)
    order = (n - 2).astype(np.int32)
    fast, ref = np.zeros((len(n), 5)), np.zeros((len(n), 5))
    twin.twin_aak_bessel5.argtypes = [P, P, ctypes.c_long, P, P]
    twin.twin_aak_bessel5(_p(order), _p(x), len(n), _p(fast), _p(ref))
    use = (order[:, None] + np.arange(5)) >= 0
    assert np.all(np.isfinite(fast[use])) and np.all(np.isfinite(ref[use]))
    steps = (n + 2 + np.sqrt(40.0 * (n + 2)))[:, None]
    err = np.abs(fast - ref)
    print("largest relative difference", np.max((err / np.maximum(np.abs(ref), 1e-300))[use]))
    assert np.all((err <= 4 * steps * 2.0 ** -53 * np.abs(ref) + 1e-300)[use])


def test_bessel5_degenerate(twin):
    """x = 0, negative and NaN take the reference's routines."""
    order = np.array([-1, 0, 3, 3, 3, 10], np.int32)
    x = np.array([0.0, 0.0, 0.0, -1.5, np.nan, np.inf])
    fast, ref = np.zeros((6, 5)), np.zeros((6, 5))
    twin.twin_aak_bessel5.argtypes = [P, P, ctypes.c_long, P, P]
    twin.twin_aak_bessel5(_p(order), _p(x), 6, _p(fast), _p(ref))
    np.testing.assert_array_equal(fast, ref)


@pytest.mark.parametrize("mich", [False, True])
@pytest.mark.parametrize("case", [dict(), dict(e0=0.7, e1=0.5), dict(e0=0.0, e1=0.0),
                                  dict(dopr=True), dict(e0=1e-7, e1=1e-6), dict(Y0=-0.6),
                                  dict(S=0.0), dict(nmodes=1), dict(nmodes=2), dict(nmodes=3),
                                  dict(nmodes=40, e0=0.6, e1=0.6)])
def test_sample_fast(twin, case, mich):
    """The kernel's form of a sample against the oracle; the bar of the GPU
    comparison (phases of 1e4 rad; their operations are the same)."""
    case = dict(case)
    nmodes, S = case.pop("nmodes", 15), case.pop("S", 0.5)
    t, c, prm, n_out = aak_input(T_years=0.005, L=10, seed=4, **case)
    prm = dict(prm, S=S)
    ref = oracle_aak(t, c, prm, n_out, nmodes=nmodes, mich=mich)
    dense = np.ascontiguousarray(np.transpose(c, (2, 0, 1)))
    got = np.zeros(n_out, dtype=np.complex128)
    twin.twin_aak_waveform_fast.argtypes = [P, P] + [ctypes.c_double] * 8 + [
        ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_double, P]
    twin.twin_aak_waveform_fast(_p(got), _p(dense), prm["M"], prm["S"], prm["mu"], prm["qS"],
                                prm["phiS"], prm["qK"], prm["phiK"], prm["dist"], nmodes, int(mich),
                                len(t), n_out, 10.0, _p(t))
    scale = np.linalg.norm(ref)
    assert scale > 0 or not np.any(got)
    assert np.linalg.norm(got - ref) <= 1e-12 * scale

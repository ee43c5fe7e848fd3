"""The pieces of the FP64 sum over cells (modes sharing (m, k, n)) on the CPU,
through the host twin: the half-turn sincos and the combined cell term."""

import ctypes

import numpy as np
import pytest

from test_host_twin import _p, _sincos_ref, tw  # noqa: F401  (fixture)

P = ctypes.c_void_p


def test_sincos_half_turns(tw):
    """Against an 80-digit reference, up to the ends of the range and at the
    half-turn boundaries.  Rounding: the reduced argument, two products and the
    last addition, each at most half an ulp of values below 1.6: 2 ulp of 1."""
    tw.twin_sincos_half_turns.argtypes = [P, P, P, P, ctypes.c_long]
    rng = np.random.default_rng(1)
    k = np.arange(-40, 41) * (np.pi / 2)
    x = np.concatenate([rng.uniform(-1e8, 1e8, 1500), rng.uniform(-1e4, 1e4, 500),
                        rng.uniform(-4, 4, 500), k, np.nextafter(k, 99), np.nextafter(k, -99),
                        [0.0, -0.0, 1e-300, 1.05e8, -1.05e8, 355.0, 103993.0]])
    s, c, ok = np.zeros_like(x), np.zeros_like(x), np.zeros(len(x), np.int32)
    tw.twin_sincos_half_turns(_p(x), _p(s), _p(c), _p(ok), len(x))
    assert ok.all()
    rs, rc = _sincos_ref(x)
    ulp = np.spacing(1.0)
    print("sin", np.max(np.abs(s - rs)), "cos", np.max(np.abs(c - rc)))
    assert np.max(np.abs(s - rs)) <= 2 * ulp
    assert np.max(np.abs(c - rc)) <= 2 * ulp
    big = np.array([1.06e8, -3.0e9, 1e300, np.inf, -np.inf, np.nan])
    s, c, ok = np.zeros_like(big), np.zeros_like(big), np.ones(len(big), np.int32)
    tw.twin_sincos_half_turns(_p(big), _p(s), _p(c), _p(ok), len(big))
    assert not ok.any()


@pytest.mark.parametrize("members", [1, 2, 9])
@pytest.mark.parametrize("mkn", [(0, 0, 3), (2, 0, -30), (10, -2, 30), (-3, 1, 0)])
def test_cell_term(tw, members, mkn):
    """The combined term equals the members' terms, each written as the two
    complex exponentials: at most ~20 rounded operations per member on values
    below the sum of the members' magnitudes."""
    D = ctypes.c_double
    tw.twin_cell_term.argtypes = [ctypes.c_int, P, P] + [D] * 7 + [ctypes.c_int, P]
    rng = np.random.default_rng(members)
    m, k, n = mkn
    coef = rng.normal(size=(members, 8)) * 10.0 ** -np.array([0, 4, 8, 12] * 2)
    ylm = rng.normal(size=(members, 4))
    for x, ph in [(0.0, (1.0, 2.0, 3.0)), (3e4, (1.2e5, -40.0, 9.9e4)), (2e4, (4e8, 1e3, -3e9))]:
        big = max(abs(p) for p in ph) > 1e6
        phase = float(m) * ph[0] + float(k) * ph[1] + float(n) * ph[2]
        xs = x ** np.arange(4)
        A = coef[:, :4] @ xs + 1j * (coef[:, 4:] @ xs)
        yp, ym = ylm[:, 0] + 1j * ylm[:, 1], ylm[:, 2] + 1j * ylm[:, 3]
        Pq = np.exp(-1j * phase) * A
        ref = np.sum(Pq * yp) + (np.sum(np.conj(Pq) * ym) if m else 0.0)
        scale = np.sum(np.abs(A) * (np.abs(yp) + np.abs(ym)))
        out = np.zeros(2)
        tw.twin_cell_term(members, _p(coef), _p(ylm), m, k, n, x, *ph, int(big), _p(out))
        assert abs(out[0] + 1j * out[1] - ref) <= 20 * 2.3e-16 * scale, (x, mkn)

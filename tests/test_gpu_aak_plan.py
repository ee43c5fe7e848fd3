"""GPU test of the AAK segment plan (one knot per lane) around its 64-knot steps, with
outputs that end before the last knot, at it and past it, against the oracle's plan."""

import numpy as np
import pytest

from fastemriwaveforms_amd import pyinterp
from helpers import aak_input, oracle_aak

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [2, 63, 64, 65, 66, 129, 130])
@pytest.mark.parametrize("extent", [0.02, 0.6, 1.0, 1.02])
def test_plan(gpu, L, extent):
    t, c, prm, n_full = aak_input(T_years=0.004, L=max(L, 4), seed=L)
    t, c = np.ascontiguousarray(t[:L]), np.ascontiguousarray(c[:L - 1])
    last = int(np.ceil(t[-1] / 10.0))
    n = max(2, int(extent * last))
    ref = oracle_aak(t, c, prm, n, nmodes=4)
    wave = np.full(n, 3.0 + 4.0j)
    dense = np.ascontiguousarray(np.transpose(c, (2, 0, 1))).flatten()
    pyinterp.pyWaveform(wave, dense, prm["M"], prm["S"], prm["mu"], prm["qS"], prm["phiS"],
                        prm["qK"], prm["phiK"], prm["dist"], 4, False, L, n, 10.0, t.copy())
    covered = min(n, last)
    assert np.linalg.norm(wave[:covered] - ref[:covered]) <= 1e-12 * np.linalg.norm(ref[:covered])
    assert np.all(wave[covered:] == 3.0 + 4.0j)   # past the last knot: untouched

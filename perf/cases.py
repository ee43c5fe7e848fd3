"""Workloads of the interpolated mode sum and its neighbours, for timing and comparison.

Each case is what a program using this package does with one call, through the
public entry points, from data it already holds on the GPU:

* ``class``  -- ``InterpolatedModeSum`` called like FEW's summation module (knot
  amplitudes, dense-output phases, mode arrays in; waveform out);
* ``step``   -- ``ModeSumProblem.run``: knots to waveform with every buffer kept,
  the inner loop of a sampler working on one waveform shape;
* ``batch``  -- ``BatchProblem.run``: many uneven waveforms in one call;
* ``grad``   -- ``DifferentiableModeSum`` forward and backward (waveform and the
  gradients of all knot values);
* ``fd``     -- ``FDInterpolatedModeSum``, the frequency-domain waveform;
* ``aak``    -- ``AAKSummation``;
* ``amp``    -- ``AmpInterp2D``, the amplitudes of a mode set along a trajectory;
* ``spline`` -- ``CubicSplineInterpolant`` built and evaluated.

Sizes are those of the package's own workloads (``synthetic.WORKLOADS``, the
256-waveform batch) and of the ranges around them.
"""

import functools
import math

import numpy as np
import torch

from fastemriwaveforms_amd import synthetic
from fastemriwaveforms_amd.aakwave import AAKSummation
from fastemriwaveforms_amd.amplitude import AmpInterp2D
from fastemriwaveforms_amd.autograd import DifferentiableModeSum
from fastemriwaveforms_amd.fdinterp import FDInterpolatedModeSum
from fastemriwaveforms_amd.pipeline import BatchProblem, ModeSumProblem
from fastemriwaveforms_amd.summation import CubicSplineInterpolant, InterpolatedModeSum

YEAR = synthetic.YRSID_SI
F64, C128 = torch.float64, torch.complex128


# ------------------------------------------------------------------ the cases

def _sum_case(kind, **kw):
    c = dict(kind=kind, T=1.0, dt=10.0, L=120, K=3843, set="m_nonneg_30", phases="spline")
    c.update(kw)
    return c


def listed():
    return [
        # A short segment of a waveform with a polar mode set (k != 0), as a
        # quick-look or a test does: every launch and the host call count.
        dict(_sum_case("class", T=0.02, L=50, K=300, set="k1_20", phases="dopr",
                       precision="mixed16"), name="class_mixed16_short"),
        # The default call of the drop-in class (FP64, the reference's arithmetic)
        # on a month-long waveform with the strongest 500 modes.
        dict(_sum_case("class", T=0.1, L=100, K=500, precision="fp64"), name="class_fp64_month"),
        # The same default call on a year with the whole Schwarzschild mode set.
        dict(_sum_case("class", precision="fp64"), name="class_fp64_year"),
        # One step of a sampler on one year, all modes, mixed precision.
        dict(_sum_case("step", precision="mixed16"), name="step_mixed16_year"),
        # Two years at 5 s with the wide explicit +-m mode set (n up to 55).
        dict(_sum_case("step", T=2.0, dt=5.0, L=200, K=2000, set="m_all_55", precision="mixed16"),
             name="step_mixed16_2yr"),
        # The population call: 256 uneven waveforms (0.1-2 yr, 50-200 knots,
        # 50-3000 modes).
        dict(kind="batch", count=256, T_lo=0.1, T_hi=2.0, L_lo=50, L_hi=200, K_lo=50, K_hi=3000,
             sizes=1003, precision="mixed16", name="batch_mixed16_256"),
        # A Fisher-matrix step: waveform and knot gradients in FP64-class precision.
        dict(_sum_case("grad", precision="fact64", backward="fact64"), name="grad_fact64_year"),
        # The reference-arithmetic gradient on the month-long waveform.
        dict(_sum_case("grad", T=0.1, L=100, K=500, precision="fp64", backward="fp64"),
             name="grad_fp64_month"),
        # The frequency-domain waveform of one year, all modes.
        dict(kind="fd", T=1.0, dt=10.0, L=120, K=3843, set="m_nonneg_30", name="fd_year"),
        # AAK for one year with the LISA response.
        dict(kind="aak", T=1.0, dt=10.0, L=100, nmodes=30, mich=True, name="aak_year"),
        # Amplitudes of the whole mode set at a trajectory's knots.
        dict(kind="amp", modes=3843, nw=38, nu=48, points=120, name="amp_full_set"),
        # Spline build of the whole set's amplitude arrays and their values on a
        # finer grid (plots, resampling).
        dict(kind="spline", arrays=7686, L=120, points=1000, name="spline_full_set"),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _modes(rng, lo, hi):
    return int(round(_log(rng, lo, hi)))


def draw(rng):
    kind = rng.choice(["class", "class", "step", "step", "batch", "grad", "fd", "aak", "amp",
                       "spline"])
    L = rng.randint(20, 200)
    if kind in ("class", "step"):
        mode_set = rng.choice(["m_nonneg_30", "m_nonneg_30", "k1_20", "m_all_55"])
        prec = rng.choice(["fp64", "fp64", "mixed16", "fact64"] if kind == "class"
                          else ["mixed16", "mixed16", "fact64"])
        K = {"m_nonneg_30": _modes(rng, 20, 3843), "k1_20": _modes(rng, 20, 1476),
             "m_all_55": _modes(rng, 20, 2000)}[mode_set]
        if mode_set == "m_all_55" and prec == "fact64":
            prec = "mixed16"  # the FP64 tile of the wide set does not fit
        dt = rng.choice([5.0, 10.0, 15.0])
        hi = 1.0 if prec == "fp64" else 2.0
        return _sum_case(kind, T=round(_log(rng, 0.01, hi * dt / 15.0), 4), dt=dt, L=L, K=K,
                         set=mode_set, phases=rng.choice(["spline", "dopr"]), precision=prec)
    if kind == "batch":
        T_hi = round(rng.uniform(0.2, 2.0), 3)
        K_hi = rng.randint(300, 3000)
        return dict(kind="batch", count=_modes(rng, 3, 160), T_lo=round(T_hi * 0.05, 4), T_hi=T_hi,
                    L_lo=20, L_hi=L, K_lo=20, K_hi=K_hi, sizes=rng.randrange(1 << 30),
                    precision="mixed16")
    if kind == "grad":
        pair = rng.choice([("fact64", "fact64"), ("fact64", "fact64"), ("mixed16", "fact64"),
                           ("fp64", "fp64")])
        T = round(_log(rng, 0.01, 0.3 if pair[1] == "fp64" else 1.0), 4)
        return _sum_case("grad", T=T, L=L, K=_modes(rng, 20, 3843), precision=pair[0],
                         backward=pair[1])
    if kind == "fd":
        return dict(kind="fd", T=round(_log(rng, 0.02, 1.0), 4), dt=10.0, L=max(L, 30),
                    K=_modes(rng, 10, 3843), set="m_nonneg_30")
    if kind == "aak":
        return dict(kind="aak", T=round(_log(rng, 0.02, 1.0), 4), dt=rng.choice([10.0, 15.0]), L=L,
                    nmodes=rng.randint(4, 30), mich=rng.random() < 0.5)
    if kind == "amp":
        return dict(kind="amp", modes=_modes(rng, 10, 3843), nw=rng.randint(12, 38),
                    nu=rng.randint(12, 48), points=_modes(rng, 10, 200))
    return dict(kind="spline", arrays=_modes(rng, 3, 7686), L=L, points=_modes(rng, 10, 1000))


# ----------------------------------------------------------- inputs and calls

def _dev(x, dtype=None):
    t = torch.from_numpy(np.ascontiguousarray(x)).cuda()
    return t if dtype is None else t.to(dtype)


def _input(case, seed, chirp="smooth"):
    return synthetic.make_input(case["T"], case["dt"], case["L"], case["set"], case["K"], seed,
                                minus_m_ylm=case["set"] != "m_all_55", chirp=chirp,
                                phases=case.get("phases", "spline"))


def _knots(case, rng):
    """Knot times of one trajectory: ends and sorted uniform draws between them."""
    Ts = case["T"] * YEAR
    return np.concatenate([[0.0], np.sort(rng.uniform(0.0, 1.0, case["L"] - 2)) * Ts, [Ts]])


def _ylm_public(inp):
    """Y+ and Y- as the summation classes take them ((-1)^l not applied yet)."""
    y = inp.ylms.copy()
    y[inp.K:] *= (-1.0) ** inp.l
    return y


def _aak_knots(case, seed):
    rng = np.random.default_rng(seed)
    t = _knots(case, rng)
    tau = t / (case["T"] * YEAR)
    ph = synthetic.phase_phi(t, case["T"] * YEAR, "rising")
    e0, y0 = rng.uniform(0.2, 0.5), rng.uniform(0.5, 0.8)
    orbit = [12.0 - 4.0 * tau, e0 - 0.5 * e0 * tau ** 2, y0 + 0.05 * tau]
    phases = [ph, rng.uniform(0.95, 0.99) * ph, rng.uniform(0.8, 0.9) * ph]
    angles = rng.uniform(0.3, 2.5, 4)
    return t, np.stack(orbit + phases), angles, rng.uniform(0.2, 0.8)


def _amp_inputs(case, seed):
    rng = np.random.default_rng(seed)

    def grid(n):
        return np.concatenate([[0.0] * 4, np.sort(rng.uniform(0, 1, n - 8)), [1.0] * 4])

    tw, tu = grid(case["nw"]), grid(case["nu"])
    gen = torch.Generator("cuda").manual_seed(seed)
    coeff = torch.randn((case["modes"], 2, (case["nw"] - 4) * (case["nu"] - 4)), dtype=F64,
                        device="cuda", generator=gen)
    w, u = np.sort(rng.uniform(0, 1, case["points"])), rng.uniform(0, 1, case["points"])
    return _dev(tw), _dev(tu), coeff, _dev(w), _dev(u)


def _spline_inputs(case, seed):
    rng = np.random.default_rng(seed)
    t = np.concatenate([[0.0], np.sort(rng.uniform(0.0, 1.0, case["L"] - 2)), [1.0]])
    a = rng.normal(size=(4, case["arrays"]))
    y = a[0][:, None] + sum(0.3 * a[k][:, None] * t[None] ** k for k in (1, 2, 3))
    return _dev(t), _dev(y), _dev(rng.uniform(0.0, 1.0, case["points"]))


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case, kind = case, case["kind"]
    if kind == "class":
        inp = _input(case, seed)
        s.summ = InterpolatedModeSum(precision=case["precision"])
        t = _dev(inp.t)
        dense = _dev(inp.dense) if inp.dense is not None else _dense_of_cubic(
            _spline(t, _dev(inp.phase_knots.T)), t)
        s.args = (t, _dev(inp.teuk), _dev(_ylm_public(inp)), t, dense.permute(1, 2, 0).contiguous(),
                  inp.l, inp.m, inp.k, inp.n)
        s.kw = dict(T=inp.T_years, dt=inp.dt)
    elif kind == "step":
        s.prob = ModeSumProblem(_input(case, seed))
    elif kind == "batch":
        s.prob = BatchProblem(_batch_inputs(case, seed))
    elif kind == "grad":
        inp = _input(case, seed)
        s.eng = DifferentiableModeSum(inp.t, inp.m, inp.k, inp.n, inp.ylms, inp.dt, inp.num_pts,
                                      precision=case["precision"], backward=case["backward"])
        s.teuk = _dev(inp.teuk).requires_grad_(True)
        s.phase = _dev(inp.phase_knots).requires_grad_(True)
        s.weight = _cotangent(inp, seed)
    elif kind == "fd":
        inp = _input(case, seed, "rising")
        s.summ = FDInterpolatedModeSum(output_type="fd")
        t = _dev(inp.t)
        dense = _dense_of_cubic(_spline(t, _dev(inp.phase_knots.T)), t)
        s.args = (t, _dev(inp.teuk), _dev(_ylm_public(inp)), t, dense.permute(1, 2, 0).contiguous(),
                  inp.l, inp.m, inp.k, inp.n)
        s.kw = dict(T=inp.T_years, dt=inp.dt, frequencies=tuple(_dev(f) for f in inp.freqs))
    elif kind == "aak":
        t, knots, angles, spin = _aak_knots(case, seed)
        td = _dev(t)
        coef = _dense_of_cubic(_spline(td, _dev(knots.T)), td).permute(1, 2, 0).contiguous()
        s.summ = AAKSummation()
        s.args = (td, 1e6, spin, 1.0, 10.0, *(float(x) for x in angles), case["nmodes"], td, coef)
        s.kw = dict(mich=case["mich"], T=case["T"], dt=case["dt"])
    elif kind == "amp":
        tw, tu, coeff, s.w, s.u = _amp_inputs(case, seed)
        idx = np.arange(case["modes"])
        s.amp = AmpInterp2D(tw, tu, coeff, idx, idx, idx, idx)
    else:
        s.t, s.y, s.tnew = _spline_inputs(case, seed)
    return s


def _batch_inputs(case, seed):
    """Sizes from the case (every seed gives a batch of the same shape), values from the seed."""
    sizes, values = np.random.default_rng(case["sizes"]), np.random.default_rng(seed)
    out = []
    for _ in range(case["count"]):
        T = float(sizes.uniform(case["T_lo"], case["T_hi"]))
        L = int(sizes.integers(case["L_lo"], case["L_hi"] + 1))
        K = int(sizes.integers(case["K_lo"], case["K_hi"] + 1))
        out.append(synthetic.make_input(T, 10.0, L, "m_nonneg_30", K, int(values.integers(1 << 31))))
    return out


def _cotangent(inp, seed):
    """The loss's derivative with respect to the waveform: noise-like data."""
    gen = torch.Generator("cuda").manual_seed(seed)
    return torch.view_as_complex(torch.randn((inp.num_pts, 2), dtype=F64, device="cuda",
                                             generator=gen))


def run(s):
    kind = s.case["kind"]
    if kind in ("class", "fd", "aak"):
        return s.summ(*s.args, **s.kw)
    if kind in ("step", "batch"):
        return s.prob.run(s.case["precision"])
    if kind == "grad":
        h = s.eng(s.teuk, s.phase)
        gt, gp = torch.autograd.grad(h, (s.teuk, s.phase), s.weight)
        return {"waveform": h.detach(), "grad_amplitudes": gt, "grad_phases": gp}
    if kind == "amp":
        return s.amp(s.w, s.u)
    spl = CubicSplineInterpolant(s.t, s.y)
    return {"coefficients": spl.interp_array, "values": spl(s.tnew)}


# ------------------------------------------------------------- work of a pass

@functools.lru_cache(maxsize=None)
def _multiplicities(kind):
    ms = synthetic.mode_set(kind)
    cells = np.stack([*ms[1:]], axis=1)
    return np.unique(cells, axis=0, return_counts=True)[1], len(ms[0])


def _distinct(kind, K):
    """Expected number of distinct (m, k, n) among K random modes of a set."""
    mult, total = _multiplicities(kind)
    if K >= total:
        return float(len(mult))
    return float(np.sum(1.0 - (1.0 - K / total) ** mult))


def work(case):
    kind = case["kind"]
    if kind == "batch":
        n = case["count"]
        T, L, K = (0.5 * (case[a + "_lo"] + case[a + "_hi"]) for a in "TLK")
        N = n * T * YEAR / 10.0
        return {"bytes": 16 * N + n * 16 * L * K, "flops": 8 * _distinct("m_nonneg_30", K) * N}
    if kind in ("class", "step", "grad", "fd"):
        L, K = case["L"], case["K"]
        N = case["T"] * YEAR / case["dt"]
        cells = _distinct(case["set"], K)
        b = 16 * N + 16 * L * K + 44 * K + 100 * L
        if kind == "fd":
            ms = synthetic.mode_set(case["set"])
            # bins a mode sweeps: |m + 0.875 n| (1e-3 Hz to 2.5e-3 Hz) over 1 / T
            bins = np.minimum(np.abs(ms[1] + 0.875 * ms[-1]) * 1.5e-3 * case["T"] * YEAR, N)
            return {"bytes": b + 16 * N, "flops": 100 * cells * float(np.mean(bins))}
        if kind == "grad":  # waveform, its cotangent, two gradients
            return {"bytes": b + 16 * N + 16 * L * K, "flops": 24 * cells * N}
        return {"bytes": b, "flops": 8 * cells * N}
    if kind == "aak":
        N = case["T"] * YEAR / case["dt"]
        return {"bytes": 16 * N, "flops": 150 * case["nmodes"] * N}
    if kind == "amp":
        sets = 2 * case["modes"]
        return {"bytes": 8 * sets * ((case["nw"] - 4) * (case["nu"] - 4) + case["points"]),
                "flops": 32 * sets * case["points"]}
    M, L = case["arrays"], case["L"]
    return {"bytes": 8 * M * (5 * L + case["points"]), "flops": M * (30 * L + 6 * case["points"])}


# --------------------------------------- the same quantities in plain 64 bits

def _spline(t, y):
    """Not-a-knot cubic spline of the columns of y (L, M): coefficients of
    x = t - t_j in the pieces, (4, L - 1, M), from a dense solve for the slopes."""
    L = len(t)
    h = t[1:] - t[:-1]
    d = (y[1:] - y[:-1]) / h[:, None]
    A = torch.zeros((L, L), dtype=F64, device=t.device)
    i = torch.arange(1, L - 1, device=t.device)
    A[i, i - 1] = h[1:]
    A[i, i] = 2.0 * (h[1:] + h[:-1])
    A[i, i + 1] = h[:-1]
    rhs_mid = 3.0 * (h[1:, None] * d[:-1] + h[:-1, None] * d[1:])
    s0, s1 = h[0] + h[1], h[-1] + h[-2]
    A[0, 0], A[0, 1] = h[1], s0
    A[-1, -1], A[-1, -2] = h[-2], s1
    r0 = ((h[0] + 2.0 * s0) * h[1] * d[0] + h[0] ** 2 * d[1]) / s0
    r1 = ((h[-1] + 2.0 * s1) * h[-2] * d[-1] + h[-1] ** 2 * d[-2]) / s1
    s = torch.linalg.solve(A, torch.cat([r0[None], rhs_mid, r1[None]]))
    hh = h[:, None]
    return torch.stack([y[:-1], s[:-1], (3.0 * d - 2.0 * s[:-1] - s[1:]) / hh,
                        (s[:-1] + s[1:] - 2.0 * d) / hh ** 2])


def _dense_of_cubic(c, t):
    """Cubic pieces (4, L - 1, M) as dense-output coefficients (8, L - 1, M)."""
    h = (t[1:] - t[:-1])[:, None]
    c1, c2, c3 = c[1] * h, c[2] * h ** 2, c[3] * h ** 3
    delta = c1 + c2 + c3
    slope1 = c1 + 2.0 * c2 + 3.0 * c3
    r3 = c1 - delta
    zero = torch.zeros_like(delta)
    return torch.stack([c[0], delta, r3, delta - slope1 - r3, zero, zero, zero, zero])


def _dense_eval(r, s):
    """r: (8, 3) or (8, n, 3); s: (n,) -> phases (n, 3)."""
    s = s[:, None]
    q = 1.0 - s
    v = r[7]
    for k, x in ((6, s), (5, q), (4, s), (3, q), (2, s), (1, q), (0, s)):
        v = r[k] + x * v
    return v


class _Lattice:
    """Rows (signed (m, k)) and columns (n) of a mode set: h = sum_r u_r sum_n C v_n."""

    def __init__(self, inp):
        K = inp.K
        m, k, n = (np.asarray(x, np.int64) for x in (inp.m, inp.k, inp.n))
        keys = np.concatenate([np.stack([m, k], 1), np.stack([-m, -k], 1)])
        self.rows, r = np.unique(keys, axis=0, return_inverse=True)
        r = r.reshape(-1)
        self.n_max = int(np.abs(n).max())
        self.cols = np.arange(-self.n_max, self.n_max + 1)
        nc = len(self.cols)
        self.plus = _dev(r[:K] * nc + n + self.n_max)
        self.minus = _dev(r[K:] * nc + self.n_max - n)
        self.yp = _dev(inp.ylms[:K])
        self.ym = _dev(np.where(m != 0, inp.ylms[K:], 0.0))
        self.m, self.k = _dev(self.rows[:, 0]).to(F64), _dev(self.rows[:, 1]).to(F64)
        self.n = _dev(self.cols).to(F64)

    def waveform(self, a, x, ph):
        """a: (4, K) complex amplitude cubic, x: (n,), ph: (n, 3) -> (n,) complex."""
        R, nc = len(self.rows), len(self.cols)
        C = torch.zeros((4, R * nc), dtype=C128, device=a.device)
        C = C.index_add(1, self.plus, a * self.yp).index_add(1, self.minus, a.conj() * self.ym)
        v = torch.polar(torch.ones((), dtype=F64, device=x.device), -self.n * ph[:, 2:])
        u = torch.polar(torch.ones((), dtype=F64, device=x.device),
                        -(self.m * ph[:, :1] + self.k * ph[:, 1:2]))
        W = (v @ C.reshape(4 * R, nc).T).reshape(-1, 4, R)
        W = (W * u[:, None]).sum(-1)
        return W[:, 0] + x * (W[:, 1] + x * (W[:, 2] + x * W[:, 3]))


def _pieces(inp, t):
    """(interval, first sample, end) of the sample ranges between knots."""
    edges = np.clip(np.ceil(inp.t / inp.dt), 0, inp.num_pts).astype(np.int64)
    edges[0], edges[-1] = 0, inp.num_pts
    for j in range(inp.L - 1):
        for a in range(int(edges[j]), int(edges[j + 1]), 1 << 16):
            yield j, a, min(a + (1 << 16), int(edges[j + 1]))


def _exact_waveform(inp, out):
    t = _dev(inp.t)
    amp = _spline(t, torch.view_as_real(_dev(inp.teuk)).reshape(inp.L, -1))
    amp = torch.view_as_complex(amp.reshape(4, inp.L - 1, inp.K, 2).contiguous())
    dense = (_dev(inp.dense) if inp.dense is not None
             else _dense_of_cubic(_spline(t, _dev(inp.phase_knots.T)), t))
    lat = _Lattice(inp)
    for j, a, b in _pieces(inp, t):
        ts = torch.arange(a, b, device="cuda", dtype=F64) * inp.dt
        x = ts - float(inp.t[j])
        ph = _dense_eval(dense[:, j], x / float(inp.t[j + 1] - inp.t[j]))
        out[a:b] = lat.waveform(amp[:, j], x, ph)


def _exact_grad(case, seed):
    inp = _input(case, seed)
    t = _dev(inp.t)
    teuk = _dev(inp.teuk).requires_grad_(True)
    phase = _dev(inp.phase_knots).requires_grad_(True)
    g = _cotangent(inp, seed)
    amp = torch.view_as_complex(_spline(t, torch.view_as_real(teuk).reshape(inp.L, -1)).reshape(
        4, inp.L - 1, inp.K, 2).contiguous())
    dense = _dense_of_cubic(_spline(t, phase.T), t)
    a_leaf, p_leaf = amp.detach().requires_grad_(True), dense.detach().requires_grad_(True)
    lat = _Lattice(inp)
    h = torch.zeros(inp.num_pts, dtype=C128, device="cuda")
    ga, gp = torch.zeros_like(a_leaf), torch.zeros_like(p_leaf)
    for j, a, b in _pieces(inp, t):
        ts = torch.arange(a, b, device="cuda", dtype=F64) * inp.dt
        x = ts - float(inp.t[j])
        aj = a_leaf[:, j].detach().requires_grad_(True)
        pj = p_leaf[:, j].detach().requires_grad_(True)
        hj = lat.waveform(aj, x, _dense_eval(pj, x / float(inp.t[j + 1] - inp.t[j])))
        h[a:b] = hj.detach()
        da, dp = torch.autograd.grad(hj, (aj, pj), g[a:b])
        ga[:, j] += da
        gp[:, j] += dp
    gt, gk = torch.autograd.grad((amp, dense), (teuk, phase), (ga, gp))
    return {"waveform": h, "grad_amplitudes": gt, "grad_phases": gk}


def _bspline_basis(knots, x):
    """Cubic B-spline basis at the points x: (points, len(knots) - 4)."""
    nk = len(knots)
    span = torch.clamp(torch.searchsorted(knots, x, right=True) - 1, 3, nk - 5)
    B = torch.zeros((len(x), nk - 1), dtype=F64, device=x.device)
    B[torch.arange(len(x), device=x.device), span] = 1.0
    X = x[:, None]
    for p in range(1, 4):
        n = nk - 1 - p
        dl, dr = knots[p:p + n] - knots[:n], knots[p + 1:p + 1 + n] - knots[1:1 + n]
        left = torch.where(dl > 0, (X - knots[:n]) / torch.where(dl > 0, dl, 1.0), 0.0)
        right = torch.where(dr > 0, (knots[p + 1:p + 1 + n] - X) / torch.where(dr > 0, dr, 1.0), 0.0)
        B = left * B[:, :n] + right * B[:, 1:n + 1]
    return B


def exact(case, seed):
    kind = case["kind"]
    if kind in ("class", "step"):
        inp = _input(case, seed)
        out = torch.zeros(inp.num_pts, dtype=C128, device="cuda")
        _exact_waveform(inp, out)
        return out
    if kind == "batch":
        inputs = _batch_inputs(case, seed)
        out = torch.zeros(sum(x.num_pts for x in inputs), dtype=C128, device="cuda")
        at = 0
        for x in inputs:
            _exact_waveform(x, out[at:at + x.num_pts])
            at += x.num_pts
        return out
    if kind == "grad":
        return _exact_grad(case, seed)
    if kind == "amp":
        tw, tu, coeff, w, u = _amp_inputs(case, seed)
        grid = coeff.reshape(case["modes"] * 2, case["nw"] - 4, case["nu"] - 4)
        Bw, Bu = _bspline_basis(tw, w), _bspline_basis(tu, u)
        z = torch.stack([((grid @ Bu[p]) @ Bw[p]) for p in range(case["points"])])
        z = z.reshape(case["points"], case["modes"], 2).contiguous()
        return torch.view_as_complex(z)
    if kind == "spline":
        t, y, tnew = _spline_inputs(case, seed)
        c = _spline(t, y.T.contiguous())
        j = torch.clamp(torch.searchsorted(t, tnew, right=True) - 1, 0, case["L"] - 2)
        x = (tnew - t[j])[:, None]
        c = c[:, j]
        return {"coefficients": None,
                "values": (c[0] + x * (c[1] + x * (c[2] + x * c[3]))).T.contiguous()}
    # the stationary-phase sum and the AAK Bessel fits are defined by their own
    # truncated series, which plain torch has no independent value for
    return None

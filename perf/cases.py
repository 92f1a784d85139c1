"""Performance cases: the batch solves a user of this package has it do.

Each case is one call through the public entry points (``Solver.solve`` with
host inputs and host or device-resident results, ``solve_adjoint`` followed by
``backward``) on a batch of independent systems. The systems and options are
those of this repository's benchmark and tests; sizes run from a few dozen
systems, where a call is latency, to batches that fill the GPU several times,
with odd batch sizes among them.

``exact`` integrates the same inputs with two textbook schemes in 64-bit torch
(Gragg-Bulirsch-Stoer extrapolation for the smooth problems, extrapolated
linearly implicit Euler for the stiff ones) far below the tolerances the cases
ask for.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import cubie_amd as ca

F64, F32 = np.float64, np.float32


# ---------------------------------------------------------------------------
# Systems
# ---------------------------------------------------------------------------

# alpha_m and alpha_n have removable singularities at V = -40 / -55 mV; their
# first-order expansion stands in within 1e-3 mV of them.
HH_EQUATIONS = """
alpha_m = Piecewise((1 + (V + 40)/20, Abs(V + 40) < 1e-3), (0.1*(V + 40)/(1 - exp(-(V + 40)/10)), True))
beta_m = 4*exp(-(V + 65)/18)
alpha_h = 0.07*exp(-(V + 65)/20)
beta_h = 1/(1 + exp(-(V + 35)/10))
alpha_n = Piecewise((0.1 + (V + 55)/200, Abs(V + 55) < 1e-3), (0.01*(V + 55)/(1 - exp(-(V + 55)/10)), True))
beta_n = 0.125*exp(-(V + 65)/80)
dV = (I_ext - gNa*m**3*h*(V - ENa) - gK*n**4*(V - EK) - gL*(V - EL))/Cm
dm = alpha_m*(1 - m) - beta_m*m
dh = alpha_h*(1 - h) - beta_h*h
dn = alpha_n*(1 - n) - beta_n*n
"""
HH_STATES = {"V": -65.0, "m": 0.0529, "h": 0.5961, "n": 0.3177}
HH_G = {"gNa": 120.0, "gK": 36.0, "gL": 0.3}
HH_E = {"ENa": 50.0, "EK": -77.0, "EL": -54.387}
L96_N = 20


def _lorenz(precision):
    return ca.create_ODE_system(
        ["dx = sigma*(y - x)", "dy = x*(rho - z) - y", "dz = x*y - beta*z"],
        states={"x": 1.0, "y": 0.0, "z": 25.0},
        parameters={"sigma": 10.0, "rho": 28.0, "beta": 8.0 / 3.0},
        precision=precision, name="lorenz")


def _van_der_pol(precision):
    return ca.create_ODE_system(
        ["dx = y", "dy = mu*(1 - x**2)*y - x"], states={"x": 2.0, "y": 0.0},
        parameters={"mu": 1.0}, precision=precision, name="van_der_pol")


def _robertson(precision):
    return ca.create_ODE_system(
        ["dy1 = -k1*y1 + k3*y2*y3", "dy2 = k1*y1 - k2*y2**2 - k3*y2*y3", "dy3 = k2*y2**2"],
        states={"y1": 1.0, "y2": 0.0, "y3": 0.0},
        parameters={"k1": 0.04, "k2": 3e7, "k3": 1e4}, precision=precision, name="robertson")


def _hodgkin_huxley(precision, current):
    return ca.create_ODE_system(
        HH_EQUATIONS, states=HH_STATES, parameters=HH_G, constants=dict(HH_E, Cm=1.0),
        drivers={"I_ext": current, "dt": 0.5, "order": 1, "wrap": False},
        precision=precision, name="hodgkin_huxley")


def _hodgkin_huxley6(precision, current):
    return ca.create_ODE_system(
        HH_EQUATIONS, states=HH_STATES, parameters=dict(HH_G, **HH_E), constants={"Cm": 1.0},
        drivers={"I_ext": current, "dt": 0.5, "order": 1, "wrap": False},
        precision=precision, name="hodgkin_huxley6")


def _lorenz96(precision):
    n = L96_N
    return ca.create_ODE_system(
        [f"dx{i} = (x{(i + 1) % n} - x{(i - 2) % n})*x{(i - 1) % n} - x{i} + F" for i in range(n)],
        states={f"x{i}": 8.0 for i in range(n)}, parameters={"F": 8.0},
        precision=precision, name="lorenz96")


def _lotka_volterra(precision):
    return ca.create_ODE_system(
        ["du = a*u - b*u*v", "dv = d*u*v - g*v", "total = u + v", "ratio = u/v"],
        states={"u": 1.0, "v": 1.0}, parameters={"a": 1.5, "b": 1.0, "d": 1.0, "g": 3.0},
        observables=["total", "ratio"], precision=precision, name="lotka_volterra")


def _hh_current(seed, bias, swing):
    """1000 current samples 0.5 ms apart (FP32-representable, so that FP32 and
    FP64 kernels integrate the same problem)."""
    rng = np.random.default_rng(seed + 7)
    t = np.arange(1000) * 0.5
    noise = rng.normal(0.0, 2.0, 1000)
    return (bias + swing * np.sin(2.0 * np.pi * t / 50.0) + noise).astype(F32)


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------

# kind -> (system, precision, solver options). Spacings are binary fractions
# where the arithmetic is FP32 or the step fixed, so that step ends land on
# the output events.
SETUPS = {
    # interactive parameter scans and trajectory ensembles, explicit adaptive
    "lorenz": (_lorenz, F64, dict(
        algorithm="dormand-prince-54", atol=1e-8, rtol=1e-6, save_every=0.01,
        output_types=["state", "time"])),
    "lorenz_f32": (_lorenz, F32, dict(
        algorithm="dormand-prince-54", atol=1e-6, rtol=1e-5, save_every=1.0 / 64,
        output_types=["state", "time"])),
    # runs of very different cost, per-run tolerance and end time, final state
    "vdp": (_van_der_pol, F64, dict(
        algorithm="dormand-prince-54", atol=1e-10, rtol=1e-6, dt_min=1e-10, dt_max=1.0,
        output_types=["state"], kernel_mode="persistent")),
    # stiff kinetics on an explicit table of log-spaced save times
    "robertson_ros3p": (_robertson, F64, dict(
        algorithm="ros3p", atol=1e-10, rtol=1e-6, linear_correction_type="bicgstab",
        output_types=["state"])),
    "robertson_radau": (_robertson, F64, dict(
        algorithm="radau", atol=1e-10, rtol=1e-6, linear_correction_type="bicgstab",
        output_types=["state"])),
    # neuron batches driven by a sampled current, fixed steps, summaries only
    "hh": (_hodgkin_huxley, F64, dict(
        algorithm="l_stable_dirk_3", dt=2.0 ** -6, atol=1e-6, rtol=1e-6,
        linear_correction_type="bicgstab", summarise_every=12.5,
        sample_summaries_every=2.0 ** -4, summarise_variables=["V"],
        output_types=["mean", "max", "spike_count[0]"])),
    "hh_compensated": (_hodgkin_huxley, F32, dict(
        algorithm="l_stable_dirk_3", dt=2.0 ** -6, atol=1e-6, rtol=1e-6,
        linear_correction_type="bicgstab", summarise_every=12.5,
        sample_summaries_every=2.0 ** -4, summarise_variables=["V"],
        output_types=["mean", "max", "spike_count[0]"], run_order="sorted",
        kernel_mode="persistent", precision_mode="compensated")),
    # gradients of a fit to mean potentials: forward and backward
    "adjoint": (_hodgkin_huxley6, F64, dict(
        algorithm="dormand-prince-54", atol=1e-6, rtol=1e-6, summarise_every=12.5,
        sample_summaries_every=0.5, summarise_variables=["V"], output_types=["mean"])),
    "adjoint_ros3p": (_hodgkin_huxley6, F64, dict(
        algorithm="ros3p", atol=1e-6, rtol=1e-6, linear_correction_type="bicgstab",
        summarise_every=12.5, sample_summaries_every=0.5, summarise_variables=["V"],
        output_types=["mean"])),
    # more states than fit in registers
    "lorenz96": (_lorenz96, F64, dict(
        algorithm="dormand-prince-54", atol=1e-8, rtol=1e-6, save_every=0.05,
        output_types=["state"])),
    # fixed explicit steps in FP32, states and observables at every save
    "lotka": (_lotka_volterra, F32, dict(
        algorithm="rk4", dt=2.0 ** -7, save_every=2.0 ** -4,
        output_types=["state", "observables"])),
}

# kind -> ((smallest, largest batch), run lengths) of the drawn cases
RANGES = {
    "lorenz": ((2048, 131072), (0.5, 1.0, 1.5, 2.5)),
    "lorenz_f32": ((2048, 250000), (0.5, 1.0, 1.5, 2.5)),
    "vdp": ((4096, 131072), (10.0, 30.0, 100.0)),
    "robertson_ros3p": ((1024, 40000), (1e2, 1e3, 1e4)),
    "robertson_radau": ((1024, 40000), (1e2, 1e3)),
    "hh": ((1024, 100000), (12.5, 25.0, 50.0)),
    "hh_compensated": ((1024, 131072), (12.5, 25.0, 50.0)),
    "adjoint": ((512, 100000), (12.5, 25.0)),
    "adjoint_ros3p": ((512, 40000), (12.5, 25.0)),
    "lorenz96": ((512, 50000), (0.5, 1.0, 2.0)),
    "lotka": ((4096, 400000), (2.0, 4.0, 8.0)),
}


def listed():
    def case(name, kind, n, duration, host=False):
        return {"name": name, "kind": kind, "n": n, "duration": duration, "host": host}

    return [
        # a scan of a few dozen parameter sets from a notebook, results as
        # arrays: the smallest call, all latency
        case("lorenz_scan_64", "lorenz", 64, 1.0, host=True),
        # a trajectory ensemble whose saved rows are the bulk of the bytes
        case("lorenz_ensemble_f64", "lorenz", 131072, 2.5),
        # the same in single precision, at a batch size that divides nothing
        case("lorenz_ensemble_f32", "lorenz_f32", 250003, 2.5),
        # uneven work on the persistent queue
        case("vdp_uneven", "vdp", 131072, 100.0),
        # Rosenbrock and fully implicit stiff solves
        case("robertson_ros3p", "robertson_ros3p", 20001, 1e4),
        case("robertson_radau", "robertson_radau", 30000, 1e3),
        # implicit fixed-step neuron batches, FP64 and mixed precision
        case("hh_sdirk3_f64", "hh", 65600, 50.0),
        case("hh_sdirk3_compensated", "hh_compensated", 131072, 50.0),
        # gradients, explicit and Rosenbrock
        case("hh_adjoint_dopri5", "adjoint", 100000, 25.0),
        case("hh_adjoint_ros3p", "adjoint_ros3p", 40001, 25.0),
        # a 20-state system
        case("lorenz96_dopri5", "lorenz96", 50000, 2.0),
        # fixed steps with dense outputs and observables
        case("lotka_rk4_f32", "lotka", 400000, 8.0),
    ]


def draw(rng):
    """One case of the listed ranges: any kind, a batch size spread over the
    logarithm of its range (mostly no multiple of anything), a run length of
    the kind. Small explicit ensembles also come as host calls."""
    if rng.random() < 0.15:
        return {"kind": "lorenz", "n": int(round(math.exp(rng.uniform(0.0, math.log(2048.0))))),
                "duration": rng.choice(RANGES["lorenz"][1]), "host": True}
    kind = rng.choice(sorted(RANGES))
    (lo, hi), durations = RANGES[kind]
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return {"kind": kind, "n": n, "duration": rng.choice(durations), "host": False}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _inputs(case, seed):
    """Host inputs of a case: inits (states, n), params (parameters, n) and
    the per-run or driver arrays of its kind, in the case's precision."""
    kind, n = case["kind"], case["n"]
    precision = SETUPS[kind][1]
    rng = np.random.default_rng(seed)
    extra = {}
    if kind in ("lorenz", "lorenz_f32"):
        params = np.array([10.0, 28.0, 8.0 / 3.0])[:, None] * rng.uniform(0.9, 1.1, (3, n))
        inits = rng.uniform(-1, 1, (3, n)) + np.array([0.0, 0.0, 25.0])[:, None]
    elif kind == "vdp":
        params = np.exp(rng.uniform(math.log(0.1), math.log(1000.0), n))[None, :]
        inits = rng.uniform(-2.0, 2.0, (2, n))
        extra["rtol"] = np.exp(rng.uniform(math.log(1e-8), math.log(1e-4), n))
        extra["ends"] = rng.uniform(0.01, 1.0, n) * case["duration"]
    elif kind.startswith("robertson"):
        params = np.array([0.04, 3e7, 1e4])[:, None] * np.exp(
            rng.uniform(math.log(0.8), math.log(1.25), (3, n)))
        inits = np.tile(np.array([[1.0], [0.0], [0.0]]), (1, n))
    elif kind in ("hh", "hh_compensated"):
        params = np.array(list(HH_G.values()))[:, None] * rng.uniform(0.7, 1.3, (3, n))
        params = params.astype(F32)
        inits = np.tile(np.array(list(HH_STATES.values()), dtype=F32)[:, None], (1, n))
        extra["current"] = _hh_current(seed, 0.0, 10.0)
    elif kind.startswith("adjoint"):
        base = np.array(list(HH_G.values()) + list(HH_E.values()))[:, None]
        params = base * rng.uniform(0.9, 1.1, (6, n))
        inits = np.tile(np.array(list(HH_STATES.values()))[:, None], (1, n))
        inits[0] = rng.uniform(-70.0, -60.0, n)
        extra["target"] = rng.normal(-60.0, 2.0, n)
        # well above threshold: every neuron fires throughout, as in a fit to
        # recordings, and no gradient hangs on whether a spike happens
        extra["current"] = _hh_current(seed, 30.0, 5.0)
    elif kind == "lorenz96":
        params = rng.uniform(7.0, 9.0, (1, n))
        inits = 8.0 + rng.normal(0.0, 1.0, (L96_N, n))
    else:
        params = np.array([1.5, 1.0, 1.0, 3.0])[:, None] * rng.uniform(0.8, 1.2, (4, n))
        inits = rng.uniform(0.5, 2.0, (2, n))
    return inits.astype(precision), params.astype(precision), extra


def _save_table(duration):
    """200 log-spaced save times from 1e-5 up to the end."""
    table = np.logspace(-5.0, math.log10(duration), 200)
    table[-1] = duration
    return table


def _solver(case, current=None):
    factory, precision, options = SETUPS[case["kind"]]
    options = dict(options)
    if case["kind"].startswith("robertson"):
        options["save_times"] = _save_table(case["duration"])
    system = factory(precision) if current is None else factory(precision, current.astype(F64))
    return ca.Solver(system, **options)


def prepare(case, seed):
    """Inputs and the solver, its kernel compiled and loaded by a call on one
    run of the batch, as a program holds them before it starts calling."""
    inits, params, extra = _inputs(case, seed)
    solver = _solver(case, extra.get("current"))
    state = {"case": case, "solver": solver, "duration": case["duration"], "options": {}}
    if case["kind"].startswith("adjoint"):
        state["inits"] = torch.from_numpy(inits).cuda()
        state["params"] = torch.from_numpy(params).cuda()
        state["target"] = torch.from_numpy(extra["target"]).cuda()
        ca.solve_adjoint(solver, state["inits"][:, :1], state["params"][:, :1],
                         case["duration"])
        return state
    state["inits"], state["params"] = inits, params
    if "rtol" in extra:
        state["options"] = {"rtol_per_run": extra["rtol"], "duration_per_run": extra["ends"]}
    one = {k: v[:1] for k, v in state["options"].items()}
    solver.solve(inits[:, :1], params[:, :1], duration=case["duration"],
                 on_device=not case["host"], **one)
    return state


def run(state):
    """One solve (or one solve and its gradient)."""
    case, solver = state["case"], state["solver"]
    if case["kind"].startswith("adjoint"):
        inits = state["inits"].detach().requires_grad_()
        params = state["params"].detach().requires_grad_()
        _, means, status = ca.solve_adjoint(solver, inits, params, state["duration"])
        ((means - state["target"]) ** 2).sum().backward()
        return {"means": means.detach(), "grad_inits": inits.grad, "grad_params": params.grad,
                "status": status}
    res = solver.solve(state["inits"], state["params"], duration=state["duration"],
                       on_device=not case["host"], **state["options"])
    if case["kind"].startswith("hh"):
        return {"summaries": res.state_summaries, "status": res.status_codes}
    out = {"state": res.state, "status": res.status_codes}
    if case["kind"] == "lotka":
        out["observables"] = res.observables
    return out


# ---------------------------------------------------------------------------
# Work
# ---------------------------------------------------------------------------

# kind -> (attempted steps per unit of time, flops per attempted step): the
# solver's own step counts on these inputs, and the right-hand sides, stage
# sums, Newton and Krylov iterations of a step at one operation per add,
# multiply, divide or elementary function
STEPS = {
    "lorenz": (105.0, 302), "lorenz_f32": (68.0, 302), "vdp": (74.0, 200),
    "robertson_ros3p": (1.05, 2000), "robertson_radau": (1.29, 3200), "hh": (64.0, 3650),
    "hh_compensated": (64.0, 3650), "adjoint": (14.1, 3000), "adjoint_ros3p": (54.0, 4500),
    "lorenz96": (96.0, 1950), "lotka": (128.0, 65),
}


def _shapes(case):
    """Values in and out of one pass: (inputs per run, outputs per run,
    bytes per value)."""
    kind, d = case["kind"], case["duration"]
    opts = SETUPS[kind][2]
    size = 8 if SETUPS[kind][1] is F64 else 4
    rows = int(round(d / opts["save_every"])) + 1 if "save_every" in opts else 1
    if kind in ("lorenz", "lorenz_f32"):
        return 6, 4 * rows, size
    if kind == "vdp":
        return 5, 4, size
    if kind.startswith("robertson"):
        return 6, 3 * 201, size
    if kind.startswith("hh"):
        return 7, 3 * int(round(d / 12.5)), size
    if kind.startswith("adjoint"):
        return 10, int(round(d / 12.5)) + 10, size
    if kind == "lorenz96":
        return L96_N + 1, L96_N * rows, size
    return 6, 4 * rows, size


def work(case):
    n = case["n"]
    ins, outs, size = _shapes(case)
    per_time, flops = STEPS[case["kind"]]
    # per-run end times are uniform on (0, duration]
    span = case["duration"] * (0.505 if case["kind"] == "vdp" else 1.0)
    return {"bytes": n * ((ins + outs) * size + 4), "flops": n * span * per_time * flops}


# ---------------------------------------------------------------------------
# The same outputs in 64 bits, without the package
# ---------------------------------------------------------------------------

def _extrapolate(table, ratios):
    """Aitken-Neville on a column of approximations; ratios(j, k) is the
    divisor of T[j] - T[j-1] at level k. Returns the best value and the one
    of the order below it."""
    prev = list(table)
    best = below = prev[-1]
    for k in range(1, len(table)):
        nxt = []
        for j in range(k, len(table)):
            a, b = prev[j - k + 1], prev[j - k]
            nxt.append(a + (a - b) / ratios(j, k))
        below, best, prev = best, nxt[-1], nxt
    return best, below


_GBS = (2, 4, 6, 8, 10)


def _gbs(f, t, y, H):
    """One Gragg-Bulirsch-Stoer step of order 10 (modified midpoint with 2, 4,
    ..., 10 substeps, smoothed, extrapolated in h^2)."""
    f0 = f(t, y)
    table = []
    for m in _GBS:
        h = H / m
        z0, z1 = y, y + h * f0
        for i in range(1, m):
            z0, z1 = z1, z0 + 2.0 * h * f(t + i * h, z1)
        table.append(0.5 * (z1 + z0 + h * f(t + H, z1)))
    return _extrapolate(table, lambda j, k: (_GBS[j] / _GBS[j - k]) ** 2 - 1.0)[0]


_COLS = 8


def _seulex(f, solve, y, H):
    """One step of the linearly implicit Euler method with 1, 2, ..., 8
    substeps, extrapolated in h; solve(y, h, r) is (I - h J(y))^-1 r with the
    Jacobian at the step's start. H is per run. Returns the new state and the
    error estimate."""
    table = []
    for m in range(1, _COLS + 1):
        h = H / m
        z = y
        inv = solve(y, h)
        for _ in range(m):
            z = z + inv(h * f(z))
        table.append(z)
    best, below = _extrapolate(table, lambda j, k: (j + 1.0) / (j + 1.0 - k) - 1.0)
    return best, best - below


def _seulex_to(f, solve, y, length, H, rtol, atol):
    """Advance every run by its own ``length`` with adaptive steps; ``H`` is
    the step to start with. Returns the state and the step to go on with."""
    done = torch.zeros_like(length)
    while True:
        left = length - done
        if not bool((left > 0).any()):
            return y, H
        h = torch.minimum(H, left)
        new, err = _seulex(f, solve, y, h)
        scale = atol + rtol * torch.maximum(y.abs(), new.abs())
        e = ((err / scale) ** 2).mean(0).sqrt()
        e = torch.where(torch.isfinite(e), e, torch.full_like(e, 1e6))
        ok = e <= 1.0
        y = torch.where(ok, new, y)
        last = h >= left
        done = torch.where(ok, torch.where(last, length, done + h), done)
        grow = (0.8 * e.clamp(1e-12, 1e12) ** (-1.0 / _COLS)).clamp(0.1, 4.0)
        # a step cut short by the end says nothing against the longer one
        H = torch.where(ok & last, torch.maximum(H, h * grow), h * grow)


def _lorenz_rhs(p):
    def f(_t, y):
        x, v, z = y[0], y[1], y[2]
        return torch.stack((p[0] * (v - x), x * (p[1] - z) - v, x * v - p[2] * z))
    return f


def _lorenz96_rhs(p):
    def f(_t, y):
        return (torch.roll(y, -1, 0) - torch.roll(y, 2, 0)) * torch.roll(y, 1, 0) - y + p[0]
    return f


def _lotka_rhs(p):
    def f(_t, y):
        uv = y[0] * y[1]
        return torch.stack((p[0] * y[0] - p[1] * uv, p[2] * uv - p[3] * y[1]))
    return f


def _vdp_implicit(mu):
    def f(y):
        return torch.stack((y[1], mu * (1.0 - y[0] ** 2) * y[1] - y[0]))

    def solve(y, h):
        a = h * (-2.0 * mu * y[0] * y[1] - 1.0)
        d = 1.0 - h * mu * (1.0 - y[0] ** 2)
        det = d - h * a

        def inv(r):
            return torch.stack(((d * r[0] + h * r[1]) / det, (r[1] + a * r[0]) / det))
        return inv
    return f, solve


def _robertson_implicit(k):
    """The first two components; y3 = 1 - y1 - y2 by conservation of mass."""
    def f(y):
        y3 = 1.0 - y[0] - y[1]
        a, c = k[0] * y[0], k[2] * y[1] * y3
        return torch.stack((c - a, a - k[1] * y[1] ** 2 - c))

    def solve(y, h):
        y3 = 1.0 - y[0] - y[1]
        j11 = -k[0] - k[2] * y[1]
        j12 = k[2] * (y3 - y[1])
        m11, m12 = 1.0 - h * j11, -h * j12
        m21, m22 = h * j11, 1.0 + h * (2.0 * k[1] * y[1] + j12)
        det = m11 * m22 - m12 * m21

        def inv(r):
            return torch.stack(((m22 * r[0] - m12 * r[1]) / det, (m11 * r[1] - m21 * r[0]) / det))
        return inv
    return f, solve


def _ratio(x):
    """x / (1 - exp(-x / 10)) and its derivative, continued over x = 0."""
    near = x.abs() < 1e-3
    s = torch.where(near, torch.ones_like(x), x)
    q = -torch.expm1(-s / 10.0)
    v = torch.where(near, 10.0 + x / 2.0, s / q)
    d = torch.where(near, 0.5 + x / 60.0, (1.0 - v * (1.0 - q) / 10.0) / q)
    return v, d


def _hh_rhs(g, e, current, sensitivities):
    """Hodgkin-Huxley on rows (V, m, h, n) and, with ``sensitivities``, the
    derivatives of the four with respect to (V0, m0, h0, n0, gNa, gK, gL,
    ENa, EK, EL) as the ten rows that follow each: y is (4, 11, n) then."""
    def f(t, y):
        V, m, h, n = (y[i, 0] for i in range(4))
        i = min(int(t / 0.5), len(current) - 2)
        drive = current[i] + (current[i + 1] - current[i]) * (t / 0.5 - i)
        rm, rmd = _ratio(V + 40.0)
        rn, rnd = _ratio(V + 55.0)
        am, bm = 0.1 * rm, 4.0 * torch.exp(-(V + 65.0) / 18.0)
        ah, bh = 0.07 * torch.exp(-(V + 65.0) / 20.0), 1.0 / (1.0 + torch.exp(-(V + 35.0) / 10.0))
        an, bn = 0.01 * rn, 0.125 * torch.exp(-(V + 65.0) / 80.0)
        m2, n2 = m * m, n * n
        cNa, cK = m2 * m * h, n2 * n2
        vNa, vK, vL = V - e[0], V - e[1], V - e[2]
        rate = g[0] * cNa + g[1] * cK + g[2]
        out = torch.empty_like(y)
        out[0, 0] = drive - g[0] * cNa * vNa - g[1] * cK * vK - g[2] * vL
        out[1, 0] = am - (am + bm) * m
        out[2, 0] = ah - (ah + bh) * h
        out[3, 0] = an - (an + bn) * n
        if sensitivities:
            sV, sm, sh, sn = (y[i, 1:] for i in range(4))
            out[0, 1:] = (-rate * sV - (3.0 * g[0] * m2 * h * vNa) * sm - (g[0] * m2 * m * vNa) * sh
                          - (4.0 * g[1] * n2 * n * vK) * sn)
            out[0, 5] -= cNa * vNa
            out[0, 6] -= cK * vK
            out[0, 7] -= vL
            out[0, 8] += g[0] * cNa
            out[0, 9] += g[1] * cK
            out[0, 10] += g[2]
            dm = 0.1 * rmd * (1.0 - m) + bm / 18.0 * m
            dh = -ah / 20.0 * (1.0 - h) - bh * (1.0 - bh) / 10.0 * h
            dn = 0.01 * rnd * (1.0 - n) + bn / 80.0 * n
            out[1, 1:] = dm * sV - (am + bm) * sm
            out[2, 1:] = dh * sV - (ah + bh) * sh
            out[3, 1:] = dn * sV - (an + bn) * sn
        return out
    return f


def _exact_rows(f, y, rows, spacing, pieces):
    """States at 0, spacing, 2 spacing, ... with ``pieces`` steps each."""
    out = [y]
    H = spacing / pieces
    for r in range(rows - 1):
        for j in range(pieces):
            y = _gbs(f, r * spacing + j * H, y, H)
        out.append(y)
    return torch.stack(out)


def exact(case, seed):
    kind, duration = case["kind"], case["duration"]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    inits, params, extra = _inputs(case, seed)
    y = torch.from_numpy(inits.astype(F64)).to(dev)
    p = torch.from_numpy(params.astype(F64)).to(dev)
    n = case["n"]
    opts = SETUPS[kind][2]
    rows = int(round(duration / opts["save_every"])) + 1 if "save_every" in opts else 0
    if kind in ("lorenz", "lorenz_f32"):
        s = _exact_rows(_lorenz_rhs(p), y, rows, opts["save_every"], 1)
        t = (torch.arange(rows, device=dev, dtype=torch.float64) * opts["save_every"])
        return {"state": torch.cat((s, t[:, None, None].expand(rows, 1, n)), 1), "status": None}
    if kind == "lorenz96":
        return {"state": _exact_rows(_lorenz96_rhs(p), y, rows, opts["save_every"], 2),
                "status": None}
    if kind == "lotka":
        s = _exact_rows(_lotka_rhs(p), y, rows, opts["save_every"], 1)
        return {"state": s, "status": None,
                "observables": torch.stack((s[:, 0] + s[:, 1], s[:, 0] / s[:, 1]), 1)}
    if kind == "vdp":
        ends = torch.from_numpy(extra["ends"]).to(dev)
        f, solve = _vdp_implicit(p[0])
        last, _ = _seulex_to(f, solve, y, ends, 1e-3 / (1.0 + p[0]), 1e-10, 1e-12)
        return {"state": torch.stack((y, last)), "status": None}
    if kind.startswith("robertson"):
        f, solve = _robertson_implicit(p)
        z, out = y[:2], [y]
        H, at = torch.full((n,), 1e-6, device=dev, dtype=torch.float64), 0.0
        for t in _save_table(duration):
            z, H = _seulex_to(f, solve, z, torch.full_like(H, t - at), H, 1e-10, 1e-15)
            at = t
            out.append(torch.stack((z[0], z[1], 1.0 - z[0] - z[1])))
        return {"state": torch.stack(out), "status": None}
    current = extra["current"].astype(F64).tolist()
    window, sample = opts["summarise_every"], opts["sample_summaries_every"]
    per = int(round(window / sample))
    grads = kind.startswith("adjoint")
    width = 11 if grads else 1
    Y = torch.zeros((4, width, n), device=dev, dtype=torch.float64)
    Y[:, 0] = y
    e = p[3:] if grads else torch.tensor(list(HH_E.values()), device=dev, dtype=torch.float64)
    if grads:
        for i in range(4):
            Y[i, 1 + i] = 1.0
    f = _hh_rhs(p, e, current, grads)
    # at most 1/16 ms a step: the fastest rate near a spike's peak is ~50 / ms
    pieces = max(1, int(round(sample / 0.0625)))
    prev, summaries, grad = None, [], 0.0
    for w in range(int(round(duration / window))):
        total, top = 0.0, torch.full((n,), -math.inf, device=dev, dtype=torch.float64)
        spikes = torch.zeros(n, device=dev, dtype=torch.float64)
        for k in range(per):
            for j in range(pieces):
                Y = _gbs(f, (w * per + k) * sample + j * sample / pieces, Y, sample / pieces)
            V = Y[0, 0]
            total, top = total + Y[0], torch.maximum(top, V)
            if prev is not None:
                spikes += ((prev < 0.0) & (V >= 0.0)).double()
            prev = V
        mean = total / per
        if grads:
            miss = mean[0] - torch.from_numpy(extra["target"]).to(dev)
            grad = grad + 2.0 * miss * mean[1:]
            summaries.append(mean[:1])
        else:
            summaries.append(torch.stack((mean[0], top, spikes)))
    if grads:
        return {"means": torch.stack(summaries), "grad_inits": grad[:4], "grad_params": grad[4:],
                "status": None}
    return {"summaries": torch.stack(summaries), "status": None}

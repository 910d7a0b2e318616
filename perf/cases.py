"""The framework's work as its users meet it: what its running time is quoted on.

A case is one call (or the few calls of one pass) of a user's program through the public
entry points of ``heyoka_amd``, described by plain values:

- ``system``: the equations integrated. ``pendulum`` and ``fdp`` (the forced, damped pendulum)
  are the small systems of the tutorials, ``cr3bp`` the planar restricted three-body problem
  with its mass ratio as a runtime parameter, ``nbody6`` the six-body problem of the ensemble
  benchmark, ``j2var`` the J2 problem with its first-order variational equations;
- ``call``: ``until`` (``propagate_until`` of one batch), ``grid`` (``propagate_grid``), ``step``
  (one ``step`` that keeps the Taylor coefficients), ``event`` (``propagate_until`` that stops
  every instance at a terminal event), ``ensemble`` (``ensemble_propagate_until_batch`` over a
  Python generator) and ``cfunc`` (a compiled function at many points);
- ``n``: instances (``members`` of them for an ensemble: ``n`` per member);
- ``t``: the time integrated over (negative: backwards), ``points`` the times of a grid.

Every integration starts from a state that the program has in host memory and writes into the
integrator, as a program with new initial conditions does, and ends with the state back in host
memory. The motion is regular over the horizons used, so that results can be compared: the
three-body instances librate about L4 and L5, and the six bodies stay clear of the collisions
that would make their positions depend on the last bit.
"""

import math

import numpy as np
import torch

import heyoka_amd as hy
from heyoka_amd import workloads

EPS = float(np.finfo(np.float64).eps)


# ---- the cases -----------------------------------------------------------------------------
def listed():
    return [
        # The smallest call: the tutorials' four pendulums. Latency of one wavefront's steps,
        # of the launches and of the host's calls.
        {"name": "pendulum_4", "system": "pendulum", "call": "until", "n": 4, "t": 100.0, "ha": False},
        # The tutorials' dense output: a few trajectories sampled at many times, to plot them.
        {"name": "fdp_4_grid_500", "system": "fdp", "call": "grid", "n": 4, "t": 20.0, "points": 500},
        # A few hundred orbits taken back in time with compensated summation (high_accuracy).
        {"name": "cr3bp_200_back_ha", "system": "cr3bp", "call": "until", "n": 200, "t": -50.0, "ha": True},
        # The largest low-dimensional ensemble: horizons spread over two decades, so that
        # instances end at different times.
        {"name": "cr3bp_131072_ragged", "system": "cr3bp", "call": "until", "n": 131072, "t": 100.0, "ragged": True,
         "ha": False},
        # Sampled trajectories of a medium ensemble (a scatter plot per time, a fit).
        {"name": "cr3bp_5001_grid_100", "system": "cr3bp", "call": "grid", "n": 5001, "t": 20.0, "points": 100},
        # A surface of section: every instance stops at its first crossing of x = 1/2 - mu.
        {"name": "cr3bp_32768_section", "system": "cr3bp", "call": "event", "n": 32768, "t": 20.0},
        # One step with its Taylor coefficients, which a program then reads (dense output by hand).
        {"name": "cr3bp_20000_step_tc", "system": "cr3bp", "call": "step", "n": 20000},
        # The ensemble benchmark: 65,536 six-body systems, a slice of ten time units.
        {"name": "nbody6_65536", "system": "nbody6", "call": "until", "n": 65536, "t": 10.0, "ha": False},
        # A Monte-Carlo study through the ensemble function: eight members of 97 six-body systems
        # each, a size that fills a part of the card only.
        {"name": "nbody6_ensemble_8x97", "system": "nbody6", "call": "ensemble", "n": 97, "members": 8, "t": 10.0},
        # State transition matrices of an ensemble of satellites (42 equations), two periods.
        {"name": "j2var_32768", "system": "j2var", "call": "until", "n": 32768, "t": 17.5, "ha": False},
        # The same for a constellation's few hundred satellites.
        {"name": "j2var_301", "system": "j2var", "call": "until", "n": 301, "t": 35.0, "ha": False},
        # A diagnostic over stored states: the energy of 100,000 six-body states.
        {"name": "nbody6_energy_100000", "system": "nbody6", "call": "cfunc", "n": 100000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["small_until", "cr3bp_until", "cr3bp_until", "nbody6_until", "nbody6_until", "j2var_until",
                       "fdp_grid", "cr3bp_grid", "nbody6_grid", "event", "step", "ensemble", "cfunc"])
    if kind == "small_until":
        return {"system": rng.choice(["pendulum", "fdp"]), "call": "until", "n": _log_int(rng, 1, 20000),
                "t": rng.uniform(5.0, 20.0), "ha": rng.random() < 0.25}
    if kind == "cr3bp_until":
        return {"system": "cr3bp", "call": "until", "n": _log_int(rng, 1, 120000),
                "t": rng.choice([-1.0, 1.0]) * rng.uniform(10.0, 100.0), "ragged": rng.random() < 0.5,
                "ha": rng.random() < 0.25}
    if kind == "nbody6_until":
        return {"system": "nbody6", "call": "until", "n": _log_int(rng, 1, 60000), "t": rng.uniform(2.0, 10.0),
                "ragged": rng.random() < 0.3, "ha": rng.random() < 0.15}
    if kind == "j2var_until":
        return {"system": "j2var", "call": "until", "n": _log_int(rng, 1, 30000), "t": rng.uniform(5.0, 17.5),
                "ragged": rng.random() < 0.3, "ha": rng.random() < 0.15}
    if kind == "fdp_grid":
        return {"system": "fdp", "call": "grid", "n": _log_int(rng, 1, 5000), "t": rng.uniform(5.0, 20.0),
                "points": rng.randint(20, 600)}
    if kind == "cr3bp_grid":
        return {"system": "cr3bp", "call": "grid", "n": _log_int(rng, 1, 20000), "t": rng.uniform(5.0, 50.0),
                "points": rng.randint(10, 150)}
    if kind == "nbody6_grid":
        return {"system": "nbody6", "call": "grid", "n": _log_int(rng, 1, 4000), "t": rng.uniform(2.0, 8.0),
                "points": rng.randint(10, 60)}
    if kind == "event":
        return {"system": "cr3bp", "call": "event", "n": _log_int(rng, 1, 60000), "t": rng.uniform(5.0, 30.0)}
    if kind == "step":
        return {"system": rng.choice(["pendulum", "cr3bp"]), "call": "step", "n": _log_int(rng, 1, 60000)}
    if kind == "ensemble":
        return {"system": "nbody6", "call": "ensemble", "n": _log_int(rng, 1, 1000), "members": rng.randint(1, 16),
                "t": rng.uniform(2.0, 10.0)}
    return {"system": "nbody6", "call": "cfunc", "n": _log_int(rng, 1, 200000)}


# ---- inputs --------------------------------------------------------------------------------
_FDP_NAMES = ("x", "v")


def _equations(system):
    if system == "pendulum":
        return hy.model.pendulum(), EPS
    if system == "fdp":
        x, v = hy.make_vars(*_FDP_NAMES)
        return [(x, v), (v, hy.cos(hy.time) - hy.par[0] * v - hy.sin(x))], EPS
    if system == "cr3bp":
        return hy.model.cr3bp_planar(), 1e-15
    if system == "nbody6":
        return hy.model.nbody(6, masses=list(workloads.nbody6_base()[0])), 1e-15
    return workloads.j2var(1).sys, 1e-15


def _inputs(case, seed):
    """Host arrays of one set of inputs: state [dim, N], parameters [n_par, N] (or None) and the
    times integrated to [N]."""
    n = case["n"] * case.get("members", 1)
    rng = np.random.default_rng(seed)
    pars = None
    if case["system"] == "pendulum":
        st = np.stack([rng.uniform(-1.0, 1.0, n), rng.uniform(-0.5, 0.5, n)])
    elif case["system"] == "fdp":
        st = np.stack([rng.uniform(-1.0, 1.0, n), rng.uniform(-0.5, 0.5, n)])
        pars = rng.uniform(0.05, 0.2, (1, n))
    elif case["system"] == "cr3bp":
        mu = rng.uniform(0.004, 0.012, n)
        sign = np.where(np.arange(n) % 2 == 0, 1.0, -1.0)
        st = np.stack([0.5 - mu, sign * math.sqrt(3.0) / 2, np.zeros(n), np.zeros(n)])
        st = st + rng.uniform(-0.005, 0.005, (4, n))
        pars = mu[None, :]
    elif case["system"] == "nbody6":
        st = workloads.nbody6(n, seed=seed).state
    else:
        st = workloads.j2var(n, seed=seed).state
    tf = np.full(n, float(case.get("t", 0.0)))
    if case.get("ragged"):
        tf = tf * 10.0 ** -rng.uniform(0.0, 2.0, n)
    return np.ascontiguousarray(st), pars, tf


def _names(system):
    if system == "nbody6":
        return [f"{q}_{i}" for i in range(6) for q in ("x", "y", "z", "vx", "vy", "vz")]
    return ["x", "y", "vx", "vy"]


def prepare(case, seed):
    st, pars, tf = _inputs(case, seed)
    state = {"case": case, "st": st, "pars": pars, "tf": tf}
    if case["call"] == "cfunc":
        masses = list(workloads.nbody6_base()[0])
        state["cf"] = hy.cfunc([hy.model.nbody_energy(6, masses=masses)], list(hy.make_vars(*_names("nbody6"))))
        return state
    eqs, tol = _equations(case["system"])
    kw = {"tol": tol}
    if pars is not None:
        kw["pars"] = pars[:, :case["n"]]
    if case.get("ha"):
        kw["high_accuracy"] = True
    if case["call"] == "event":
        x = hy.make_vars(*_names("cr3bp"))[0]
        kw["t_events"] = [hy.t_event_batch(x - 0.5 + hy.par[0], direction=hy.event_direction.positive)]
    if case["call"] == "grid":
        state["grid"] = np.ascontiguousarray(np.linspace(0.0, 1.0, case["points"])[:, None] * tf)
    state["ta"] = hy.taylor_adaptive_batch(eqs, st[:, :case["n"]], **kw)
    return state


# ---- one pass --------------------------------------------------------------------------------
def run(state):
    case = state["case"]
    call = case["call"]
    if call == "cfunc":
        return state["cf"](state["st"])
    ta = state["ta"]
    if call == "ensemble":
        n, st = case["n"], state["st"]

        def gen(member, i):
            member.state[:] = st[:, i * n:(i + 1) * n]
            return member

        ret = hy.ensemble_propagate_until_batch(ta, case["t"], case["members"], gen)
        return [r[0].state for r in ret]
    ta.state[:] = state["st"]
    ta.set_time(0.0)
    if call == "step":
        ta.step(write_tc=True)
        return {"state": ta.state, "time": ta.time, "h": ta.last_h, "tc": ta.tc}
    if call == "grid":
        return {"out": ta.propagate_grid(state["grid"])[1], "state": ta.state}
    if call == "event":
        ta.reset_cooldowns()
        ta.propagate_until(state["tf"])
        return {"state": ta.state, "time": ta.time}
    ta.propagate_until(state["tf"])
    return {"state": ta.state, "time": ta.time}


# ---- the work of a pass -----------------------------------------------------------------------
# Per system: floating-point operations of one Taylor step (an addition and a multiplication count
# one each), steps per unit of time, equations and parameters.
_STEP = {"pendulum": (963, 2.8, 2, 0), "fdp": (1822, 4.0, 2, 1), "cr3bp": (3619, 1.4, 4, 1),
         "nbody6": (39333, 34.2, 36, 0), "j2var": (43936, 2.15, 42, 0)}


def work(case):
    fl, rate, dim, npar = _STEP[case["system"]]
    n = case["n"] * case.get("members", 1)
    if case["call"] == "cfunc":
        return {"bytes": 8 * n * (dim + 1), "flops": n * (15 * 10 + 6 * 7)}
    steps = rate * abs(case.get("t", 0.0))
    if case.get("ragged"):
        steps *= (1.0 - 1e-2) / math.log(100.0)
    if case["call"] == "step":
        order = 20 if case["system"] == "pendulum" else 19
        return {"bytes": 8 * n * (2 * dim + npar + 3 + dim * (order + 1)), "flops": n * fl}
    if case["call"] == "event":
        steps = min(steps, 5.0)
    b = 8 * n * (2 * dim + npar + 3)
    if case["call"] == "grid":
        b += 8 * n * case["points"] * (dim + 1)
        return {"bytes": b, "flops": n * (steps * fl + case["points"] * 40 * dim)}
    return {"bytes": b, "flops": n * steps * fl}


# ---- the same outputs from a plain integrator -----------------------------------------------------
# Gragg's modified midpoint rule with Richardson extrapolation in the square of the step (Bulirsch and
# Stoer; Hairer, Norsett and Wanner, "Solving Ordinary Differential Equations I", II.9).
def _gbs_step(f, t, y, H, stages):
    rows = []
    for j in range(1, stages + 1):
        m = 2 * j
        h = H / m
        z0 = y
        z1 = y + h * f(t, y)
        for q in range(1, m):
            z0, z1 = z1, z0 + 2 * h * f(t + q * h, z1)
        cur = [0.5 * (z0 + z1 + h * f(t + H, z1))]
        for i in range(1, j):
            r = (j / (j - i)) ** 2 - 1.0
            cur.append(cur[i - 1] + (cur[i - 1] - rows[j - 2][i - 1]) / r)
        rows.append(cur)
    return rows[-1][-1]


def _rhs(system, pars):
    """(f(t, y), macro step size(y)) over y [dim, N]."""
    if system == "pendulum":
        return (lambda t, y: torch.stack([y[1], -torch.sin(y[0])])), (lambda y: 0.4)
    if system == "fdp":
        return (lambda t, y: torch.stack([y[1], torch.cos(t) - pars[0] * y[1] - torch.sin(y[0])])), (lambda y: 0.25)
    if system == "cr3bp":
        mu = pars[0]
        om = 1.0 - mu

        def f(t, s):
            x, y, vx, vy = s
            x1, x2, yy = x + mu, x - om, y * y
            a, b = om * (x1 * x1 + yy) ** -1.5, mu * (x2 * x2 + yy) ** -1.5
            c = 1.0 - a - b
            return torch.stack([vx, vy, 2.0 * vy + x - a * x1 - b * x2, c * y - 2.0 * vx])

        return f, (lambda y: 0.5)
    if system == "nbody6":
        m = workloads.nbody6_base()[0]
        ii, jj = np.triu_indices(6, 1)
        # Per pair, the weights with which its attraction enters each body's acceleration.
        w = np.zeros((6, 15))
        w[ii, np.arange(15)] = m[jj]
        w[jj, np.arange(15)] = -m[ii]
        dev = pars
        w = torch.as_tensor(w, device=dev)
        ii, jj = torch.as_tensor(ii, device=dev), torch.as_tensor(jj, device=dev)
        mm = torch.as_tensor(m, device=dev)

        def f(t, y):
            s = y.view(6, 6, -1)
            d = s[jj, :3] - s[ii, :3]
            d = d * ((d * d).sum(1, keepdim=True) ** -1.5)
            acc = (w @ d.reshape(15, -1)).view(6, 3, -1)
            return torch.cat([s[:, 3:], acc], 1).view(36, -1)

        def size(y):
            s = y.view(6, 6, -1)
            d = s[jj, :3] - s[ii, :3]
            r2 = (d * d).sum(1)
            return float((0.25 * torch.sqrt(r2 ** 1.5 / (mm[ii] + mm[jj])[:, None])).min())

        return f, size

    j2c = 1.5 * 1.0826e-3

    def f(t, y):
        p = y[:3]
        r2 = (p * p).sum(0)
        r3, i2 = r2 ** -1.5, 1.0 / r2
        zz = p[2] * p[2] * i2
        fxy = -r3 * (1.0 + j2c * i2 * (1.0 - 5.0 * zz))
        fz = -r3 * (1.0 + j2c * i2 * (3.0 - 5.0 * zz))
        ff = torch.stack([fxy, fxy, fz])
        # d(ff_i p_i)/dp_j = ff_i [i = j] + p_i d(ff_i)/dp_j.
        c = torch.tensor([1.0, 1.0, 3.0], dtype=y.dtype, device=y.device)[:, None, None]
        ez = torch.tensor([0.0, 0.0, 1.0], dtype=y.dtype, device=y.device)[None, :, None]
        g = (3.0 * r3 * i2 * p)[None] + j2c * (r3 * i2 * i2 * p)[None] * (5.0 * c - 35.0 * zz) \
            + j2c * ez * (10.0 * r3 * i2 * i2 * p[2])
        jac = p[:, None] * g
        jac = jac + torch.diag_embed(ff.T).permute(1, 2, 0)
        var = y[6:].view(6, 6, -1)
        dv = (jac[:, :, None] * var[None, :3]).sum(1)
        return torch.cat([y[3:6], ff * p, var[3:].reshape(18, -1), dv.reshape(18, -1)])

    return f, (lambda y: 0.24)


def _integrate(system, st, pars, tf, times):
    """States at the fractions `times` (ascending, in [0, 1]) of every instance's own horizon tf."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    y = torch.as_tensor(st, dtype=torch.float64, device=dev)
    tf = torch.as_tensor(tf, dtype=torch.float64, device=dev)
    p = None if pars is None else torch.as_tensor(pars, dtype=torch.float64, device=dev)
    f, size = _rhs(system, dev if system == "nbody6" else p)
    # In the fraction s of each instance's horizon: dy/ds = tf f(tf s, y).
    g = lambda s, v: tf * f(tf * s, v)  # noqa: E731
    span = float(tf.abs().max())
    s, out = 0.0, []
    for end in times:
        while s < end:
            H = size(y) / span
            k = max(1, math.ceil((end - s) / H - 1e-9))
            H = end - s if k == 1 else (end - s) / k
            y = _gbs_step(g, s, y, H, 7)
            s = end if k == 1 else s + H
        out.append(y.cpu().numpy())
    return out


def exact(case, seed):
    st, pars, tf = _inputs(case, seed)
    call = case["call"]
    if call == "cfunc":
        m = workloads.nbody6_base()[0]
        s = st.reshape(6, 6, -1)
        e = 0.5 * (m[:, None] * (s[:, 3:] ** 2).sum(1)).sum(0)
        for i in range(6):
            for j in range(i + 1, 6):
                e = e - m[i] * m[j] / np.sqrt(((s[j, :3] - s[i, :3]) ** 2).sum(0))
        return e[None]
    if call in ("step", "event"):
        return None  # the step's size and the event's time are the integrator's own
    if call == "grid":
        out = _integrate(case["system"], st, pars, tf, np.linspace(0.0, 1.0, case["points"]))
        return {"out": np.stack(out), "state": out[-1]}
    end = _integrate(case["system"], st, pars, tf, [1.0])[0]
    if call == "ensemble":
        return [end[:, i * case["n"]:(i + 1) * case["n"]] for i in range(case["members"])]
    return {"state": end, "time": tf}

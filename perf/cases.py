"""The work a user of this package has it do, as cases that can be timed and compared.

``listed()`` names them, ``draw(rng)`` gives more of the same ranges,
``prepare(case, seed)`` builds what a program has in hand before the call,
``run(state)`` is one pass through the public entry points, ``work(case)`` the
bytes and operations a pass cannot do without, ``tolerance(case)`` how far
another correct implementation may be from it and ``exact(case, seed)`` the
result in plain torch float64 where one can be written down.

Kinds:

operators  the single operators of one level, called on their own (gradient
           checks, Newton-Krylov drivers, the reference's jvp_test and
           adjoint_test scripts): residual, linearised operator, transpose
sweeps     smoothing passes of one level, forward then adjoint, FP64
glide      GlideStep, forward and backward, in the FP64 form (the drop-in
           default) with a fixed number of V-cycles
forward    one mixed-precision implicit step from rest to a tolerance
rollout    the multi-step adjoint inversion (mixed form): loss and gradients
thermal    one thermal step of the enthalpy columns
thermal_adjoint  the adjoint of a thermal step with its input gradients
coupled    coupled momentum + enthalpy steps with their adjoint (mixed form)
ensemble   independent glaciers of uneven sizes stepped together
"""
from __future__ import annotations

import math

import numpy as np
import torch

from glide_amd import IceDynamics, ThermalModel
from glide_amd.coupled import CoupledStep
from glide_amd.ensemble import Ensemble, ensemble_sizes, valley_glacier
from glide_amd.grid import Grid
from glide_amd.inversion import misfit, rollout
from glide_amd.synthetic import dome_problem, gaussian_random_field, install, thermal_forcing
from glide_amd.torch import GlideStep, ThermalStep

SEC_PER_YR = 365.25 * 86400.0
DEV = "cuda"


def listed():
    return [
        # gradient checks on a small ragged grid with the Weertman law: launches and latency
        {"name": "operators_66x130", "kind": "operators", "ny": 66, "nx": 130, "m": 1.0 / 3.0},
        # the same operators at continental size: memory traffic
        {"name": "operators_1536x2048", "kind": "operators", "ny": 1536, "nx": 2048, "m": 1.0},
        # smoothing passes on one odd-sized level, as hooks and hand-written cycles call them
        {"name": "sweeps_193x161", "kind": "sweeps", "ny": 193, "nx": 161, "passes": 8, "multicolour": False},
        # the drop-in FP64 step with its gradients: the smallest hierarchy in use ...
        {"name": "glide_fp64_64", "kind": "glide", "n": 64, "levels": 4, "cycles": 3},
        # ... and the side length of the reference's adjoint and JVP scripts
        {"name": "glide_fp64_224", "kind": "glide", "n": 224, "levels": 5, "cycles": 3},
        # a spin-up step at continental size with a grounding line
        {"name": "forward_mixed_2048", "kind": "forward", "n": 2048, "levels": 7},
        # basal-friction inversion: loss and gradient over a few steps, one checkpointed segment
        {"name": "rollout_mixed_256", "kind": "rollout", "n": 256, "levels": 5, "steps": 2},
        # a thermal step with the default stopping test on a small ragged map
        {"name": "thermal_40x56x21", "kind": "thermal", "ny": 40, "nx": 56, "nz": 21, "rtol": 1e-5},
        # the thermal step of the 512 x 512 coupled workload
        {"name": "thermal_512x512x41", "kind": "thermal", "ny": 512, "nx": 512, "nz": 41, "rtol": 1e-8},
        # its adjoint, as the coupled adjoint calls it
        {"name": "thermal_adjoint_512x512x41", "kind": "thermal_adjoint", "ny": 512, "nx": 512, "nz": 41},
        # the benchmark's coupled step, two in a row: one from rest, one warm
        {"name": "coupled_mixed_512", "kind": "coupled", "n": 512, "levels": 5, "nz": 41, "steps": 2},
        # a mountain range of glaciers of uneven sizes, one batched step
        {"name": "ensemble_48", "kind": "ensemble", "domains": 48, "lo": 48, "hi": 384},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _square(rng, lo, hi):
    """A side length that halves exactly, odd multiples among them, and its level count."""
    n = _log_int(rng, lo, hi)
    levels = max(3, min(7, int(math.log2(n / 12.0)) + 1))
    f = 2 ** (levels - 1)
    return max(2, round(n / f)) * f, levels


def draw(rng):
    kind = rng.choice(["operators", "operators", "sweeps", "glide", "forward", "rollout", "thermal", "thermal",
                       "thermal_adjoint", "coupled", "ensemble"])
    if kind == "operators":
        return {"kind": kind, "ny": _log_int(rng, 24, 1600), "nx": _log_int(rng, 24, 1900),
                "m": rng.choice([1.0, 1.0, 1.0 / 3.0])}
    if kind == "sweeps":
        return {"kind": kind, "ny": _log_int(rng, 24, 400), "nx": _log_int(rng, 24, 400),
                "passes": rng.randint(3, 12), "multicolour": rng.random() < 0.5}
    if kind == "glide":
        n, levels = _square(rng, 32, 320)
        return {"kind": kind, "n": n, "levels": levels, "cycles": rng.randint(1, 3)}
    if kind == "forward":
        n, levels = _square(rng, 64, 1600)
        return {"kind": kind, "n": n, "levels": levels}
    if kind == "rollout":
        n, levels = _square(rng, 64, 448)
        return {"kind": kind, "n": n, "levels": levels, "steps": rng.randint(1, 3)}
    if kind in ("thermal", "thermal_adjoint"):
        c = {"kind": kind, "ny": _log_int(rng, 16, 512), "nx": _log_int(rng, 16, 512), "nz": rng.randint(9, 64)}
        if kind == "thermal":
            c["rtol"] = rng.choice([1e-5, 1e-8])
        return c
    if kind == "coupled":
        n, levels = _square(rng, 64, 448)
        return {"kind": kind, "n": n, "levels": levels, "nz": rng.choice([11, 21, 31, 41]), "steps": rng.randint(1, 2)}
    return {"kind": kind, "domains": rng.randint(6, 40), "lo": 48, "hi": rng.choice([96, 192, 384])}


# ------------------------------------------------------------------ inputs
def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=DEV)


def _dx_dt(n):
    """1500 m cells and 5-year steps; the continental runs 750 m and 2.5 a."""
    return (1500.0, 5.0) if n <= 512 else (750.0, 2.5)


def _dome(ny, nx, dx, seed):
    """A window of the dome workload with a flow down its surface slope of at
    most 150 m/a and thickness above zero everywhere."""
    n = max(ny, nx)
    p = dome_problem(n, dx, seed=seed)
    i, j = (n - ny) // 2, (n - nx) // 2
    w = (slice(i, i + ny), slice(j, j + nx))
    f = {k: getattr(p, k)[w].copy() for k in ("bed", "H", "B", "beta", "smb")}
    s = np.maximum(f["bed"] + f["H"], (1.0 - 0.917) * f["H"])
    u, v = np.zeros((ny, nx + 1)), np.zeros((ny + 1, nx))
    u[:, 1:-1] = -(s[:, 1:] - s[:, :-1]) * 0.5 * (f["H"][:, 1:] + f["H"][:, :-1])
    v[1:-1] = (s[1:] - s[:-1]) * 0.5 * (f["H"][1:] + f["H"][:-1])
    top = max(np.abs(u).max(), np.abs(v).max(), 1e-12)
    f["u"], f["v"] = u * (150.0 / top), v * (150.0 / top)
    rng = np.random.default_rng(seed + 1000)
    f["u"][:, 1:-1] += 5.0 * gaussian_random_field(rng, ny, nx - 1, dx, 6 * dx)
    f["v"][1:-1] += 5.0 * gaussian_random_field(rng, ny - 1, nx, dx, 6 * dx)
    f["H"] = np.maximum(f["H"], 0.1) + 2.0 * rng.random((ny, nx))
    return f, rng


def _level(f, dx, m=1.0):
    """A one-level grid holding the fields."""
    ny, nx = f["H"].shape
    g = Grid(ny, nx, dx, device=DEV)
    g.sliding.m.set(m)
    for k, dst in (("u", g.state.u), ("v", g.state.v), ("H", g.state.H), ("bed", g.geometry.bed),
                   ("B", g.rheology.B), ("beta", g.sliding.beta), ("smb", g.forcing.smb), ("mask", g.state.mask),
                   ("H_prev", g.state.H_prev)):
        dst.set(_t(f[k]))
    fo = g.forward_operators
    fo.f_u.copy_(_t(f["f_u"]))
    fo.f_v.copy_(_t(f["f_v"]))
    return g


def _level_fields(case, seed, masked):
    f, rng = _dome(case["ny"], case["nx"], 1500.0, seed)
    ny, nx = case["ny"], case["nx"]
    f["mask"] = (rng.random((ny, nx)) < masked).astype(np.float64)
    f["H_prev"] = f["H"] + 0.1 * rng.standard_normal((ny, nx))
    f["f_u"] = 0.3 * rng.standard_normal((ny, nx + 1))
    f["f_v"] = 0.3 * rng.standard_normal((ny + 1, nx))
    # directions and multipliers vanish on the domain's edge facets, as the solvers keep them
    for a, b in (("du", "f_u"), ("lu", "f_u")):
        f[a] = rng.standard_normal(f[b].shape)
        f[a][:, [0, -1]] = 0.0
    for a, b in (("dv", "f_v"), ("lv", "f_v")):
        f[a] = rng.standard_normal(f[b].shape)
        f[a][[0, -1]] = 0.0
    f["dH"], f["lH"] = rng.standard_normal((ny, nx)), rng.standard_normal((ny, nx))
    return f


def _model(p, levels, precision):
    n = p.H.shape[0]
    m = IceDynamics(ny=n, nx=n, dx=p.dx, n_levels=levels, device=DEV, precision=precision)
    install(m.mg, p)
    return m


def _tolerances(model, rtol):
    for s in (model.forward_solver, model.adjoint_solver):
        s.fas_options.set(report_norms=False)
        s.mixed_options.max_outer = 40
        s.mixed_options.relative_tolerance = rtol


def _keep(pairs):
    """The fields a pass starts from: (destination, initial value) pairs."""
    return [d for d, _ in pairs], [v.clone() for _, v in pairs]


def _start(model):
    g = model.mg[0]
    s = g.state
    return _keep([(t.data, t.data) for t in (s.u, s.v, s.H, s.H_prev, s.mask, g.rheology.B)])


def _restart(kept):
    torch._foreach_copy_(kept[0], kept[1])


def _columns(case, seed):
    """A thermal model over the dome with a developed temperature profile:
    surface temperature at the top, towards the pressure-melting point at the
    bed under thick ice."""
    ny, nx, nz = case["ny"], case["nx"], case["nz"]
    f, rng = _dome(ny, nx, 1500.0, seed)
    g = Grid(ny, nx, 1500.0, device=DEV)
    th = ThermalModel(g, nz=nz, n_smooth=100, strain_heating=True)
    s = np.maximum(f["bed"] + f["H"], (1.0 - 0.917) * f["H"])
    Ts = 243.15 + 6.5e-3 * (2000.0 - s)
    warm = np.clip(f["H"] / 2000.0 + 0.2 * gaussian_random_field(rng, ny, nx, 1500.0, 20e3), 0.0, 1.0)
    depth = 1.0 - np.linspace(0.0, 1.0, nz)
    T = Ts[:, :, None] + (272.0 - Ts)[:, :, None] * warm[:, :, None] * depth[None, None, :] ** 2
    dt = 10.0
    H = np.maximum(f["H"] + 0.3 * dt * gaussian_random_field(rng, ny, nx, 1500.0, 20e3), 0.0)
    for k, dst in (("u", g.state.u), ("v", g.state.v), ("B", g.rheology.B), ("beta", g.sliding.beta),
                   ("bed", g.geometry.bed)):
        dst.set(_t(f[k]))
    g.state.H.set(_t(f["H"]))
    th.initialize(_t(Ts), T_field=_t(T), Q_geo=_t(np.full((ny, nx), 0.05)))
    frc = th.ops.enthalpy_forcing
    st = {"th": th, "dt": dt * SEC_PER_YR, "E": th.enthalpy.clone(), "Q_geo": frc.Q_geo.clone(),
          "E_surface": frc.E_surface.clone(), "H_prev": _t(f["H"]), "H": _t(H)}
    for k in ("u", "v", "B", "beta"):
        st[k] = _t(f[k])
    if "rtol" in case:
        th.ops.smoother_config.relative_tolerance = case["rtol"]
        if case["rtol"] < 1e-5:  # otherwise the default absolute test too
            th.ops.smoother_config.absolute_tolerance = 0.0
    return st


def prepare(case, seed):
    kind = case["kind"]
    if kind == "operators":
        f = _level_fields(case, seed, 0.05)
        g = _level(f, 1500.0, case["m"])
        fo, ao = g.forward_operators, g.adjoint_operators
        fo.set_rhs(5.0)
        for dst, k in ((fo.var_u, "du"), (fo.var_v, "dv"), (fo.var_H, "dH"), (g.adjoint.lambda_u.data, "lu"),
                       (g.adjoint.lambda_v.data, "lv"), (g.adjoint.lambda_H.data, "lH")):
            dst.copy_(_t(f[k]))
        return {"kind": kind, "fo": fo, "ao": ao}
    if kind == "sweeps":
        f = _level_fields(case, seed, 0.0)
        f["f_u"] *= 0.0
        f["f_v"] *= 0.0
        g = _level(f, 1500.0)
        fo, ao = g.forward_operators, g.adjoint_operators
        fo.set_rhs(5.0)
        if case["multicolour"]:
            fo.vanka_config.multicolour = ao.vanka_config.multicolour = True
        ao.f_u.copy_(_t(f["u"]))
        ao.f_v.copy_(_t(f["v"]))
        a, s = g.adjoint, g.state
        kept = _keep([(t.data, t.data) for t in (s.u, s.v, s.H, s.mask, a.lambda_u, a.lambda_v, a.lambda_H)])
        return {"kind": kind, "g": g, "kept": kept, "passes": case["passes"]}
    if kind == "glide":
        dx, dt = _dx_dt(case["n"])
        p = dome_problem(case["n"], dx, seed=seed)
        m = _model(p, case["levels"], "fp64")
        for s in (m.forward_solver, m.adjoint_solver):
            s.fas_options.set(maximum_vcycles=case["cycles"], relative_tolerance=0.0, absolute_tolerance=0.0,
                              report_norms=False)
        leaves = [_t(a).requires_grad_() for a in (p.H, p.bed, p.beta, p.smb)]
        adj = m.mg[0].adjoint
        z = [m.mg[0].state.u.data, m.mg[0].state.v.data, m.mg[0].state.mask.data, adj.lambda_u.data,
             adj.lambda_v.data, adj.lambda_H.data]
        return {"kind": kind, "m": m, "dt": dt, "leaves": leaves, "zero": z}
    if kind == "forward":
        dx, dt = _dx_dt(case["n"])
        p = dome_problem(case["n"], dx, seed=seed, grounding_line=case["n"] > 512)
        m = _model(p, case["levels"], "mixed")
        _tolerances(m, 1e-9)
        return {"kind": kind, "m": m, "dt": dt, "kept": _start(m)}
    if kind == "rollout":
        p = dome_problem(case["n"], 1500.0, seed=seed)
        m = _model(p, case["levels"], "mixed")
        _tolerances(m, 1e-9)
        rng = np.random.default_rng(seed + 7)
        n = case["n"]
        log_beta = _t(np.log(p.beta) + 0.1 * gaussian_random_field(rng, n, n, 1500.0, 30e3)).requires_grad_()
        obs = (_t(20.0 * gaussian_random_field(rng, n, n + 1, 1500.0, 30e3)),
               _t(20.0 * gaussian_random_field(rng, n + 1, n, 1500.0, 30e3)))
        H0, bed, smb = (_t(a) for a in (p.H, p.bed, p.smb))
        return {"kind": kind, "m": m, "log_beta": log_beta, "H0": H0.requires_grad_(), "bed": bed, "smb": smb,
                "obs": obs, "steps": case["steps"]}
    if kind in ("thermal", "thermal_adjoint"):
        st = _columns(case, seed)
        st["kind"] = kind
        if kind == "thermal_adjoint":
            rng = np.random.default_rng(seed + 11)
            ny, nx, nz = st["E"].shape
            st["gE"] = _t(rng.standard_normal((ny, nx, nz)))
            st["gB"] = _t(rng.standard_normal((ny, nx)))
        return st
    if kind == "coupled":
        p = dome_problem(case["n"], 1500.0, seed=seed)
        m = _model(p, case["levels"], "mixed")
        _tolerances(m, 1e-9)
        th = ThermalModel(m.mg[0], nz=case["nz"], n_smooth=100, strain_heating=True)
        sc = th.ops.smoother_config
        sc.relative_tolerance, sc.absolute_tolerance = 1e-8, 0.0
        Ts, q = thermal_forcing(p)
        th.initialize(_t(Ts), Q_geo=_t(q))
        step = CoupledStep(m, th)
        a, e = m.mg[0].adjoint, th.ops.enthalpy_state
        kept = _start(m)
        more = _keep([(t, t) for t in (a.lambda_u.data, a.lambda_v.data, a.lambda_H.data, e.E, e.E_prev)])
        return {"kind": kind, "m": m, "th": th, "step": step, "kept": (kept[0] + more[0], kept[1] + more[1]),
                "steps": case["steps"]}
    if kind == "ensemble":
        sizes = ensemble_sizes(case["domains"], case["lo"], case["hi"], seed=0)
        ens = Ensemble([valley_glacier(n, seed=1000 * seed + k) for k, n in enumerate(sizes)], precision="mixed",
                       iterations=3, batched=True)
        pairs = []
        for m in ens.models:
            g = m.mg[0]
            s, a = g.state, g.adjoint
            pairs += [(t.data, t.data) for t in (s.u, s.v, s.H, s.H_prev, s.mask, a.lambda_u, a.lambda_v, a.lambda_H)]
        return {"kind": kind, "ens": ens, "kept": _keep(pairs)}
    raise ValueError(f"unknown kind {kind!r}")


# ------------------------------------------------------------------ one pass
def run(state):
    return _RUN[state["kind"]](state)


def _run_operators(s):
    fo, ao = s["fo"], s["ao"]
    fo.compute_residual(5.0)
    fo.compute_jvp(5.0, freeze_phi=True)
    ao.compute_vjp(5.0)
    return {"r_u": fo.r_u, "r_v": fo.r_v, "r_H": fo.r_H, "jvp_u": fo.jvp_u, "jvp_v": fo.jvp_v, "jvp_H": fo.jvp_H,
            "vjp_u": ao.vjp_u, "vjp_v": ao.vjp_v, "vjp_H": ao.vjp_H}


def _run_sweeps(s):
    g = s["g"]
    _restart(s["kept"])
    g.forward_operators.vanka_sweep(5.0, s["passes"])
    g.adjoint_operators.vanka_sweep(5.0, s["passes"])
    a, st = g.adjoint, g.state
    return {"u": st.u.data, "v": st.v.data, "H": st.H.data, "lambda_u": a.lambda_u.data, "lambda_v": a.lambda_v.data,
            "lambda_H": a.lambda_H.data}


def _run_glide(s):
    torch._foreach_zero_(s["zero"])
    H, bed, beta, smb = s["leaves"]
    u, v, h = GlideStep.apply(0.0, s["dt"], s["m"], 0, H, bed, beta, smb)
    loss = 0.5 * ((u ** 2).sum() + (v ** 2).sum()) + h.sum()
    grads = torch.autograd.grad(loss, s["leaves"])
    return {"u": u, "v": v, "H": h, "g_H": grads[0], "g_bed": grads[1], "g_beta": grads[2], "g_smb": grads[3]}


def _run_forward(s):
    _restart(s["kept"])
    s["m"].forward(0.0, s["dt"])
    st = s["m"].mg[0].state
    return {"u": st.u.data, "v": st.v.data, "H": st.H.data}


def _run_rollout(s):
    loss, (u, v, H, _) = rollout(s["m"], s["H0"], s["bed"], torch.exp(s["log_beta"]), s["smb"], n_steps=s["steps"],
                                 dt=5.0, step_loss=lambda k, u, v, H: misfit(u, v, *s["obs"]), checkpoint=8)
    g_beta, g_H0 = torch.autograd.grad(loss, (s["log_beta"], s["H0"]))
    return {"loss": loss, "u": u, "v": v, "H": H, "g_log_beta": g_beta, "g_H0": g_H0}


def _run_thermal(s):
    with torch.no_grad():
        E, B = ThermalStep.apply(s["th"], s["dt"], s["E"], s["Q_geo"], s["E_surface"], s["u"], s["v"], s["H"],
                                 s["H_prev"], s["beta"], s["B"])
    return {"E": E, "B": B}


def _run_thermal_adjoint(s):
    th = s["th"]
    ops, g = th.ops, th.ops.grid
    torch._foreach_copy_([ops.enthalpy_state.E_prev, ops.H_prev, g.state.H.data, g.rheology.B.data],
                         [s["E"], s["H_prev"], s["H"], s["B"]])
    th.rebuild_step(s["dt"], s["E"])
    out = th.adjoint(s["dt"], s["gE"], s["gB"], B_in=s["B"], n_iter=64, relative_tolerance=1e-10)
    return {k: out[k] for k in ("lambda", "E_prev", "Q_geo", "E_surface", "u", "v", "H", "H_prev", "beta", "B")}


def _run_coupled(s):
    _restart(s["kept"])
    for k in range(s["steps"]):
        s["step"](10.0 * k, 10.0)
    g = s["m"].mg[0]
    st, a = g.state, g.adjoint
    return {"u": st.u.data, "v": st.v.data, "H": st.H.data, "E": s["th"].enthalpy, "B": g.rheology.B.data,
            "lambda_u": a.lambda_u.data, "lambda_v": a.lambda_v.data, "g_beta": g.sliding.beta.grad,
            "g_H_prev": g.state.H_prev.grad}


def _run_ensemble(s):
    _restart(s["kept"])
    s["ens"].step(0.0, 1.0)
    out = {"u": [], "v": [], "H": [], "lambda_u": [], "lambda_v": [], "g_beta": []}
    for m in s["ens"].models:
        g = m.mg[0]
        for k, t in (("u", g.state.u.data), ("v", g.state.v.data), ("H", g.state.H.data),
                     ("lambda_u", g.adjoint.lambda_u.data), ("lambda_v", g.adjoint.lambda_v.data),
                     ("g_beta", g.sliding.beta.grad)):
            out[k].append(t.reshape(-1))
    return {k: torch.cat(v) for k, v in out.items()}


_RUN = {"operators": _run_operators, "sweeps": _run_sweeps, "glide": _run_glide, "forward": _run_forward,
        "rollout": _run_rollout, "thermal": _run_thermal, "thermal_adjoint": _run_thermal_adjoint,
        "coupled": _run_coupled, "ensemble": _run_ensemble}


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    """Inputs read once and outputs written once, 8 bytes a value; operations
    of the formulas themselves, counted per cell, patch solve or column node.
    The solves to a tolerance count the passes of a typical solve."""
    kind = case["kind"]
    if kind == "operators":
        n = case["ny"] * case["nx"]
        # fields u, v, H, bed, B, beta, mask, three forcings, gamma, direction and multipliers (3 + 3); 9 results
        return {"bytes": 8 * n * (17 + 9), "flops": n * (150 + 330 + 300)}
    if kind == "sweeps":
        n = case["ny"] * case["nx"]
        # a patch solve: about 4 local Newton steps of 320 operations; an adjoint one: transpose 300, solve 60
        return {"bytes": 8 * n * (14 + 7), "flops": n * case["passes"] * (4 * 320 + 360)}
    if kind in ("glide", "forward", "rollout", "coupled"):
        n = case["n"] ** 2
        fine = 4.0 / 3.0 * n
        if kind == "glide":  # per V-cycle and level 10 + 20 passes, 50 on the finest
            return {"bytes": 8 * n * (9 + 7), "flops": case["cycles"] * (50 * n + 10 * n) * (2 * 320 + 360)}
        fwd = (14 * 16 * fine) * 650  # 14 outer iterations of about 16 red-black passes
        adj = (15 * 12 * fine) * 360
        if kind == "forward":
            return {"bytes": 8 * n * (10 + 3), "flops": fwd}
        k = case["steps"]
        if kind == "rollout":
            return {"bytes": 8 * n * (6 * k + 8), "flops": k * (2 * fwd + adj)}
        nz = case["nz"]
        return {"bytes": 8 * n * (k * (2 * nz + 20)), "flops": k * (fwd + adj + n * nz * (50 * 3 * 200 + 40 * 20))}
    if kind == "thermal":
        n = case["ny"] * case["nx"]
        sweeps = 3 if case["rtol"] > 1e-6 else 45
        return {"bytes": 8 * n * (2 * case["nz"] + 12), "flops": n * case["nz"] * sweeps * (3 * 200 + 80)}
    if kind == "thermal_adjoint":
        n = case["ny"] * case["nx"]
        return {"bytes": 8 * n * (5 * case["nz"] + 20), "flops": n * case["nz"] * (300 + 40 * 20)}
    cells = sum(s * s for s in ensemble_sizes(case["domains"], case["lo"], case["hi"], seed=0))
    fine = 4.0 / 3.0 * cells
    return {"bytes": 8 * cells * (10 + 10), "flops": 3 * fine * (16 * 650 + 12 * 360)}


def tolerance(case):
    """Measured by repeating each pass from inputs moved by one unit in the
    last place, and for the red-black V-cycles by 6e-8, an FP32 rounding:
    FP64 passes moved by 1e-16 to 3e-13, the solves to a residual of 1e-9 by
    up to 2e-9 (an iteration more or less leaves the error of that residual
    open, about 3e-8 in the multipliers), the ensemble's fixed FP32
    iterations by 7e-6."""
    return {"rel": _REL[case["kind"]]}


_REL = {"operators": 3e-12, "sweeps": 1e-11, "glide": 1e-10, "forward": 2e-7, "rollout": 2e-7, "thermal": 1e-9,
        "thermal_adjoint": 1e-9, "coupled": 2e-7, "ensemble": 3e-5}


# ------------------------------------------------------------------ plain torch float64
def exact(case, seed):
    """The single operators from the discretisation's formulas: the residual
    written down, its directional derivative and its transpose by automatic
    differentiation.  The solves and sweeps iterate to a tolerance or a count
    and have no closed result."""
    if case["kind"] != "operators":
        return None
    f = {k: _t(a) for k, a in _level_fields(case, seed, 0.05).items()}
    dx, dt = 1500.0, 5.0
    # thickness forcing of the implicit step, and the grounded fraction, frozen in every derivative
    f["f_H"] = f["H_prev"] / dt + f["smb"]
    f["phi"] = 1.0 / (1.0 + torch.exp(-torch.clamp(0.1 * (f["bed"] + 0.917 * f["H"]), -20.0, 20.0)))

    def rows(u, v, H):
        return _mass_momentum(u, v, H, f, dx, dt, case["m"])

    x = (f["u"], f["v"], f["H"])
    with torch.no_grad():
        ru, rv, rH = rows(*x)
        r_u, r_v = ru - f["f_u"], rv - f["f_v"]
        r_u[:, 0], r_u[:, -1], r_v[0], r_v[-1] = x[0][:, 0], x[0][:, -1], x[1][0], x[1][-1]
        r_H = (1.0 - f["mask"]) * (rH - f["f_H"]) + f["mask"] * (f["H"] - 0.1)
    y = [t.clone().requires_grad_() for t in x]
    ru, rv, rH = rows(*y)
    # J d by differentiating the transpose's result along a dummy multiplier
    lam = [torch.zeros_like(t, requires_grad=True) for t in (ru, rv, rH)]
    jt = torch.autograd.grad((ru, rv, rH), y, grad_outputs=lam, create_graph=True, retain_graph=True)
    ju, jv, jH = torch.autograd.grad(jt, lam, grad_outputs=(f["du"], f["dv"], f["dH"]), retain_graph=True)
    ju, jv, jH = ju.clone(), jv.clone(), (1.0 - f["mask"]) * jH
    ju[:, [0, -1]] = 0.0
    jv[[0, -1]] = 0.0
    lu, lv = f["lu"], f["lv"]
    gu, gv, gH = torch.autograd.grad((ru, rv, rH), y, grad_outputs=(lu, lv, f["lH"] * (1.0 - f["mask"])))
    gu, gv, gH = gu.clone(), gv.clone(), gH * (1.0 - f["mask"])
    gu[:, [0, -1]] = 0.0
    gv[[0, -1]] = 0.0
    return {"r_u": r_u, "r_v": r_v, "r_H": r_H, "jvp_u": ju, "jvp_v": jv, "jvp_H": jH, "vjp_u": gu, "vjp_v": gv,
            "vjp_H": gH}


def _mass_momentum(u, v, H, f, dx, dt, m):
    """Rows of the shallow-shelf momentum and mass balance on the MAC grid
    without forcing (zero on the edge facets): u (ny, nx+1), v (ny+1, nx)
    positive towards row 0, H (ny, nx)."""
    B, beta, bed, q = f["B"], f["beta"], f["bed"], f["phi"]
    n, eps, u_reg, drag0 = 3.0, 1e-6, 1.0, 1e-5  # the physical constants a grid starts with
    D = 1.0 / dx
    du = (u[:, 1:] - u[:, :-1]) * D
    dv = (v[:-1] - v[1:]) * D
    # shear strain of the interior vertices
    sh = 0.5 * ((u[:-1, 1:-1] - u[1:, 1:-1]) + (v[1:-1, 1:] - v[1:-1, :-1])) * D
    sq = torch.nn.functional.pad(sh * sh, (1, 1, 1, 1))
    corners = sq[:-1, :-1] + sq[:-1, 1:] + sq[1:, :-1] + sq[1:, 1:]
    e2 = du * du + dv * dv + du * dv + 0.25 * corners + eps
    eH = 0.5 * B * e2 ** ((1.0 - n) / (2.0 * n)) * H
    sxx, syy = 2.0 * eH * (2.0 * du + dv), 2.0 * eH * (du + 2.0 * dv)
    eV = 0.25 * (eH[:-1, :-1] + eH[:-1, 1:] + eH[1:, :-1] + eH[1:, 1:])
    sxy = torch.nn.functional.pad(2.0 * eV * sh, (1, 1, 1, 1))
    S = q * bed + (1.0 - (1.0 - q) * 0.917) * H

    def drag(w, c, pa, pb, ba, bb):
        be = 0.5 * (ba * pa + bb * pb)
        if m == 1.0:
            return (be + drag0) * w
        s2 = w * w + 0.25 * c
        return (be * (s2 + u_reg) ** ((m - 1.0) / 2.0) + drag0) * w

    ui, vi = u[:, 1:-1], v[1:-1]
    v2, u2 = v * v, u * u
    cu = v2[:-1, :-1] + v2[:-1, 1:] + v2[1:, :-1] + v2[1:, 1:]
    cv = u2[:-1, :-1] + u2[:-1, 1:] + u2[1:, :-1] + u2[1:, 1:]
    ru = ((sxx[:, 1:] - sxx[:, :-1]) + (sxy[:-1, 1:-1] - sxy[1:, 1:-1])) * D
    ru = ru - drag(ui, cu, q[:, :-1], q[:, 1:], beta[:, :-1], beta[:, 1:])
    ru = ru - 0.5 * (H[:, :-1] + H[:, 1:]) * (S[:, 1:] - S[:, :-1]) * D
    rv = ((syy[:-1] - syy[1:]) + (sxy[1:-1, 1:] - sxy[1:-1, :-1])) * D
    rv = rv - drag(vi, cv, q[:-1], q[1:], beta[:-1], beta[1:])
    rv = rv - 0.5 * (H[:-1] + H[1:]) * (S[:-1] - S[1:]) * D
    fx = 0.5 * (H[:, :-1] + H[:, 1:]) * ui - 0.5 * torch.sqrt(ui * ui + 10.0) * (H[:, 1:] - H[:, :-1])
    fy = 0.5 * (H[:-1] + H[1:]) * vi - 0.5 * torch.sqrt(vi * vi + 10.0) * (H[:-1] - H[1:])
    fx = torch.nn.functional.pad(fx, (1, 1))
    fy = torch.nn.functional.pad(fy, (0, 0, 1, 1))
    rH = H / dt + ((fx[:, 1:] - fx[:, :-1]) + (fy[:-1] - fy[1:])) * D
    return torch.nn.functional.pad(ru, (1, 1)), torch.nn.functional.pad(rv, (0, 0, 1, 1)), rH

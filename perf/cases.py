"""The work a program asks of this package, as timed cases.

Large steps of the dycore over the range of meshes (162 to 163 842 cells),
level counts, species counts and options, ensemble groups, a step driven
phase by phase, loading and unloading a state, training the learned
corrector, and stepping with it.  Every case enters through the public
Python driver (``HexDycoreDriver``, ``EnsembleGroup``, ``CorrectorNet``,
``LearnedStepper``) or, where the driver has no method of its own, the C ABI
that it wraps.

A dycore state lives in its driver and every step replaces it, so a pass of
the stepping cases restarts the driver from a second one that keeps the
initial state (``learned.copy_state``, a device copy), takes the case's
large steps and reads the whole published state back as tensors.

The fast numerics (FMA contraction) are left out: they run at the strict
path's speed and nothing selects them by default.
"""

import ctypes as ct
import functools
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "gpuwm-hex_amd"))

from hexdyn import capi, ensemble, learned  # noqa: E402
from hexdyn.case import build_case  # noqa: E402
from hexdyn.config import DycoreConfig  # noqa: E402
from hexdyn.driver import HexDycoreDriver  # noqa: E402
from hexdyn.lib import lib  # noqa: E402

MESHES = {
    # name: (workload of the package, cells, edges, vertices, timestep in s)
    "x1.162": ("x1.162-moist", 162, 480, 320, 7200.0),
    "x1.642": ("x1.642-moist", 642, 1920, 1280, 3600.0),
    "r642": ("r642-moist", 642, 1920, 1280, 3600.0),  # ragged: pentagons, hexagons and heptagons
    "x1.2562": ("x1.2562-moist", 2562, 7680, 5120, 1800.0),
    "x1.10242": ("x1.10242-moist", 10242, 30720, 20480, 1440.0),
    "x1.40962": ("x1.40962-moist", 40962, 122880, 81920, 720.0),
    "x1.163842": ("x1.163842-qv", 163842, 491520, 327680, 360.0),
}

BASE = dict(nlev=55, species=6, mixing=True, order=3, substeps=2, splits=3, monotonic=True, wind=False,
            physics=False, budgets=False, members=1, steps=1)


def listed():
    return [
        # the smallest useful globe: a unit-test or teaching run, one step and its output
        dict(BASE, name="step-162", kind="step", mesh="x1.162"),
        # an idealised dry-run configuration: second-order Runge-Kutta, unlimited transport of two tracers,
        # one dynamics subcycle, no mixing, few levels
        dict(BASE, name="step-642-rk2", kind="step", mesh="x1.642", nlev=26, species=2, mixing=False, order=2,
             substeps=4, splits=1, monotonic=False, steps=2),
        # a ragged mesh with heptagons under held physics tendencies and a reference wind
        dict(BASE, name="step-r642-physics", kind="step", mesh="r642", nlev=40, species=3, physics=True, wind=True),
        # the dry baroclinic-wave run on 2562 cells
        dict(BASE, name="step-2562-dry", kind="step", mesh="x1.2562", species=0, mixing=False, steps=2),
        # a host model that drives the phases itself and takes the scalars before they are published
        dict(BASE, name="phases-2562", kind="phases", mesh="x1.2562", nlev=50, species=6),
        # eight perturbed members on one mesh, advanced as one group
        dict(BASE, name="ensemble-8x2562", kind="step", mesh="x1.2562", members=8),
        # a 24 h budget run: moist steps with the 64-bit mass, energy and tracer integrals after each
        dict(BASE, name="step-10242-budgets", kind="step", mesh="x1.10242", budgets=True, steps=2),
        # the headline: moist, mixed, 40 962 cells, state read back every fourth step
        dict(BASE, name="step-40962", kind="step", mesh="x1.40962", steps=4),
        # the scale-up mesh with water vapour only
        dict(BASE, name="step-163842", kind="step", mesh="x1.163842", species=1),
        # an analysis read from host arrays, its budgets, and the state written back to the host
        dict(BASE, name="load-10242", kind="load", mesh="x1.10242"),
        # one optimiser step of the learned corrector on one coarse/fine pair
        dict(BASE, name="train-10242", kind="train", mesh="x1.10242", layers=4),
        # the learned-corrected form of the headline: coarse step, network, correction and checks
        dict(BASE, name="learned-40962", kind="learned", mesh="x1.40962", layers=4),
    ]


def draw(rng):
    kind = rng.choice(["step"] * 6 + ["phases", "load", "train", "learned"])
    mesh = rng.choice(["x1.162", "x1.642", "r642", "x1.2562", "x1.10242", "x1.40962"])
    c = dict(BASE, kind=kind, mesh=mesh, nlev=rng.choice([rng.randint(10, 63), 26, 32, 41, 55]))
    c["mixing"] = rng.random() < 0.75
    c["wind"] = rng.random() < 0.2
    if kind == "train":
        c["layers"] = rng.randint(2, 6)
        c["mesh"] = mesh if mesh != "x1.40962" else "x1.10242"
        return c
    if kind == "learned":
        c["layers"] = 4
        c["nlev"] = 55
        c["mesh"] = rng.choice(["x1.642", "x1.2562", "x1.10242", "x1.40962"])
        return c
    if kind == "load":
        c["mesh"] = mesh if mesh != "x1.40962" else "x1.10242"
        c["species"] = rng.randint(0, 8)
        return c
    c["species"] = rng.choice([0, 1, 2, 3, 4, 5, 6, 6, 7, 8])
    if mesh == "x1.40962":
        c["species"] = min(c["species"], 6)
    c["substeps"] = rng.choice([2, 2, 2, 3, 4])
    c["monotonic"] = rng.random() < 0.8
    c["physics"] = kind == "step" and rng.random() < 0.25
    c["steps"] = rng.randint(1, 2)
    if kind == "step" and mesh in ("x1.162", "x1.642", "x1.2562"):
        c["members"] = rng.choice([1, 1, 3, 5])
    c["budgets"] = kind == "step" and rng.random() < 0.25
    c["order"] = rng.choice([3, 3, 3, 2])
    c["splits"] = rng.choice([3, 3, 1])
    if c["splits"] == 1:
        c["substeps"] = max(c["substeps"], 4)
    return c


# ------------------------------------------------------------------ inputs
@functools.lru_cache(maxsize=4)
def _case(mesh, nlev, species, mixing, order, substeps, splits, monotonic, wind):
    """Mesh, vertical grid, reference state and initial state: read once by a program and kept."""
    cfg = DycoreConfig(config_dt=MESHES[mesh][4], config_horiz_mixing="2d_smagorinsky" if mixing else "off",
                       config_time_integration_order=order, config_number_of_sub_steps=substeps,
                       config_dynamics_split_steps=splits, config_monotonic=monotonic)
    more = {"reference_wind": (12.0, 3.0)} if wind else {}
    return build_case(MESHES[mesh][0], nlev=nlev, config=cfg, n_scalars=species, moist=species > 0, **more)


def _built(c):
    return _case(c["mesh"], c["nlev"], c["species"], c["mixing"], c["order"], c["substeps"], c["splits"],
                 c["monotonic"], c["wind"])


def _state(built, seed):
    """A seeded theta bubble on smooth 0.05 K noise: another analysis of the same day for another seed."""
    st = learned.perturbed_state(built, seed=seed)
    rng = np.random.default_rng(seed + 7919)
    noise = rng.standard_normal(st["rtheta_m"].shape, dtype=np.float32) * np.float32(0.05)
    st["rtheta_m"] = (st["rtheta_m"] + st["rho_zz"] * noise).astype(np.float32)
    return st


def _tendencies(built, seed):
    """Held physics tendencies of ordinary size: heating of about 10 K a day, drag and moistening."""
    rng = np.random.default_rng(seed + 104729)
    L, C, E, T = built.n_levels, built.mesh.n_cells, built.mesh.n_edges, built.n_scalars
    f = lambda shape, size: (rng.standard_normal(shape, dtype=np.float32) * np.float32(size))  # noqa: E731
    return dict(rho=f((L, C), 1e-9), rho_u=f((L, E), 1e-5), rho_theta=f((L, C), 1e-4),
                scalars=f((T, L, C), 1e-10) if T else None)


def prepare(case, seed):
    built = _built(case)
    kind = case["kind"]
    if kind == "load":
        return {"kind": kind, "drv": HexDycoreDriver.from_host(built), "state": _state(built, seed)}
    if kind == "train":
        return _prepare_train(case, built, seed)
    if kind == "learned":
        return _prepare_learned(case, built, seed)
    if case["members"] > 1:
        states = [_state(built, 1000 * seed + k) for k in range(case["members"])]
        group = ensemble.EnsembleGroup(built, states)
        first = HexDycoreDriver.from_host(group.union, state=ensemble.join_states(states))
        work = group.driver
        union, start = group.union, None
    else:
        union, start, group = built, _state(built, seed), None
        first = HexDycoreDriver.from_host(built, state=start)
        work = HexDycoreDriver.from_host(built, state=start)
    if case["physics"]:
        work.set_physics_tendencies(**_tendencies(union, seed))
    if kind == "phases":
        work.set_post_transport_clamp(False)
    return {"kind": kind, "group": group, "first": first, "work": work, "steps": case["steps"],
            "budgets": case["budgets"], "built": built}


def _prepare_train(case, built, seed):
    """A pair made from the seed alone: the coarse state, and a fine state that differs from it as two short
    steps of the same day do; random weights, scales of the raw features and differences."""
    coarse = HexDycoreDriver.from_host(built, state=_state(built, seed))
    fine = HexDycoreDriver.from_host(built, state=_fine_state(built, seed))
    net = learned.CorrectorNet(coarse, case["layers"])
    net.set_params(learned.init_params(case["layers"], seed=seed))
    net.set_scales(*_scales(built))
    return {"kind": "train", "coarse": coarse, "fine": fine, "net": net}


def _fine_state(built, seed):
    st = _state(built, seed)
    rng = np.random.default_rng(seed + 15485863)
    for name, size in (("rho_zz", 1e-4), ("rtheta_m", 1e-4), ("ru", 1e-2)):
        st[name] = (st[name] * (1 + rng.standard_normal(st[name].shape, dtype=np.float32) * np.float32(size)))
    st["rw"] = st["rw"].copy()
    st["rw"][1:-1] += st["rho_zz"][1:] * rng.standard_normal(st["rw"][1:-1].shape, dtype=np.float32) * np.float32(0.02)
    return st


def _scales(built):
    """Feature and target scales of the kind training starts from: per channel, flat in the vertical."""
    L = built.n_levels
    mean, scale, out = np.zeros((6, 64), np.float32), np.zeros((6, 64), np.float32), np.ones((5, 64), np.float32)
    mean[3, :L] = 320.0
    mean[4, :L] = 0.5
    for ch, s, n in ((0, 0.1, L), (1, 0.1, L), (2, 10.0, L + 1), (3, 0.02, L), (4, 2.0, L), (5, 200.0, L)):
        scale[ch, :n] = s
    scale[0, L] = 1e4  # the Coriolis parameter
    out[0, :], out[1, :], out[2, :], out[3, :], out[4, :] = 0.3, 0.3, 0.05, 1e-4, 0.02
    return mean, scale, out


def _prepare_learned(case, built, seed):
    # the trained weights of the headline mesh on every mesh; the seeded noise lies outside the envelope of their
    # training states, so the limits are open and a step falls back only on a state that is not finite
    weights = learned.load(learned.DATA / "corrector_x1.40962-moist.npz")
    limits = learned.Limits(cfl_h=float("inf"), mass_rel=float("inf"))
    stepper = learned.LearnedStepper(built, weights, layers=case["layers"], limits=limits)
    start = _state(built, seed)
    first = HexDycoreDriver.from_host(built, state=start)
    stepper.set_state(start)
    return {"kind": "learned", "first": first, "stepper": stepper}


# ------------------------------------------------------------------ one pass
def run(s):
    return {"step": _run_step, "phases": _run_phases, "load": _run_load, "train": _run_train,
            "learned": _run_learned}[s["kind"]](s)


def _run_step(s):
    drv = s["work"]
    learned.copy_state(drv, s["first"])
    out = {}
    if s["budgets"]:
        for k in range(s["steps"]):
            drv.step_device(1)
            out[f"budgets {k}"] = np.array(list(drv.integrals().values()))
    else:
        drv.step_device(s["steps"])
    out["state"] = drv.state_tensors()
    return out


def _run_phases(s):
    """One large step by its phases, the transported scalars handed to the caller before the step ends."""
    drv, cfg = s["work"], s["built"].config
    learned.copy_state(drv, s["first"])
    drv.phase("begin_step")
    n = cfg.config_number_of_sub_steps
    half = max(1, n // 2)
    acoustic = (1, half, n) if cfg.config_time_integration_order == 3 else (half, half, n)
    for sub in range(1, cfg.config_dynamics_split_steps + 1):
        drv.phase("begin_subcycle", sub)
        for st in (1, 2, 3):
            drv.phase("dyn_tend", st)
            for ss in range(1, acoustic[st - 1] + 1):
                drv.phase("acoustic_substep", st, ss)
                drv.phase("divergence_damping", st)
            drv.phase("recover", st)
            drv.phase("solve_diagnostics", st)
        drv.phase("end_subcycle", sub)
    out = {}
    if s["built"].n_scalars:
        for st in (1, 2, 3):
            drv.phase("scalars", st)
        q = drv.export_field("SCALARS_STAGE").clamp_(min=0.0)  # the caller's own microphysics stands here
        rc = lib().hexdyn_import_field(drv.handle, capi.FIELD_ID["SCALARS_STAGE"], ct.c_void_p(q.data_ptr()),
                                       ct.c_void_p(drv.stream_ptr()))
        if rc != 0:
            raise RuntimeError(f"hexdyn_import_field failed ({rc})")
    drv.phase("end_step")
    out["state"] = drv.state_tensors()
    return out


def _run_load(s):
    s["drv"].set_state(s["state"])
    return {"budgets": np.array(list(s["drv"].integrals().values())), "state": s["drv"].get_state()}


def _run_train(s):
    net = s["net"]
    net.forward(s["coarse"], keep=True)
    net.set_target(s["coarse"], s["fine"])
    loss = net.loss()
    net.backward()
    net.adam(1e-4, 1)
    return {"loss": np.array([loss[k] for k in ("total", "u", "theta_m", "rho_zz", "w")]), "grads": net.get_grads(),
            "params": net.get_params(), "outputs": net.export("Y")}


def _run_learned(s):
    st = s["stepper"]
    learned.copy_state(st.coarse, s["first"])
    st.step(1)
    return {"state": st.coarse.state_tensors()}


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    _, C, E, V, _ = MESHES[case["mesh"]]
    L, T, n = case["nlev"], case["species"], case["members"]
    cells, edges = L * C * 4, L * E * 4
    state = (9 + T) * cells + 2 * edges  # the published fields
    # the dycore's arithmetic: counted operations per level of a cell, with its three edges and two vertices
    stage = 600
    sub = 180
    moist = 450 * T
    net = 2.0 * C * (384 * 128 + case.get("layers", 0) * 256 * 128 + 128 * 320)
    if case["kind"] == "load":
        return {"bytes": float((4 + T) * cells + 2 * edges + state), "flops": 40.0 * L * C}
    if case["kind"] == "train":
        return {"bytes": float(2 * (4 * cells + edges) + C * 320 * 4), "flops": 3 * net}
    static = (8 + 12) * cells + 2 * edges  # vertical metrics and reference state
    if case["kind"] == "learned":
        flops = L * C * (3 * (stage + 4 * sub) + 3 * moist / 3) + net
        return {"bytes": float(3 * state + static), "flops": float(flops)}
    per_sub = 3 * stage + (4 * sub if case["order"] == 3 else 8 * sub)
    flops = case["steps"] * L * C * (case["splits"] * per_sub + moist)
    return {"bytes": float(n * (2 * state + static)), "flops": float(n * flops)}


# ------------------------------------------------------------------ the same in 64 bits
def exact(case, seed):
    """Loading (the diagnostics of a state, its integrals) and the training step in 64 bits.  A large step has
    no short statement: it is some forty operators applied thousands of times."""
    if case["kind"] == "load":
        return _exact_load(case, seed)
    if case["kind"] == "train":
        return _exact_train(case, seed)
    return None


def _f64(a):
    return np.asarray(a, dtype=np.float64)


def _diagnose(built, st):
    """Published diagnostics of a prognostic state in 64 bits: theta_m, Exner, perturbations, u and w."""
    g, r, m = built.grid, built.reference, built.mesh
    rho, rt, ru, rw = (_f64(st[k]) for k in ("rho_zz", "rtheta_m", "ru", "rw"))
    zz, rtb, exb = _f64(g.zz), _f64(r.rtheta_base), _f64(r.exner_base)
    rgas, cp, p0 = 287.0, 1004.5, 1e5
    exner = (zz * (rgas / p0) * rt) ** (rgas / (cp - rgas))
    rtp = rt - rtb
    c0, c1 = m.cellsOnEdge[:, 0], m.cellsOnEdge[:, 1]
    L = rho.shape[0]
    fzm, fzp = _f64(g.fzm)[1:, None], _f64(g.fzp)[1:, None]
    col = np.zeros((L + 1, m.n_cells))
    col[1:L] = rw[1:L] / (fzm * zz[1:] + fzp * zz[:-1])
    zb, zb3 = _f64(g.zb_cell), _f64(g.zb3_cell)
    cf = np.array([g.cf1, g.cf2, g.cf3], dtype=np.float64)
    for s in range(m.max_edges):
        has = s < m.nEdgesOnCell
        e = np.where(has, m.edgesOnCell[:, s], 0)
        sign = np.where(has, np.where(c0[e] == np.arange(m.n_cells), 1.0, -1.0), 0.0)
        flux = np.empty((L, m.n_cells))
        flux[0] = cf @ ru[:3, e]
        flux[1:] = fzm * ru[1:, e] + fzp * ru[:-1, e]
        col[:L] += sign * (zb[:L, :, s] + np.copysign(1.0, flux) * zb3[:L, :, s]) * flux
    w = np.zeros_like(col)
    w[0] = col[0] / (cf @ rho[:3])
    w[1:L] = col[1:L] / (fzm * rho[1:] + fzp * rho[:-1])
    return {"rho_zz": rho, "rtheta_m": rt, "ru": ru, "rw": rw, "scalars": _f64(st["scalars"]), "theta_m": rt / rho,
            "exner": exner, "rho_p": rho - _f64(r.rho_base), "rtheta_p": rtp,
            "pressure_p": zz * rgas * (exner * rtp + rtb * (exner - exb)), "u": 2 * ru / (rho[:, c0] + rho[:, c1]),
            "w": w}


def _exact_load(case, seed):
    built = _built(case)
    d = _diagnose(built, _state(built, seed))
    m, g = built.mesh, built.grid
    volume = (1.0 / _f64(built.inv_area_cell))[None, :] * (1.0 / _f64(g.rdzw))[:, None]
    ke = np.zeros_like(d["rho_zz"])
    part = 0.25 * _f64(m.dcEdge) * _f64(m.dvEdge) * d["u"] ** 2
    for s in range(m.max_edges):
        has = s < m.nEdgesOnCell
        ke += np.where(has, part[:, np.where(has, m.edgesOnCell[:, s], 0)], 0.0)
    ke *= _f64(built.inv_area_cell)
    qv = d["scalars"][0] if built.n_moist else 0.0
    temp = d["theta_m"] * d["exner"] / (1.0 + 461.6 / 287.0 * qv)
    z = 0.5 * (_f64(g.zgrid)[:-1] + _f64(g.zgrid)[1:])
    energy = (volume * d["rho_zz"] * ((1004.5 - 287.0) * temp + 9.80616 * z + ke)).sum()
    sums = [(volume * d["rho_zz"]).sum(), (volume * d["rtheta_m"]).sum(), energy]
    sums += [(volume * d["rho_zz"] * q).sum() for q in d["scalars"]]
    return {"budgets": np.array(sums), "state": d}


def _exact_train(case, seed):
    built = _built(case)
    m, L, layers = built.mesh, built.n_levels, case["layers"]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    a, b = _diagnose(built, _state(built, seed)), _diagnose(built, _fine_state(built, seed))
    mean, scale, oscale = (t(_f64(x)) for x in _scales(built))
    C, E = m.n_cells, m.n_edges
    has = t((np.arange(m.max_edges)[None, :] < m.nEdgesOnCell[:, None]).astype(np.float64))
    eoc, coc = t(np.maximum(m.edgesOnCell, 0).astype(np.int64)), t(np.maximum(m.cellsOnCell, 0).astype(np.int64))
    coe, count = t(m.cellsOnEdge.astype(np.int64)), t(m.nEdgesOnCell.astype(np.float64))
    cos, sin = t(_f64(built.cos_angle_edge)), t(_f64(built.sin_angle_edge))
    # features: least-squares wind of the cell from its edges, w, theta_m, rho_zz, vapour, Coriolis parameter
    u = t(a["u"]).T
    x = torch.zeros(C, 6, 64, dtype=torch.float64, device=dev)
    cs, sn = cos[eoc] * has, sin[eoc] * has
    m11, m12, m22 = (cs * cs).sum(1), (cs * sn).sum(1), (sn * sn).sum(1)
    b1, b2 = ((k[:, :, None] * u[eoc]).sum(1) for k in (cs, sn))
    det = (m11 * m22 - m12 * m12)[:, None]
    x[:, 0, :L] = (m22[:, None] * b1 - m12[:, None] * b2) / det
    x[:, 1, :L] = (m11[:, None] * b2 - m12[:, None] * b1) / det
    x[:, 0, L] = (t(_f64(m.fEdge))[eoc] * has).sum(1) / count
    x[:, 2, :L + 1] = t(a["w"]).T
    x[:, 3, :L] = t(a["theta_m"]).T
    x[:, 4, :L] = t(a["rho_zz"]).T
    if built.n_scalars:
        x[:, 5, :L] = t(a["scalars"][0]).T
    x = ((x - mean) * scale).reshape(C, 384)
    flat = t(_f64(_first_params(layers, seed))).requires_grad_()
    shapes = [(384, 128), (128,)] + [(256, 128), (128,)] * layers + [(128, 320), (320,)]
    parts = [p.reshape(s) for p, s in zip(flat.split([int(np.prod(s)) for s in shapes]), shapes)]
    h = torch.relu(x @ parts[0] + parts[1])
    for k in range(layers):
        near = (h[coc] * has[:, :, None]).sum(1) / count[:, None]
        h = h + torch.relu(torch.cat([h, near], 1) @ parts[2 + 2 * k] + parts[3 + 2 * k])
    y = h @ parts[-2] + parts[-1]
    out = y.reshape(C, 5, 64)
    du = cos[:, None] * out[coe, 0].mean(1) + sin[:, None] * out[coe, 1].mean(1)
    want = {k: (t(b[k]) - t(a[k])).T for k in ("u", "theta_m", "rho_zz", "w")}
    errs = [(du[:, :L] - want["u"] / oscale[0, :L]), (out[:, 2, :L] - want["theta_m"] / oscale[2, :L]),
            (out[:, 3, :L] - want["rho_zz"] / oscale[3, :L]),
            (out[:, 4, 1:L] - want["w"][:, 1:L] / oscale[4, 1:L])]
    loss = [e.square().mean() for e in errs]
    total = sum(loss)
    total.backward()
    g = flat.grad
    # Adam's first step: the moments' bias corrections leave g / (|g| + eps)
    new = flat.detach() - 1e-4 * g / (g.abs() + 1e-8)
    return {"loss": torch.stack([total.detach()] + [v.detach() for v in loss]), "grads": g, "params": new,
            "outputs": y.detach()}


def _first_params(layers, seed):
    """He-normal matrices, zero biases, the decoder scaled down: the same draw the training case starts from."""
    rng = np.random.default_rng(seed)
    parts = []
    for name, shape in ([("in", (384, 128)), ("b", (128,))] + [("l", (256, 128)), ("b", (128,))] * layers
                        + [("out", (128, 320)), ("b", (320,))]):
        if len(shape) == 1:
            parts.append(np.zeros(shape, dtype=np.float32))
        else:
            std = np.sqrt(2.0 / shape[0]) * (0.01 if name == "out" else 1.0)
            parts.append((rng.standard_normal(shape) * std).astype(np.float32).ravel())
    return np.concatenate([p.ravel() for p in parts])

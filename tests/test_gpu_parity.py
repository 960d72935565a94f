"""HIP dycore (libhexdyn.so through its C ABI) against the CPU oracle.

Strict numerics: every phase and every whole step bit for bit equal to the
binary32 restatement.  Fast numerics (FMA contraction): within relative L2
1e-5 of the FP64 restatement on u, w, theta_m and rho_zz after one step.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from hexdyn.case import initial_state_arrays  # noqa: E402
from hexdyn.config import DycoreConfig  # noqa: E402
from hexdyn.setup import rk_schedule  # noqa: E402
from oracle.oracle import Oracle  # noqa: E402


def _driver(case):
    from hexdyn.driver import HexDycoreDriver

    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    return HexDycoreDriver.from_host(case)


def _bits_equal(a, b):
    a = np.ascontiguousarray(a, dtype=np.float32).ravel()
    b = np.ascontiguousarray(b, dtype=np.float32).ravel()
    return a.size == b.size and np.array_equal(a.view(np.uint32), b.view(np.uint32))


def _diff(a, b):
    a = np.asarray(a, dtype=np.float64).ravel()
    b = np.asarray(b, dtype=np.float64).ravel()
    ne = np.flatnonzero(a.astype(np.float32).view(np.uint32) != b.astype(np.float32).view(np.uint32))
    return f"{ne.size} words differ, max |d| {np.abs(a - b).max():.3e}"


STATE = ["RHO_ZZ", "RTHETA_M", "RU", "RW", "THETA_M", "EXNER", "RHO_P", "RTHETA_P", "PRESSURE_P", "U", "W"]


def _phase_walk(case, physics=None):
    o = Oracle(case, 32)
    o.set_state(initial_state_arrays(case), rebuild=True)
    d = _driver(case)
    if physics is not None:
        o.set_physics(**physics)
        d.set_physics_tendencies(**physics)
    bad = []

    def cmp(tag, fields):
        for f in fields:
            a = o.export_field(f)
            b = d.export_field(f).cpu().numpy()
            if not _bits_equal(a, b):
                bad.append(f"{tag}:{f}: {_diff(a, b)}")

    state = STATE + (["SCALARS"] if case.n_scalars else [])
    mixing = case.config.config_horiz_mixing != "off"
    cmp("init", state)
    o.begin_step(); d.phase("begin_step")
    cmp("begin_step", ["V", "PV_EDGE", "KE", "DIVERGENCE", "VORTICITY"] + (["QTOT", "CQW", "CQU"] if case.n_moist else []))
    cfg = case.config
    sched = rk_schedule(cfg.config_dt, acoustic_substeps=cfg.config_number_of_sub_steps,
                        dynamics_splits=cfg.config_dynamics_split_steps)
    for sub in range(1, cfg.config_dynamics_split_steps + 1):
        o.begin_subcycle(sub); d.phase("begin_subcycle", sub)
        cmp(f"s{sub}", ["A_TRI", "ALPHA_TRI", "GAMMA_TRI", "COFWZ", "COFWT", "COFTZ", "EULER_RU", "EULER_RW",
                        "TEND_RHO"] + (["KDIFF", "EULER_THETA"] if mixing else []))
        for st in (1, 2, 3):
            o.dyn_tend(st); d.phase("dyn_tend", st)
            cmp(f"s{sub}t{st}", ["TEND_RU", "TEND_RT", "TEND_RW"])
            for ss in range(1, sched[st - 1].acoustic_steps + 1):
                o.acoustic_substep(st, ss); d.phase("acoustic_substep", st, ss)
                cmp(f"s{sub}t{st}a{ss}", ["RU_P", "RU_AVG", "RW_P", "WW_AVG", "RHO_PP", "RTHETA_PP"])
                o.divergence_damping(st); d.phase("divergence_damping", st)
                cmp(f"s{sub}t{st}d{ss}", ["RU_P"])
            o.recover(st); d.phase("recover", st)
            cmp(f"s{sub}t{st}r", STATE + ["FLUX_U", "FLUX_W"])
            o.solve_diagnostics(st); d.phase("solve_diagnostics", st)
            cmp(f"s{sub}t{st}g", ["V", "PV_EDGE", "KE", "DIVERGENCE", "VORTICITY"])
        o.end_subcycle(sub); d.phase("end_subcycle", sub)
    if case.n_scalars:
        for st in (1, 2, 3):
            o.scalars(st); d.phase("scalars", st)
            cmp(f"q{st}", ["SCALARS_STAGE"])
    o.end_step(); d.phase("end_step")
    cmp("end", state)
    return bad


@pytest.mark.parametrize("name", ["x1.642-moist", "x1.2562-dry", "r642-moist"])
def test_phase_by_phase_bitwise(get_case, name):
    # r642: ragged mesh with heptagons, which runs the maxEdges-7 kernels
    print(f"[gpu] phase walk {name}", flush=True)
    bad = _phase_walk(get_case(name))
    assert not bad, "\n".join(bad[:20])


def _mixing(get_case, name, **kw):
    import dataclasses

    base = get_case(name)
    return get_case(name, config=dataclasses.replace(base.config, config_horiz_mixing="2d_smagorinsky", **kw))


@pytest.mark.parametrize("name,visc4", [("x1.642-moist", 0.05), ("x1.2562-dry", 0.05), ("x1.2562-dry", 0.0),
                                        ("r642-moist", 0.05)])
def test_phase_by_phase_bitwise_with_mixing(get_case, name, visc4):
    print(f"[gpu] phase walk with 2d_smagorinsky mixing {name} visc4={visc4}", flush=True)
    bad = _phase_walk(_mixing(get_case, name, config_visc4_2dsmag=visc4))
    assert not bad, "\n".join(bad[:20])


def test_ragged_mesh_three_steps_bitwise(get_case):
    """Pentagons, hexagons and heptagons (maxEdges 7): three whole steps on
    the replayed graph bit for bit equal to the oracle."""
    print("[gpu] r642-moist (maxEdges 7) 3 steps", flush=True)
    case = get_case("r642-moist")
    assert case.mesh.max_edges == 7
    o = Oracle(case, 32)
    o.set_state(initial_state_arrays(case), rebuild=True)
    assert o.step(3) == 0
    d = _driver(case)
    d.step_device(3)
    ref, got = o.get_state(), d.get_state()
    for k in ref:
        assert _bits_equal(ref[k], got[k]), f"{k}: {_diff(ref[k], got[k])}"


@pytest.mark.parametrize("nlev", [10, 50, 63])
def test_level_counts_two_steps_bitwise(get_case, nlev):
    """A short column, one whose rows (56 floats apart) end in padding
    lanes, and the deepest one a 64-lane row holds (L + 1 = 64, the
    interface row on the last lane), with mixing: 2 steps bit for bit."""
    print(f"[gpu] x1.642-moist at {nlev} levels, mixing on, 2 steps", flush=True)
    import dataclasses

    base = get_case("x1.642-moist", nlev=nlev)
    case = get_case("x1.642-moist", nlev=nlev,
                    config=dataclasses.replace(base.config, config_horiz_mixing="2d_smagorinsky"))
    assert case.n_levels == nlev
    o = Oracle(case, 32)
    o.set_state(initial_state_arrays(case), rebuild=True)
    assert o.step(2) == 0
    d = _driver(case)
    d.step_device(2)
    ref, got = o.get_state(), d.get_state()
    for k in ref:
        assert _bits_equal(ref[k], got[k]), f"{k}: {_diff(ref[k], got[k])}"


def test_three_steps_bitwise_moist(get_case):
    print("[gpu] x1.2562-moist 3 steps", flush=True)
    case = get_case("x1.2562-moist")
    o = Oracle(case, 32)
    o.set_state(initial_state_arrays(case), rebuild=True)
    assert o.step(3) == 0
    d = _driver(case)
    d.step_device(3)
    ref, got = o.get_state(), d.get_state()
    for k in ref:
        assert _bits_equal(ref[k], got[k]), f"{k}: {_diff(ref[k], got[k])}"


@pytest.mark.parametrize("mixing", ["off", "2d_smagorinsky"])
def test_headline_mesh_step_bitwise_and_conservative(get_case, mixing):
    print(f"[gpu] x1.40962-moist 1 step, mixing {mixing}", flush=True)
    case = get_case("x1.40962-moist") if mixing == "off" else _mixing(get_case, "x1.40962-moist")
    d = _driver(case)
    s0 = d.get_state()
    d.step_device(1)
    got = d.get_state()
    o = Oracle(case, 32)
    o.set_state(initial_state_arrays(case), rebuild=True)
    assert o.step(1) == 0
    ref = o.get_state()
    for k in ref:
        assert _bits_equal(ref[k], got[k]), f"{k}: {_diff(ref[k], got[k])}"
    # size-independent properties of the GPU result
    area = 1.0 / case.inv_area_cell.astype(np.float64)[None, :]
    dz = (1.0 / case.grid.rdzw.astype(np.float64))[:, None]
    m0 = (area * s0["rho_zz"].astype(np.float64) * dz).sum()
    m1 = (area * got["rho_zz"].astype(np.float64) * dz).sum()
    assert abs(m1 / m0 - 1) < 1e-6
    assert got["scalars"].min() >= 0.0
    for k, v in got.items():
        assert np.isfinite(v).all(), k


@pytest.mark.parametrize("name", ["x1.10242-moist", "x1.163842-qv"])
def test_other_mesh_sizes_step_bitwise(get_case, name, capsys, monkeypatch):
    """The ensemble mesh (x1.10242, T=6, dt 1440 s) and the scale-up mesh
    (x1.163842, water vapour only, dt 360 s), with 2-D Smagorinsky mixing:
    one large step bit for bit equal to the oracle, then 4 more steps with
    dry and tracer masses held in FP64 integrals.  Building the x1.163842
    case takes a minute or two of host time; its stages are printed."""
    print(f"[gpu] {name} 1 step bitwise + 4 steps of budgets, mixing on", flush=True)
    monkeypatch.setenv("HEXDYN_VERBOSE", "1")
    with capsys.disabled():
        case = _mixing(get_case, name)
    d = _driver(case)
    a = d.integrals()
    d.step_device(1)
    got = d.get_state()
    o = Oracle(case, 32)
    o.set_state(initial_state_arrays(case), rebuild=True)
    assert o.step(1) == 0
    ref = o.get_state()
    del o
    for k in ref:
        assert _bits_equal(ref[k], got[k]), f"{k}: {_diff(ref[k], got[k])}"
    d.step_device(4)
    b = d.integrals()
    assert abs(b["dry_mass"] / a["dry_mass"] - 1) < 1e-9
    for s in range(case.n_scalars):
        assert abs(b[f"tracer_mass_{s}"] / a[f"tracer_mass_{s}"] - 1) < 1e-6, s
    st = d.get_state()
    assert np.isfinite(st["rho_zz"]).all() and (st["scalars"] >= 0).all()


def test_fast_numerics_within_tolerance_of_fp64(get_case):
    """Tolerance: relative L2 <= 1e-5 against FP64 on u, theta_m and rho_zz.
    For w, a small residual of cancelling terms, binary32 evaluated in the
    reference's own order already sits near 1e-4 (the strict path, equal to
    the binary32 restatement bit for bit); fast numerics must be no worse than
    1.5 times that floor."""
    print("[gpu] fast numerics vs FP64", flush=True)
    base = get_case("x1.2562-moist")
    import dataclasses

    fast = dataclasses.replace(base, config=dataclasses.replace(base.config, numerics="fast"))
    d = _driver(fast)
    d.step_device(1)
    got = d.get_state()
    o = Oracle(base, 64)
    o.set_state(initial_state_arrays(base), rebuild=True)
    assert o.step(1) == 0
    ref = o.get_state()
    o32 = Oracle(base, 32)
    o32.set_state(initial_state_arrays(base), rebuild=True)
    assert o32.step(1) == 0
    strict = o32.get_state()

    def rel(x, k):
        return np.linalg.norm(x[k].astype(np.float64) - ref[k]) / np.linalg.norm(ref[k].astype(np.float64))

    for k in ("u", "w", "theta_m", "rho_zz"):
        print(f"  {k}: fast rel L2 vs FP64 = {rel(got, k):.3e}, strict binary32 = {rel(strict, k):.3e}")
    for k in ("u", "theta_m", "rho_zz"):
        assert rel(got, k) <= 1e-5, k
    assert rel(got, "w") <= 1.5 * rel(strict, "w")
    assert not _bits_equal(got["u"], strict["u"])  # the fast path really is a different instruction stream


def test_validation_flag_refuses_and_keeps_state(get_case):
    print("[gpu] validation flag", flush=True)
    case = get_case("x1.642-dry")
    d = _driver(case)
    before = d.get_state()
    # the carried theta_m feeds the theta flux; a NaN there must trip the flag
    bad = before["theta_m"].copy()
    bad[3, 7] = np.nan
    t = torch.from_numpy(bad).cuda()
    from hexdyn import capi
    from hexdyn.lib import lib
    import ctypes as ct

    rc = lib().hexdyn_import_field(d.handle, capi.FIELD_ID["THETA_M"], ct.c_void_p(t.data_ptr()),
                                   ct.c_void_p(d.stream_ptr()))
    assert rc == 0
    with pytest.raises(FloatingPointError):
        d.step_device(1)
    after = d.get_state()
    for k in ("rho_zz", "rtheta_m", "ru", "rw", "exner", "u", "w"):
        assert _bits_equal(after[k], before[k]), k
    assert np.isnan(after["theta_m"][3, 7])
    # the published state is intact: with the carried theta restored the step runs
    tt = torch.from_numpy(before["theta_m"].copy()).cuda()
    assert lib().hexdyn_import_field(d.handle, capi.FIELD_ID["THETA_M"], ct.c_void_p(tt.data_ptr()),
                                     ct.c_void_p(d.stream_ptr())) == 0
    d.step_device(1)


def test_determinism_and_restart(get_case):
    print("[gpu] determinism and restart", flush=True)
    case = get_case("x1.2562-moist")
    a = _driver(case)
    a.step_device(3)
    sa = a.get_state()
    b = _driver(case)
    b.step_device(1)
    mid = b.get_state()
    from hexdyn.driver import HexDycoreDriver

    c = HexDycoreDriver.from_host(case, state=mid, saved=mid)
    c.step_device(2)
    sc = c.get_state()
    b.step_device(2)
    sb = b.get_state()
    for k in sa:
        assert _bits_equal(sa[k], sb[k]), f"determinism {k}"
        assert _bits_equal(sa[k], sc[k]), f"restart {k}"


def test_fp64_integrals_match_host_sums_and_repeat(get_case):
    print("[gpu] FP64 integrals x1.2562-moist", flush=True)
    case = get_case("x1.2562-moist")
    d = _driver(case)
    st = d.get_state()
    a = d.integrals()
    assert a == d.integrals()  # fixed reduction order: identical bits
    m = case.mesh
    area = (1.0 / case.inv_area_cell.astype(np.float64))[None, :]
    dzw = (1.0 / case.grid.rdzw.astype(np.float64))[:, None]
    wgt = area * dzw
    rho = st["rho_zz"].astype(np.float64)
    assert abs(a["dry_mass"] / (wgt * rho).sum() - 1) < 1e-13
    assert abs(a["rho_theta"] / (wgt * st["rtheta_m"].astype(np.float64)).sum() - 1) < 1e-13
    dcdv = (m.dcEdge.astype(np.float32) * m.dvEdge.astype(np.float32)).astype(np.float64)
    u = st["u"].astype(np.float64)
    ke = np.zeros_like(rho)
    for s in range(m.max_edges):
        ok = s < m.nEdgesOnCell
        e = m.edgesOnCell[:, s]
        ke += np.where(ok[None, :], 0.25 * dcdv[e][None, :] * u[:, e] ** 2, 0.0)
    ke *= case.inv_area_cell.astype(np.float64)[None, :]
    qv = st["scalars"][0].astype(np.float64)
    temp = st["theta_m"].astype(np.float64) * st["exner"].astype(np.float64) / (1.0 + (461.6 / 287.0) * qv)
    zg = case.grid.zgrid.astype(np.float32).astype(np.float64)
    zmid = (0.5 * (zg[:-1] + zg[1:])).astype(np.float32).astype(np.float64)
    energy = (wgt * rho * ((1004.5 - 287.0) * temp + 9.80616 * zmid + ke)).sum()
    assert abs(a["total_energy"] / energy - 1) < 1e-12
    for s in range(case.n_scalars):
        ref = (wgt * rho * st["scalars"][s].astype(np.float64)).sum()
        assert abs(a[f"tracer_mass_{s}"] - ref) <= 1e-12 * abs(ref) + 1e-300
    # one step: dry and tracer mass conserved to binary32 rounding of the state
    d.step_device(1)
    b = d.integrals()
    assert abs(b["dry_mass"] / a["dry_mass"] - 1) < 1e-6
    for s in range(case.n_scalars):
        assert abs(b[f"tracer_mass_{s}"] / a[f"tracer_mass_{s}"] - 1) < 1e-5, s


def test_graph_replays_match_eager_steps(get_case):
    # two buffer layouts alternate, so steps 1-2 capture and 3-5 replay; eager
    # host work (state download) runs between replays
    print("[gpu] hipGraph replays vs eager x1.642-moist", flush=True)
    case = get_case("x1.642-moist")
    runs = {}
    for graphs in (True, False):
        d = _driver(case)
        d.use_graphs(graphs)
        states = []
        for _ in range(5):
            d.step_device(1)
            states.append(d.get_state())
        runs[graphs] = states
    for i, (g, e) in enumerate(zip(runs[True], runs[False])):
        for k in g:
            assert _bits_equal(g[k], e[k]), f"step {i + 1} {k}: {_diff(g[k], e[k])}"


def test_graph_cache_captures_once_per_layout(get_case):
    """The dynamics buffers return to their layout every 2 steps (one
    publish swap per step) and the scalar buffers every 3 (three stage swaps
    and a publish swap make a 3-cycle), so the layouts repeat every 6 steps:
    steps 1-6 capture one graph each and steps 7-12 replay them (the cache
    key is stable)."""
    print("[gpu] hipGraph cache x1.642-moist", flush=True)
    d = _driver(get_case("x1.642-moist"))
    d.step_device(6)
    assert d.graph_count() == 6
    d.step_device(6)
    assert d.graph_count() == 6


def test_restart_file_continues_bitwise(get_case, tmp_path):
    print("[gpu] restart file x1.642-moist", flush=True)
    case = get_case("x1.642-moist")
    a = _driver(case)
    a.step_device(3)
    ref = a.get_state()
    b = _driver(case)
    b.step_device(2)
    p = tmp_path / "restart.nc"
    b.write_restart(p, xtime="0000-01-01_00:24:00")
    c = _driver(case)
    meta = c.read_restart(p)
    assert meta["model_time_s"] == 2 * case.config.config_dt
    c.step_device(1)
    got = c.get_state()
    for k in ref:
        assert _bits_equal(ref[k], got[k]), f"{k}: {_diff(ref[k], got[k])}"


# Configurations that take the other branches of the fused whole-step
# sequence: more than two acoustic substeps (ru_avg stored and read back), one
# substep everywhere (the average taken from ru_p), one dynamics subcycle,
# no divergence damping, unlimited transport with the final clamp, the RK2
# schedule, and mixing without its fourth-order part.
STEP_VARIANTS = [
    dict(config_number_of_sub_steps=6),
    dict(config_number_of_sub_steps=1),
    dict(config_dynamics_split_steps=1),
    dict(config_divergence_damping=False),
    dict(config_monotonic=False),
    dict(config_time_integration_order=2),
    dict(config_horiz_mixing="2d_smagorinsky", config_visc4_2dsmag=0.0),
    dict(config_rayleigh_damp_u=True, config_number_rayleigh_damp_u_levels=8,
         config_rayleigh_damp_u_timescale_days=0.5),
    dict(config_horiz_mixing="2d_smagorinsky", config_mpas_cam_coef=0.2, config_number_cam_damping_levels=4),
]


def test_partial_mass_loading_bitwise(get_case):
    """physics_mass_loading_count below the carried species count
    (cuda_driver.py:5063-5068): 4 of 6 species load the air, all 6 are
    transported; 2 steps bit for bit, and qtot is the leading-4 sum."""
    import dataclasses

    print("[gpu] x1.642-moist, mass loading by 4 of 6 species, 2 steps", flush=True)
    case = dataclasses.replace(get_case("x1.642-moist"), n_moist=4)
    d = _driver(case)
    d.phase("begin_step")
    q = np.asarray(case.state.scalars, dtype=np.float32)
    t = np.zeros(q.shape[1:], dtype=np.float32)
    for s in range(4):
        t = t + q[s]
    assert _bits_equal(d.export_field("QTOT").cpu().numpy(), t)
    d.close()
    o = Oracle(case, 32)
    o.set_state(initial_state_arrays(case), rebuild=True)
    assert o.step(2) == 0
    d = _driver(case)
    d.step_device(2)
    ref, got = o.get_state(), d.get_state()
    for k in ref:
        assert _bits_equal(ref[k], got[k]), f"{k}: {_diff(ref[k], got[k])}"


@pytest.mark.parametrize("variant", STEP_VARIANTS, ids=lambda v: ",".join(f"{k[7:]}={x}" for k, x in v.items()))
def test_whole_step_variants_bitwise(get_case, variant):
    import dataclasses

    print(f"[gpu] x1.642-moist 2 steps with {variant}", flush=True)
    base = get_case("x1.642-moist")
    case = get_case("x1.642-moist", config=dataclasses.replace(base.config, **variant))
    o = Oracle(case, 32)
    o.set_state(initial_state_arrays(case), rebuild=True)
    assert o.step(2) == 0
    d = _driver(case)
    d.step_device(2)
    ref, got = o.get_state(), d.get_state()
    for k in ref:
        assert _bits_equal(ref[k], got[k]), f"{k}: {_diff(ref[k], got[k])}"


def test_unlimited_transport_with_held_scalar_tendency_bitwise(get_case):
    """config_monotonic off: all three transport stages take the unlimited
    form, each with the held scalar tendency; 2 whole steps bit for bit."""
    import dataclasses

    print("[gpu] x1.642-moist, unlimited transport with a held scalar tendency, 2 steps", flush=True)
    base = get_case("x1.642-moist")
    case = get_case("x1.642-moist", config=dataclasses.replace(base.config, config_monotonic=False))
    q = np.asarray(case.state.scalars, dtype=np.float32)
    src = ((q * np.random.default_rng(13).uniform(-0.3, 0.3, q.shape).astype(np.float32))
           / np.float32(3600.0)).astype(np.float32)
    o = Oracle(case, 32)
    o.set_state(initial_state_arrays(case), rebuild=True)
    o.set_physics(scalars=src)
    assert o.step(2) == 0
    d = _driver(case)
    d.set_physics_tendencies(scalars=src)
    d.step_device(2)
    ref, got = o.get_state(), d.get_state()
    for k in ref:
        assert _bits_equal(ref[k], got[k]), f"{k}: {_diff(ref[k], got[k])}"


def test_post_transport_handoff_bitwise(get_case):
    print("[gpu] unclamped post-transport handoff x1.642-moist, unlimited transport, 2 steps", flush=True)
    import dataclasses

    base = get_case("x1.642-moist")
    case = get_case("x1.642-moist", config=dataclasses.replace(base.config, config_monotonic=False))
    o = Oracle(case, 32)
    o.set_state(initial_state_arrays(case), rebuild=True)
    o.set_post_transport_clamp(False)
    assert o.step(2) == 0
    d = _driver(case)
    d.set_post_transport_clamp(False)
    d.step_device(2)
    ref, got = o.get_state(), d.get_state()
    assert (ref["scalars"] < 0).any()
    for k in ref:
        assert _bits_equal(ref[k], got[k]), f"{k}: {_diff(ref[k], got[k])}"


def test_day_long_run_x1_2562_dry_bitwise(get_case):
    """The CPU-runnable workload (x1.2562 dry, dt 1800 s) over 24 h: 48 steps,
    replayed as graphs on the GPU, bit for bit against the oracle."""
    print("[gpu] x1.2562-dry 24 h (48 steps)", flush=True)
    case = get_case("x1.2562-dry")
    o = Oracle(case, 32)
    o.set_state(initial_state_arrays(case), rebuild=True)
    assert o.step(48) == 0
    d = _driver(case)
    d.step_device(48)
    ref, got = o.get_state(), d.get_state()
    for k in ref:
        assert _bits_equal(ref[k], got[k]), f"{k}: {_diff(ref[k], got[k])}"


def test_day_long_headline_run_conserves_mass(get_case):
    """x1.40962 moist over 24 h (120 steps of 720 s): the validation flag never
    trips, dry mass and every tracer mass (FCT) hold to the rounding of the
    binary32 state, and no mixing ratio goes negative.  Integrals in FP64."""
    print("[gpu] x1.40962-moist 24 h (120 steps), FP64 budgets", flush=True)
    case = get_case("x1.40962-moist")
    d = _driver(case)
    a = d.integrals()
    d.step_device(120)
    b = d.integrals()
    # measured on MI355X: dry mass -2.1e-11, water vapour -2.6e-10, condensates ~ -6e-8
    assert abs(b["dry_mass"] / a["dry_mass"] - 1) < 1e-9
    for s in range(case.n_scalars):
        assert abs(b[f"tracer_mass_{s}"] / a[f"tracer_mass_{s}"] - 1) < 1e-6, s
    st = d.get_state()
    assert np.isfinite(st["rho_zz"]).all() and (st["scalars"] >= 0).all()


@pytest.mark.parametrize("public", [False, True])
def test_case_read_from_an_mpas_init_file_steps_bitwise(get_case, tmp_path, public):
    """A model-dump file (rho_zz, theta_m, ru, rw) and an init_atmosphere-style
    file (rho, theta, u, w: converted, w -> rw with the terrain terms)."""
    print(f"[gpu] case from an MPAS init file x1.642-moist (public fields: {public}), 2 steps", flush=True)
    from hexdyn import mpas_io

    case = get_case("x1.642-moist")
    p = tmp_path / "x1.642.init.nc"
    w = None
    if public:
        o0 = Oracle(case, 32)
        o0.set_state(initial_state_arrays(case), rebuild=True)
        w = o0.get_state()["w"]
    mpas_io.write_mpas_init(case, p, public_w=w)
    back = mpas_io.case_from_mpas(p, config=case.config, cold_start=public)
    o = Oracle(back, 32)
    o.set_state(initial_state_arrays(back), rebuild=True)
    assert o.step(2) == 0
    d = _driver(back)
    d.step_device(2)
    ref, got = o.get_state(), d.get_state()
    for k in ref:
        assert _bits_equal(ref[k], got[k]), f"{k}: {_diff(ref[k], got[k])}"


def test_phase_by_phase_bitwise_with_physics_tendencies(get_case):
    print("[gpu] phase walk with held physics tendencies x1.2562-moist + mixing", flush=True)
    case = _mixing(get_case, "x1.2562-moist")
    L, C, E = case.n_levels, case.mesh.n_cells, case.mesh.n_edges
    rng = np.random.default_rng(11)
    physics = {"rho": (1e-9 * rng.standard_normal((L, C))).astype(np.float32),
               "rho_u": (1e-6 * rng.standard_normal((L, E))).astype(np.float32),
               "rho_theta": (1e-6 * rng.standard_normal((L, C))).astype(np.float32)}
    # a held scalar tendency that pushes some mixing ratios negative before the limiter
    q = np.asarray(case.state.scalars, dtype=np.float32)
    physics["scalars"] = ((q * rng.uniform(-0.5, 0.5, q.shape).astype(np.float32)) / np.float32(3600.0)).astype(
        np.float32)
    bad = _phase_walk(case, physics)
    assert not bad, "\n".join(bad[:20])


def test_phase_by_phase_bitwise_nonzero_reference_wind(get_case):
    """A non-zero u_init/v_init profile: the perturbation-Coriolis term
    (neighbour angle, target f) is live in every stage's momentum tendency."""
    print("[gpu] phase walk x1.642-moist with reference wind (12, -7) m/s", flush=True)
    case = get_case("x1.642-moist", reference_wind=(12.0, -7.0))
    assert np.any(case.u_init) and np.any(case.v_init)
    bad = _phase_walk(case)
    assert not bad, "\n".join(bad[:20])


def test_phase_by_phase_bitwise_upper_damping(get_case):
    """Rayleigh damping of u (8 levels, half a day) and the CAM kdiff floor
    (4 levels) with 2-D Smagorinsky mixing, phase by phase."""
    import dataclasses

    print("[gpu] phase walk x1.642-moist with Rayleigh u damping and the CAM floor", flush=True)
    base = get_case("x1.642-moist")
    cfg = dataclasses.replace(base.config, config_horiz_mixing="2d_smagorinsky", config_mpas_cam_coef=0.2,
                              config_number_cam_damping_levels=4, config_rayleigh_damp_u=True,
                              config_number_rayleigh_damp_u_levels=8, config_rayleigh_damp_u_timescale_days=0.5)
    bad = _phase_walk(get_case("x1.642-moist", config=cfg))
    assert not bad, "\n".join(bad[:20])


def test_variable_mesh_density_mixing_bitwise(get_case):
    """A variable meshDensity in [1, 4]: del2/del4 scaled per edge; 2 steps
    with mixing bit for bit."""
    import copy
    import dataclasses
    import sys
    from pathlib import Path

    sys.path.insert(0, str(Path(__file__).resolve().parent / "golden"))
    from reference_walk import mixing_density

    print("[gpu] x1.642-moist variable mesh density, mixing, 2 steps", flush=True)
    base = _mixing(get_case, "x1.642-moist")
    mesh = copy.deepcopy(base.mesh)
    mesh.arrays["meshDensity"] = mixing_density(mesh)
    case = dataclasses.replace(base, mesh=mesh)
    o = Oracle(case, 32)
    o.set_state(initial_state_arrays(case), rebuild=True)
    assert o.step(2) == 0
    d = _driver(case)
    d.step_device(2)
    ref, got = o.get_state(), d.get_state()
    for k in ref:
        assert _bits_equal(ref[k], got[k]), f"{k}: {_diff(ref[k], got[k])}"


def test_passive_tracers_clamped_without_moisture_bitwise(get_case):
    """n_moist = 0 with six carried species, unlimited transport and negative
    patches: the end-of-step clamp of every species, 2 steps bit for bit."""
    import dataclasses

    print("[gpu] x1.642 passive tracers, unlimited transport, 2 steps", flush=True)
    base = get_case("x1.642-moist")
    case = dataclasses.replace(base, n_moist=0, config=dataclasses.replace(base.config, config_monotonic=False))
    st = initial_state_arrays(case)
    q = st["scalars"].copy()
    q[1] = (q[1] - np.float32(2e-6)).astype(np.float32)
    st["scalars"] = q
    o = Oracle(case, 32)
    o.set_state(st, rebuild=True)
    assert o.step(2) == 0
    from hexdyn.driver import HexDycoreDriver

    d = HexDycoreDriver.from_host(case, state=st)
    d.step_device(2)
    ref, got = o.get_state(), d.get_state()
    for k in ref:
        assert _bits_equal(ref[k], got[k]), f"{k}: {_diff(ref[k], got[k])}"
    assert (got["scalars"] >= 0).all()


def test_cells_on_cell_out_of_edge_order_bitwise(get_case):
    """cellsOnCell rotated one slot against edgesOnCell in every cell (a
    table order MPAS files do not use, so slot s no longer names the cell
    across edge s): the FCT cell pass then reads each edge's other cell on
    its own, and the limiter bounds keep the given order; 2 moist steps bit
    for bit."""
    import copy
    import dataclasses

    print("[gpu] x1.642-moist cellsOnCell rotated one slot, 2 steps", flush=True)
    base = get_case("x1.642-moist")
    assert base.config.config_monotonic
    mesh = copy.deepcopy(base.mesh)
    coc = mesh.arrays["cellsOnCell"].copy()
    n = mesh.arrays["nEdgesOnCell"]
    for c in range(coc.shape[0]):
        coc[c, : n[c]] = np.roll(coc[c, : n[c]], 1)
    mesh.arrays["cellsOnCell"] = coc
    case = dataclasses.replace(base, mesh=mesh)
    o = Oracle(case, 32)
    o.set_state(initial_state_arrays(case), rebuild=True)
    assert o.step(2) == 0
    d = _driver(case)
    d.step_device(2)
    ref, got = o.get_state(), d.get_state()
    for k in ref:
        assert _bits_equal(ref[k], got[k]), f"{k}: {_diff(ref[k], got[k])}"


@pytest.mark.parametrize("name,nlev,species", [("x1.162-moist", 10, 0), ("x1.162-moist", 55, 1), ("r642-moist", 26, 3),
                                               ("x1.642-moist", 63, 8)])
def test_state_transfer_round_trips_bitwise(get_case, name, nlev, species):
    """Every field set from host arrays comes back word for word (entity
    counts that end in part of a 64-entity tile, the shortest and the longest
    rows, several species planes), and a field exported and imported again is
    unchanged."""
    import ctypes as ct

    from hexdyn import capi
    from hexdyn.lib import lib

    print(f"[gpu] state round trip {name} L{nlev} T{species}", flush=True)
    case = get_case(name, nlev=nlev, n_scalars=species, moist=species > 0)
    d = _driver(case)
    rng = np.random.default_rng(3)
    state = {k: rng.uniform(0.5, 2.0, shape).astype(np.float32) for k, shape in d.shapes.items()}
    d.set_state(state, saved=state)
    got = d.get_state()
    for k, v in state.items():
        assert _bits_equal(v, got[k]), k
    for name_f in ("RU", "W", "EXNER") + (("SCALARS",) if species else ()):
        t = d.export_field(name_f)
        rc = lib().hexdyn_import_field(d.handle, capi.FIELD_ID[name_f], ct.c_void_p(t.data_ptr()),
                                       ct.c_void_p(d.stream_ptr()))
        assert rc == 0
        assert _bits_equal(t.cpu().numpy(), d.export_field(name_f).cpu().numpy()), name_f


@pytest.mark.parametrize("name,turn", [("x1.642-moist", 1), ("x1.642-moist", -1), ("r642-moist", 1)])
def test_other_vertex_slot_order_step_bitwise(get_case, name, turn):
    """verticesOnCell turned against edgesOnCell (MPAS files keep vertex slot
    s between edge slots s - 1 and s; in another order the vertices keep a
    pass of their own), with mixing: 2 steps bit for bit."""
    import copy
    import dataclasses

    print(f"[gpu] {name} verticesOnCell turned by {turn}, 2 steps", flush=True)
    base = _mixing(get_case, name)
    mesh = copy.deepcopy(base.mesh)
    n = mesh.arrays["nEdgesOnCell"]
    for table in ("verticesOnCell", "kiteForCell"):
        t = mesh.arrays[table].copy()
        for c in range(t.shape[0]):
            t[c, : n[c]] = np.roll(t[c, : n[c]], turn)
        mesh.arrays[table] = t
    case = dataclasses.replace(base, mesh=mesh)
    o = Oracle(case, 32)
    o.set_state(initial_state_arrays(case), rebuild=True)
    assert o.step(2) == 0
    d = _driver(case)
    d.step_device(2)
    ref, got = o.get_state(), d.get_state()
    for k in ref:
        assert _bits_equal(ref[k], got[k]), f"{k}: {_diff(ref[k], got[k])}"


@pytest.mark.parametrize("waves", [4, 16])
def test_paired_launches_bitwise(get_case, waves):
    """Passes that share a launch: at 16 wavefronts a block the 480 edges of
    x1.162 fill 30 blocks, which the launch rounds up to a multiple of the 8
    XCDs; the cells' blocks follow.  2 steps bit for bit."""
    from hexdyn import autotune

    print(f"[gpu] x1.162-moist mixing, {waves} wavefronts a block, 2 steps", flush=True)
    case = _mixing(get_case, "x1.162-moist")
    o = Oracle(case, 32)
    o.set_state(initial_state_arrays(case), rebuild=True)
    assert o.step(2) == 0
    d = _driver(case)
    autotune.set_launch(d, "*", waves)
    d.step_device(2)
    ref, got = o.get_state(), d.get_state()
    for k in ref:
        assert _bits_equal(ref[k], got[k]), f"{k}: {_diff(ref[k], got[k])}"


@pytest.mark.parametrize("scale", [1.0, 1e30])
def test_implicit_coefficients_out_of_reciprocal_range(get_case, scale):
    """Every third column with exner scaled so that the denominators of its
    implicit system leave the range of the corrected reciprocal (above
    2**100): those columns take the division.  Coefficients bit for bit."""
    print(f"[gpu] implicit coefficients x1.162-moist, exner x {scale:g} in every third column", flush=True)
    case = get_case("x1.162-moist")
    o = Oracle(case, 32)
    o.set_state(initial_state_arrays(case), rebuild=True)
    a = o.get_state()
    a["exner"][:, ::3] *= np.float32(scale)
    o.set_state(a, rebuild=False)
    d = _driver(case)
    d.set_state(a, saved=a)
    o.begin_step(); d.phase("begin_step")
    o.begin_subcycle(1); d.phase("begin_subcycle", 1)
    alpha = o.export_field("ALPHA_TRI")
    small = (alpha != 0.0) & (np.abs(alpha) < 2.0 ** -100)
    assert bool(small.any()) == (scale > 1.0) and np.isfinite(alpha).all()
    for f in ("A_TRI", "ALPHA_TRI", "GAMMA_TRI", "COFWZ", "COFWT", "COFTZ"):
        x, y = o.export_field(f), d.export_field(f).cpu().numpy()
        assert _bits_equal(x, y), f"{f}: {_diff(x, y)}"


@pytest.mark.parametrize("species", [0, 1, 6, 7, 13])
def test_integrals_by_species_count(get_case, species):
    """Species are summed in groups of six, cells in blocks of four (162
    leave the last block half empty): host sums in binary64."""
    print(f"[gpu] FP64 integrals x1.162, {species} species", flush=True)
    case = get_case("x1.162-moist", n_scalars=species, moist=species > 0)
    d = _driver(case)
    st, a = d.get_state(), d.integrals()
    wgt = (1.0 / case.inv_area_cell.astype(np.float64))[None, :] * (1.0 / case.grid.rdzw.astype(np.float64))[:, None]
    rho = st["rho_zz"].astype(np.float64)
    assert len(a) == 3 + species
    assert abs(a["dry_mass"] / (wgt * rho).sum() - 1) < 1e-13
    assert abs(a["rho_theta"] / (wgt * st["rtheta_m"].astype(np.float64)).sum() - 1) < 1e-13
    for s in range(species):
        ref = (wgt * rho * st["scalars"][s].astype(np.float64)).sum()
        assert abs(a[f"tracer_mass_{s}"] - ref) <= 1e-12 * abs(ref) + 1e-300


@pytest.mark.parametrize("by_phases", [False, True])
def test_step_after_a_flagged_one(get_case, by_phases):
    """A step whose validation flag was set (a negative rho*theta), refused by
    the whole step or left unpublished by its phases: the next whole step
    starts from a clear flag and gives the oracle's bits."""
    print(f"[gpu] x1.162-moist step after a flagged one, by phases {by_phases}", flush=True)
    case = get_case("x1.162-moist")
    good = initial_state_arrays(case)
    o = Oracle(case, 32)
    o.set_state(good, rebuild=True)
    assert o.step(2) == 0
    d = _driver(case)
    d.step_device(1)
    bad = dict(good, rtheta_m=-good["rtheta_m"])
    d.set_state(bad)
    if by_phases:
        d.phase("begin_step"); d.phase("begin_subcycle", 1); d.phase("dyn_tend", 1)
        d.phase("acoustic_substep", 1, 1); d.phase("divergence_damping", 1); d.phase("recover", 1)
    else:
        with pytest.raises(Exception, match="validation flag"):
            d.step_device(1)
    d.set_state(good)
    d.step_device(2)
    ref, got = o.get_state(), d.get_state()
    for k in ref:
        assert _bits_equal(ref[k], got[k]), f"{k}: {_diff(ref[k], got[k])}"


@pytest.mark.parametrize("counts", [[1], [0, 7, 0, 1029], [1 << 19, (1 << 19) + 1, 3], [2097149, 5, 2097152, 4194311, 1]])
def test_download_sizes(get_case, counts):
    """Host copies through the pinned staging: empty and tiny arrays, and
    arrays that end before, at and after a thread's share (2 MiB) and a half of
    the staging (8 MiB), into host arrays at odd offsets."""
    import ctypes as ct

    from hexdyn.lib import lib

    print(f"[gpu] download {counts}", flush=True)
    d = _driver(get_case("x1.162-moist"))
    gen = torch.Generator(device="cuda").manual_seed(5)
    dev = [torch.rand(n, device="cuda", generator=gen) for n in counts]
    host = [np.full(n + 3, -1.0, dtype=np.float32) for n in counts]
    n = len(counts)
    for _ in range(2):  # the second call finds the staging of the first
        rc = lib().hexdyn_download(
            d.handle, n, (ct.c_void_p * n)(*(h.ctypes.data + 4 for h in host)),
            (ct.c_void_p * n)(*(x.data_ptr() for x in dev)), (ct.c_int64 * n)(*counts), ct.c_void_p(d.stream_ptr()))
        assert rc == 0
        for h, x, m in zip(host, dev, counts):
            assert np.array_equal(h[1:1 + m], x.cpu().numpy()) and h[0] == -1.0 and (h[1 + m:] == -1.0).all()
            h[1:1 + m] = 0.0
    assert lib().hexdyn_download(d.handle, 1, (ct.c_void_p * 1)(None), (ct.c_void_p * 1)(dev[0].data_ptr()),
                                 (ct.c_int64 * 1)(1), ct.c_void_p(d.stream_ptr())) != 0


@pytest.mark.parametrize("device_checks", [False, True])
def test_state_arrays_in_any_memory_order(get_case, device_checks, monkeypatch):
    """Prognostic arrays in C, Fortran, sliced, reversed, read-only and
    binary64 form upload the same values, and the refusals name the first
    array that fails, checked on the host or on the device."""
    import hexdyn.driver as driver

    print(f"[gpu] state upload orders, device checks {device_checks}", flush=True)
    monkeypatch.setattr(driver, "_CHECK_ON_DEVICE", 1 if device_checks else 1 << 60)
    case = get_case("x1.162-moist")
    a = {k: np.ascontiguousarray(v) for k, v in initial_state_arrays(case).items()}
    d = _driver(case)
    ref = d.get_state()

    def sliced(x):
        big = np.zeros(tuple(2 * n for n in x.shape), dtype=x.dtype)
        big[tuple(slice(None, None, 2) for _ in x.shape)] = x
        return big[tuple(slice(None, None, 2) for _ in x.shape)]

    def read_only(x):
        y = np.asfortranarray(x)
        y.flags.writeable = False
        return y

    forms = [np.asfortranarray, sliced, lambda x: x[::-1].copy()[::-1], read_only, lambda x: x.astype(np.float64),
             lambda x: np.moveaxis(np.ascontiguousarray(np.moveaxis(x, 0, -1)), -1, 0)]
    for f in forms:
        d.set_state({k: f(v) for k, v in a.items()})
        got = d.get_state()
        for k in ref:
            assert _bits_equal(ref[k], got[k]), k
    for names, first in ((("ru",), "ru"), (("scalars", "rtheta_m"), "rtheta_m")):
        for value in (np.nan, np.inf, -np.inf):
            bad = {k: v.copy() for k, v in a.items()}
            for k in names:
                bad[k].reshape(-1)[-1] = value
            with pytest.raises(FloatingPointError, match=f"^{first} contains"):
                d.set_state(bad)
            with pytest.raises(FloatingPointError, match=f"^{first} contains"):  # before a later array's shape
                d.set_state(dict(bad, rw=a["rw"][:-1]) if first != "ru" else dict(bad, scalars=a["scalars"][:-1]))
    for value in (0.0, -1.0):
        bad = dict(a, rho_zz=a["rho_zz"].copy())
        bad["rho_zz"][3, 5] = value
        with pytest.raises(ValueError, match="strictly positive"):
            d.set_state(bad)
    with pytest.raises(ValueError, match="rw shape"):
        d.set_state(dict(a, rw=a["rw"][:-1]))
    got = d.get_state()  # refused states leave the driver's as it was
    for k in ref:
        assert _bits_equal(ref[k], got[k]), k


@pytest.mark.parametrize("species", [1, 2, 4, 7])
def test_species_batches_side_by_side_bitwise(get_case, species):
    """Small meshes run the transport passes with a grid row per batch of
    species (batches of 2, 3 and 6, the last one partly filled): 2 steps bit
    for bit, monotonic and not."""
    import dataclasses

    for mono in (True, False):
        print(f"[gpu] x1.162, {species} species, monotonic {mono}, 2 steps", flush=True)
        base = get_case("x1.162-moist", n_scalars=species, moist=True)
        case = get_case("x1.162-moist", config=dataclasses.replace(base.config, config_monotonic=mono),
                        n_scalars=species, moist=True)
        o = Oracle(case, 32)
        o.set_state(initial_state_arrays(case), rebuild=True)
        assert o.step(2) == 0
        d = _driver(case)
        d.step_device(2)
        ref, got = o.get_state(), d.get_state()
        for k in ref:
            assert _bits_equal(ref[k], got[k]), f"{k}: {_diff(ref[k], got[k])}"
        d.close()


@pytest.mark.parametrize("field,scale", [("exner", 1e37), ("exner", np.inf), ("w", np.inf), ("w", np.nan)])
def test_columns_that_are_not_finite(get_case, field, scale):
    """Every third column with a field scaled out of range at its upper half:
    the recurrences carry infinities and NaN to the levels the serial sweeps
    carry them to, and to no other column's (phases of a first stage, values
    equal with NaN where NaN is)."""
    print(f"[gpu] x1.162-moist, {field} x {scale} in every third column", flush=True)
    case = get_case("x1.162-moist")
    o = Oracle(case, 32)
    o.set_state(initial_state_arrays(case), rebuild=True)
    a = o.get_state()
    a[field][30:, ::3] = (a[field][30:, ::3] + np.float32(1e-3)) * np.float32(scale)
    o.set_state(a, rebuild=False)
    d = _driver(case)
    d.set_state(a, saved=a)
    o.begin_step(); d.phase("begin_step")
    o.begin_subcycle(1); d.phase("begin_subcycle", 1)
    o.dyn_tend(1); d.phase("dyn_tend", 1)
    o.acoustic_substep(1, 1); d.phase("acoustic_substep", 1, 1)
    seen = False
    for f in ("ALPHA_TRI", "GAMMA_TRI", "RW_P", "WW_AVG", "RHO_PP", "RTHETA_PP"):
        x, y = o.export_field(f), d.export_field(f).cpu().numpy().ravel()
        seen |= not np.isfinite(x).all()
        assert np.array_equal(x, y, equal_nan=True), f"{f}: {np.sum(~((x == y) | (np.isnan(x) & np.isnan(y))))} differ"
    assert seen or scale == 1e37


def _refused_by_phases(d):
    """A step by phases up to its first recovery, then its end, which refuses it."""
    d.phase("begin_step"); d.phase("begin_subcycle", 1); d.phase("dyn_tend", 1)
    d.phase("acoustic_substep", 1, 1); d.phase("divergence_damping", 1); d.phase("recover", 1)
    with pytest.raises(FloatingPointError, match="validation flag"):
        d.phase("end_step")


@pytest.mark.parametrize("by_phases", [False, True])
def test_a_refused_step_stays_refused(get_case, by_phases):
    """The end of a step asked for again after it was refused is refused again
    and publishes nothing, whether the whole step or its phases were refused;
    the next step is judged by its own flag."""
    print(f"[gpu] x1.162-moist end of a refused step, by phases {by_phases}", flush=True)
    case = get_case("x1.162-moist")
    good = initial_state_arrays(case)
    o = Oracle(case, 32)
    o.set_state(good, rebuild=True)
    assert o.step(1) == 0
    d = _driver(case)
    d.set_state(dict(good, rtheta_m=-good["rtheta_m"]))
    before, t = d.get_state(), d.model_time()
    if by_phases:
        _refused_by_phases(d)
    else:
        with pytest.raises(FloatingPointError, match="validation flag"):
            d.step_device(1)
    for _ in range(2):
        with pytest.raises(FloatingPointError, match="validation flag"):
            d.phase("end_step")
    assert d.model_time() == t
    got = d.get_state()
    for k in before:
        assert _bits_equal(before[k], got[k]), k
    d.set_state(good)
    d.step_device(1)
    ref, got = o.get_state(), d.get_state()
    for k in ref:
        assert _bits_equal(ref[k], got[k]), f"{k}: {_diff(ref[k], got[k])}"


@pytest.mark.parametrize("call", ["recover", "scalars"])
def test_step_after_a_phase_outside_a_step(get_case, call):
    """A phase called outside a step on fields that set the validation flag: the
    next whole step is judged by its own flag and gives the oracle's bits."""
    import ctypes as ct

    from hexdyn import capi
    from hexdyn.lib import lib

    print(f"[gpu] x1.162-moist, {call} outside a step, then a step", flush=True)
    case = get_case("x1.162-moist")
    good = initial_state_arrays(case)
    o = Oracle(case, 32)
    o.set_state(good, rebuild=True)
    assert o.step(1) == 0
    name, args = ("RHO_PP", (1,)) if call == "recover" else ("RHO_ZZ", (3,))

    def called_outside():
        d = _driver(case)
        d.step_device(1)
        t = torch.full_like(d.export_field(name), -1e6)
        assert lib().hexdyn_import_field(d.handle, capi.FIELD_ID[name], ct.c_void_p(t.data_ptr()),
                                         ct.c_void_p(d.stream_ptr())) == 0
        d.phase(call, *args)
        return d

    with pytest.raises(FloatingPointError, match="validation flag"):  # the flag is set
        called_outside().phase("end_step")
    d = called_outside()
    d.set_state(good)
    d.step_device(1)
    ref, got = o.get_state(), d.get_state()
    for k in ref:
        assert _bits_equal(ref[k], got[k]), f"{k}: {_diff(ref[k], got[k])}"


def test_download_behind_queued_work_leaves_the_cores_alone(get_case):
    """A download queued behind work on its stream waits for it without the
    threads that carry the pieces out: the process's CPU time stays near the one
    core that a synchronisation may take."""
    import ctypes as ct
    import time

    from hexdyn.lib import lib

    print("[gpu] download of 64 MiB behind queued matrix products", flush=True)
    d = _driver(get_case("x1.162-moist"))
    x = torch.rand(1 << 24, device="cuda")
    host = np.empty(x.numel(), dtype=np.float32)
    m = torch.rand(4096, 4096, device="cuda")

    def download():
        assert lib().hexdyn_download(d.handle, 1, (ct.c_void_p * 1)(host.ctypes.data), (ct.c_void_p * 1)(x.data_ptr()),
                                     (ct.c_int64 * 1)(x.numel()), ct.c_void_p(d.stream_ptr())) == 0

    download()
    torch.cuda.synchronize()
    for _ in range(400):
        m @ m
    w0, c0 = time.perf_counter(), time.process_time()
    download()
    wall, cpu = time.perf_counter() - w0, time.process_time() - c0
    print(f"[gpu] waited {wall:.3f} s, CPU time {cpu:.3f} s", flush=True)
    assert np.array_equal(host, x.cpu().numpy())
    assert wall > 0.05, "too little work queued"
    assert cpu < 2.5 * wall


@pytest.mark.parametrize("name,nlev,species", [("x1.162-moist", 10, 7), ("x1.642-moist", 63, 7), ("x1.2562-moist", 26, 4),
                                               ("x1.2562-moist", 55, 1)])
def test_single_fields_by_row_count(get_case, name, nlev, species):
    """A field alone goes a row at a time up to 4096 rows when exported and 8192 when
    imported and in tiles above (here 162 to 10 248): the values of the whole state."""
    import ctypes as ct

    from hexdyn import capi
    from hexdyn.lib import lib

    print(f"[gpu] fields alone {name} L{nlev} T{species}", flush=True)
    d = _driver(get_case(name, nlev=nlev, n_scalars=species, moist=True))
    rng = np.random.default_rng(11)
    first, second = ({k: rng.uniform(0.5, 2.0, s).astype(np.float32) for k, s in d.shapes.items()} for _ in range(2))
    d.set_state(first, saved=first)
    names = {k: k.upper() for k in d.shapes}
    for k, f in names.items():
        assert _bits_equal(first[k], d.export_field(f).cpu().numpy()), f
    for k, f in names.items():
        t = torch.from_numpy(second[k].reshape(-1, second[k].shape[-1])).cuda()
        assert lib().hexdyn_import_field(d.handle, capi.FIELD_ID[f], ct.c_void_p(t.data_ptr()),
                                         ct.c_void_p(d.stream_ptr())) == 0
    got = d.get_state()
    for k in names:
        assert _bits_equal(second[k], got[k]), k


@pytest.mark.parametrize("splits,substeps", [(1, 4), (3, 2)])
@pytest.mark.parametrize("field,scale", [("exner", 1e15), ("exner", 1e30), ("exner", np.inf), ("w", np.inf), ("w", np.nan)])
def test_whole_step_with_a_column_out_of_range(get_case, splits, substeps, field, scale):
    """One column with a field scaled out of range at its upper half, through the
    stages' whole column passes: their coefficients take the division (exner), the
    recurrences carry what is not finite, the step is refused as the oracle's is,
    and its working fields are the oracle's, NaN where NaN is."""
    import dataclasses

    print(f"[gpu] x1.2562-moist whole step, {splits} subcycles, {field} x {scale} in one column", flush=True)
    base = get_case("x1.2562-moist")
    case = get_case("x1.2562-moist", nlev=26, n_scalars=1, moist=True, config=dataclasses.replace(
        base.config, config_dt=600.0, config_dynamics_split_steps=splits, config_number_of_sub_steps=substeps))
    o = Oracle(case, 32)
    o.set_state(initial_state_arrays(case), rebuild=True)
    a = o.get_state()
    a[field][13:, 1234] = (a[field][13:, 1234] + np.float32(1e-3)) * np.float32(scale)
    o.set_state(a, rebuild=False)
    d = _driver(case)
    d.set_state(a, saved=a)
    assert o.step(1) != 0
    with pytest.raises(FloatingPointError, match="validation flag"):
        d.step_device(1)
    share = []
    for f in ("TEND_RU", "TEND_RT", "TEND_RW", "TEND_RHO", "RU_P", "RW_P", "RHO_PP", "RTHETA_PP", "RU_AVG", "WW_AVG",
              "ALPHA_TRI", "GAMMA_TRI", "COFWZ", "COFWT", "COFTZ", "EULER_RU", "EULER_RW"):
        y = d.export_field(f).cpu().numpy().ravel()
        x = np.asarray(o.export_field(f)).ravel()
        share.append(np.isfinite(x).mean())
        same = (x.view(np.uint32) == y.view(np.uint32)) | (np.isnan(x) & np.isnan(y))
        assert same.all(), f"{f}: {(~same).sum()} differ"
    assert 0.2 < min(share) < 1.0


@pytest.mark.parametrize("monotonic", [False, True])
def test_transport_phases_without_species(get_case, monotonic):
    """A host that runs the transport phases whatever the species count: on a dry
    case they are accepted and change nothing, a step by phases as the whole step."""
    import dataclasses

    print(f"[gpu] x1.162 dry, transport phases, monotonic {monotonic}", flush=True)
    base = get_case("x1.162-moist")
    case = get_case("x1.162-moist", n_scalars=0, moist=False,
                    config=dataclasses.replace(base.config, config_monotonic=monotonic))
    assert not _phase_walk(case)
    o = Oracle(case, 32)
    o.set_state(initial_state_arrays(case), rebuild=True)
    assert o.step(1) == 0
    d = _driver(case)
    for st in (1, 2, 3):
        d.phase("scalars", st)
    d.step_device(1)
    ref, got = o.get_state(), d.get_state()
    for k in ref:
        assert _bits_equal(ref[k], got[k]), f"{k}: {_diff(ref[k], got[k])}"

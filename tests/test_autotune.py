"""Launch shapes of the gather kernels (wavefronts per block) and the
autotuner: every shape gives the same bits; the tuner's choice is no slower
than the default over whole steps; refusals."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _bits(a, b):
    return np.array_equal(np.asarray(a).view(np.uint32), np.asarray(b).view(np.uint32))


def test_launch_shapes_give_the_same_bits(get_case):
    from hexdyn import autotune
    from hexdyn.config import DycoreConfig
    from hexdyn.driver import HexDycoreDriver

    print("[gpu] launch shapes x1.2562-moist", flush=True)
    case = get_case("x1.2562-moist", config=DycoreConfig(config_dt=1800.0, config_horiz_mixing="2d_smagorinsky"))
    runs = []
    # the last table sets the edge-flux pass's gather form explicitly (the
    # others run its edge-tiled form): both give the same bits
    for table in ({"*": 4}, {"*": 1}, {"*": 2}, {"*": 8}, {"*": 16},
                  {"*": 4, "k_diag_edge_flux": 16, "k_tend_mom_ac": 2, "k_sc_edge": 8}):
        d = HexDycoreDriver.from_host(case)
        for k, w in table.items():
            autotune.set_launch(d, k, w)
        d.step_device(2)
        runs.append(d.get_state())
        assert autotune.get_launch(d, "k_rec_cell") == table.get("k_rec_cell", table["*"])
        d.close()
    for r in runs[1:]:
        for k in runs[0]:
            assert _bits(r[k], runs[0][k]), k


def test_refusals(get_case):
    from hexdyn import autotune
    from hexdyn.driver import HexDycoreDriver

    d = HexDycoreDriver.from_host(get_case("x1.642-moist"))
    for k, w in (("k_vcoef", 2), ("k_ac_cell", 1), ("k_diag_edge_flux_t", 4), ("k_rec_cell", 3), ("k_rec_cell", 32),
                 ("notakernel", 2)):
        with pytest.raises(ValueError):
            autotune.set_launch(d, k, w)
    d.close()


def test_tuner_is_not_slower_and_keeps_bits(get_case, tmp_path, monkeypatch):
    from hexdyn import autotune
    from hexdyn.driver import HexDycoreDriver

    print("[gpu] autotune x1.2562-moist", flush=True)
    monkeypatch.setenv("HEXDYN_CACHE", str(tmp_path))
    case = get_case("x1.2562-moist")
    ref = HexDycoreDriver.from_host(case)
    ref.step_device(3)
    want = ref.get_state()
    ref.close()
    d = HexDycoreDriver.from_host(case)
    rec = autotune.tune(d, steps=1, check_steps=4)
    assert rec["tuned_ms_per_step"] <= rec["default_ms_per_step"] or rec["table"] == {}
    path = autotune.save(rec)
    assert path.exists()
    d.close()
    d2 = HexDycoreDriver.from_host(case)  # picks the stored table up at create
    assert d2.tuning is not None and d2.tuning["table"] == rec["table"]
    for k, w in rec["table"].items():
        assert autotune.get_launch(d2, k) == w
    d2.step_device(3)
    got = d2.get_state()
    d2.close()
    for k in want:
        assert _bits(got[k], want[k]), k


@pytest.mark.parametrize("name,waves", [("x1.2562-moist", 4), ("x1.10242-moist", 4), ("x1.40962-dry", 8)])
def test_default_launch_shapes(get_case, name, waves):
    """Three edge passes take larger blocks from 32 768 edges on; a reset sets
    every kernel alike, and the bits stay."""
    from hexdyn import autotune
    from hexdyn.driver import HexDycoreDriver

    print(f"[gpu] default launch shapes {name}", flush=True)
    runs = []
    for reset in (None, 4):
        d = HexDycoreDriver.from_host(get_case(name))
        if reset:
            autotune.set_launch(d, "*", reset)
        for k in ("k_tend_mom_ac", "k_sc_edge", "k_rec_edge"):
            assert autotune.get_launch(d, k) == (reset or waves)
        assert autotune.get_launch(d, "k_sub_edge") == 4
        d.step_device(1)
        runs.append(d.get_state())
        d.close()
    for k in runs[0]:
        assert _bits(runs[0][k], runs[1][k]), k


@pytest.mark.parametrize("name,waves", [("x1.10242-moist", 4), ("x1.40962-dry", 8)])
@pytest.mark.parametrize("picks_win", [False, True])
def test_tuner_is_judged_by_the_untuned_handle(get_case, tmp_path, monkeypatch, name, waves, picks_win):
    """The step that the tuner compares with runs every kernel at the shape of a
    handle without a table; picks that lose leave those shapes, here and in a
    later handle of the mesh; picks that win are the ones that differ from them."""
    from hexdyn import autotune
    from hexdyn.driver import HexDycoreDriver

    print(f"[gpu] tuner against the untuned handle {name}, picks win {picks_win}", flush=True)
    monkeypatch.setenv("HEXDYN_CACHE", str(tmp_path))
    passes = ("k_tend_mom_ac", "k_sc_edge", "k_rec_edge", "k_sub_edge")
    d = HexDycoreDriver.from_host(get_case(name))
    shapes = {k: autotune.get_launch(d, k) for k in passes}
    assert shapes == {**dict.fromkeys(passes, waves), "k_sub_edge": 4}
    seen = []

    def times(drv, steps):  # k_sub_edge is fastest at 16, k_rec_edge at 4, the others at their own shape
        w = autotune.get_launch(drv, "k_sub_edge")
        best = {**shapes, "k_sub_edge": 16, "k_rec_edge": 4}
        return {k: 1.0 + (w != best[k]) for k in passes}

    def step_ms(drv, steps):
        seen.append({k: autotune.get_launch(drv, k) for k in passes})
        return 1.0 if len(seen) == 1 else 0.5 if picks_win else 2.0

    monkeypatch.setattr(autotune, "_kernel_times", times)
    monkeypatch.setattr(autotune, "_step_ms", step_ms)
    rec = autotune.tune(d)
    assert seen[0] == shapes
    want = {"k_sub_edge": 16, **({"k_rec_edge": 4} if waves != 4 else {})}
    assert seen[1] == {**shapes, **want}
    assert rec["table"] == (want if picks_win else {})
    left = {**shapes, **rec["table"]}
    assert {k: autotune.get_launch(d, k) for k in passes} == left
    d.close()
    autotune.save(rec)
    d = HexDycoreDriver.from_host(get_case(name))
    assert d.tuning["table"] == rec["table"]
    assert {k: autotune.get_launch(d, k) for k in passes} == left
    d.close()

"""The step instances compiled for 1, 2, 4 and 8 worlds per wave (any dimensions, any State layout) and the rule that
picks the wave size, against the oracle bit for bit."""
import numpy as np
import pytest

from util import b2, leaf_mismatches, perturbed
import scene_defs

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _compare(model, state, settings, dt, launches, oracle, n_steps=1, pitch=None, nan_equal=False):
    dev, ref = b2.layout.to_device(state, "cuda", pitch), oracle.copy(state)
    for k in range(launches):
        b2.step_n_(model, dev, settings, dt, n_steps)
        for _ in range(n_steps):
            oracle.step_(model, ref, settings, dt)
        bad = leaf_mismatches(ref, b2.layout.to_host(dev), nan_equal)
        assert bad == [], f"launch {k + 1}: {bad[:4]}"
    return ref


@pytest.mark.parametrize("wpw", [1, 2, 4, 8])
@pytest.mark.parametrize("case", ["quad_41", "native", "joints", "pile", "full"])
def test_wave_instances_parity(oracle, monkeypatch, case, wpw):
    """Each wave size's instances, plain and not, single- and multi-step: 61 worlds (the last block partly filled
    except at 1 a wave) of the rig with an odd slot count, the rig on a native chain, every joint type (the general
    joint rows), box piles, and a State in the full fixture layout; stock settings, then the v2.3.1 revolute solver."""
    from dataclasses import replace
    monkeypatch.setenv("GOI_WORLDS_PER_WAVE", str(wpw))
    n, dt = 61, 1.0 / 60.0
    if case in ("quad_41", "native"):
        s, m, st, cfg = b2.scenes.make_config(4, n, edges="native" if case == "native" else "quad",
                                              capacity=41 if case == "quad_41" else None)
        dt = cfg.dt
    elif case == "full":
        cfg = b2.scenes.CONFIGS[4]
        s = b2.scenes.settings_for(cfg)
        m, one, pts = b2.scenes.build_world(cfg, s)
        st, dt = b2.scenes.place_worlds(cfg, m, one, pts, n), cfg.dt
    else:
        s, m, one = scene_defs.build_test_scene(case, iterations=(8, 3))
        st = perturbed(one, n)
    for settings in (s, replace(s, revolute_v24=False)):
        ref = _compare(m, st, settings, dt, 6, oracle)
        ref = _compare(m, ref, settings, dt, 2, oracle, n_steps=3)
        assert b2.last_launch()["worlds_per_wave"] == wpw


@pytest.mark.parametrize("n,slots", [(1, 40), (2047, 40), (2048, 40), (2049, 40), (4097, 40), (8193, 40), (16383, 40),
                                     (16384, 40), (16385, 40), (16384, 24), (16385, 24), (20000, 8), (40000, 12)])
def test_wave_size_rule(oracle, n, slots):
    """The smallest wave size whose blocks all fit the GPU at once (8 blocks a CU for the rig), the most resident one
    above that, up to 8 (a CU holds more rig worlds of 24 slots or fewer at 16 or 32 a wave); two steps at the edges of
    each range."""
    s, m, st, cfg = b2.scenes.make_config(4, min(n, 256), capacity=slots)
    idx = np.arange(n) % min(n, 256)
    st = b2.world.from_leaves([np.ascontiguousarray(x[idx]) for x in b2.world.leaves(st)])
    _compare(m, st, s, cfg.dt, 2, oracle)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    info = b2.last_launch()
    want = next((w for w in (1, 2, 4, 8) if -(-n // w) <= 8 * cus), 8)
    assert info["worlds_per_wave"] == want and info["blocks"] == -(-n // want), info


@pytest.mark.parametrize("wpw,case", [(8, "piles"), (4, "piles"), (8, "negzero"), (1, "negzero"), (2, "nan"),
                                      (1, "negpose"), (4, "negpose"), (8, "negpose")])
def test_solver_rows_beyond_the_lanes(oracle, monkeypatch, wpw, case):
    """Solve's rows in the lanes' registers and the cases that leave them: more touching contacts than a group's lanes
    hold (piles at 8 worlds a wave: 16 rows; some worlds have more, others fewer), a static body whose velocity or pose
    is -0 (x - 0 * P may turn it into +0, which the other lanes' rows must see: the velocity phase runs again, or the
    position phase on rows written from the registers), and a NaN that reaches the terrain."""
    monkeypatch.setenv("GOI_WORLDS_PER_WAVE", str(wpw))
    s, m, st, cfg = b2.scenes.make_config(5, 48)
    for _ in range(60):
        oracle.step_(m, st, s, cfg.dt)
    touching = np.asarray(st.contacts.touching).sum(1)
    assert touching.max() > 16 and touching.min() < 16
    if case == "negzero":
        st.bodies.v[:, 0] = np.float32(-0.0)
        st.bodies.w[:, 0] = np.float32(-0.0)
    elif case == "negpose":
        st = scene_defs.with_odd_static(st, case)
    elif case == "nan":
        st.bodies.v[1::7, 9, 1] = np.nan
    _compare(m, st, s, cfg.dt, 6, oracle, nan_equal=True)


@pytest.mark.parametrize("scene,slots,wpw", [(5, 128, 1), (5, 128, 2), (5, 128, 4), (5, 128, 8), (5, 20, 1), (5, 20, 8),
                                             (4, 40, 16), (4, 40, 32), (4, 3, 32), (4, 3, 4)])
def test_search_on_lane_groups(oracle, monkeypatch, scene, slots, wpw):
    """FindNewContacts on lane groups of 64 down to 2: several leaves of the static tree at once or a leaf in parts, more
    rows and non-static candidates than lanes and fewer, a first search that fills an empty contact list, later ones of
    every pair beside the contacts that exist, a full table (pairs dropped), a row whose fat box is NaN (it meets every
    leaf) and an inactive body."""
    monkeypatch.setenv("GOI_WORLDS_PER_WAVE", str(wpw))
    s, m, st, cfg = b2.scenes.make_config(scene, 37, capacity=slots)
    dev, ref = b2.layout.to_device(st, "cuda"), oracle.copy(st)
    for k in range(6):
        if k in (2, 4):
            ref = b2.layout.to_host(dev)
            ref.new_fixture[:] = 1
            if k == 4:
                ref.bodies.active[::5, 2] = 0
                ref.fixtures.fat[3::11, -1, 1] = np.nan
            dev = b2.layout.to_device(ref, "cuda")
        b2.step_(m, dev, s, cfg.dt)
        oracle.step_(m, ref, s, cfg.dt)
        bad = leaf_mismatches(ref, b2.layout.to_host(dev), True)
        assert bad == [], f"step {k + 1}: {bad[:4]}"
    live = (np.asarray(ref.contacts.pair) >= 0).sum(1)
    assert live.max() == slots if slots in (3, 20) else live.max() > 4


@pytest.mark.parametrize("wpw", [1, 2, 4, 8])
@pytest.mark.parametrize("kind,count", [("rigs", 6), ("anchored", 8), ("pairs", 8), ("mixed", 9)])
def test_jointed_islands(oracle, monkeypatch, kind, count, wpw):
    """Several islands with joints of their own: revolute rows in registers, islands side by side in levels (1 and 2 worlds
    a wave; more rows than lanes at 4 and 8), and row tiles with an island a lane (other joints, the v2.3.1 solver, too
    many rows). Then static bodies with -0 velocities or poses, and a NaN, where the rows must run one after another."""
    from dataclasses import replace
    monkeypatch.setenv("GOI_WORLDS_PER_WAVE", str(wpw))
    s, m, one = scene_defs.jointed_islands(kind, count)
    ref = perturbed(one, 29)
    for settings in (s, replace(s, revolute_v24=False)):
        ref = _compare(m, ref, settings, 0.02, 12, oracle)
        ref = _compare(m, ref, settings, 0.02, 2, oracle, n_steps=3)
        assert b2.last_launch()["worlds_per_wave"] == wpw
        assert int(np.asarray(ref.contacts.touching).sum(1).max()) >= 2
        for case in ("negzero", "negpose", "nan"):
            _compare(m, scene_defs.with_odd_static(oracle.copy(ref), case), settings, 0.02, 4, oracle, nan_equal=True)


@pytest.mark.parametrize("kind,n,v24", [("pairs", 256, True), ("rigs", 256, True), ("rigs", 256, False)])
def test_islands_do_not_add_up(kind, n, v24):
    """A world's islands are solved side by side, whatever their joints: six of them in a world take less than half of six
    times one (one after another they took most of it, at 300 / 30 iterations, where Solve is the step)."""
    def step_us(count):
        s, m, one = scene_defs.jointed_islands(kind, count, iterations=(300, 30), revolute_v24=v24)
        dev = b2.layout.to_device(perturbed(one, n), "cuda")
        for _ in range(8):
            b2.step_(m, dev, s, 0.02)
        times = []
        for _ in range(5):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(4):
                b2.step_(m, dev, s, 0.02)
            end.record()
            end.synchronize()
            times.append(start.elapsed_time(end) / 4 * 1000)
        return min(times)
    one, six = step_us(1), step_us(6)
    print(f"one island {one:.0f} us a step, six {six:.0f}")
    assert six < 3 * one, f"one island {one:.0f} us a step, six {six:.0f}"

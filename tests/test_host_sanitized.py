"""The step's own code on the CPU under AddressSanitizer and UBSan: the library's translation units compiled for
the host (GOI_HOST_BUILD: blocks and lanes run one after another, every workspace, row tile and State leaf an
exactly-sized heap block) step the same worlds as the oracle (also sanitized), and every State leaf is compared bit
for bit after every launch (tests/host_step). An out-of-bounds access or an undefined operation in the step stops
the run with its source line; a wrong result shows as a mismatch. This is where a device fault is localised: the
same code, the same scenario, on the CPU.

Covers the step for one world a wave and any State (k_step_waves<1>, one buffer per leaf), the general k_step (launches
with debug arrays, which are compared too), the fixed-dimension rig and island steps (packed States), goi_step_n and
goi_step_n_noalloc, the TOI and edge scenes and the island-heavy configuration. The host build runs one world per
one-lane block, so the lane-group exchanges it checks are those of groups of one lane, and a lane keeps up to 32 contact
and 8 joint rows in "registers"; the device's wider groups are covered by the GPU parity tests."""
import fcntl
import importlib
import os
import shutil
import struct
import subprocess
from pathlib import Path

import numpy as np
import pytest

from util import b2, negative_zero_kinematic, perturbed, wd
import scene_defs

_abi = importlib.import_module("getting-over-it-rl_amd.box2d._abi")

HOST = Path(__file__).resolve().parent / "host_step"
EXE = HOST / "_build" / "host_step"

I32, F32, U8 = np.int32, np.float32, np.uint8
DESC_DTYPES = dict(fixture_body=I32, shape_type=I32, radius=F32, count=I32, verts=F32, normals=F32, joint_type=I32,
                   joint_a=I32, joint_b=I32, local_anchor_a=F32, local_anchor_b=F32, local_axis_a=F32,
                   local_yaxis_a=F32, reference_angle=F32, pair_a=I32, pair_b=I32, fixture_slot=I32, static_fat=F32,
                   static_friction=F32, static_restitution=F32, body_type=I32, toi_bodies=U8, centroid=F32,
                   edge_flags=I32)


@pytest.fixture(scope="module")
def host_step():
    if shutil.which("g++") is None or shutil.which("make") is None:
        pytest.skip("g++ and make are needed for the host build")
    # one make at a time (parallel test workers share the build folder)
    EXE.parent.mkdir(parents=True, exist_ok=True)
    with open(EXE.parent / ".lock", "w") as lock:
        fcntl.flock(lock, fcntl.LOCK_EX)
        r = subprocess.run(["make", "-C", str(HOST), "-j4"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]
    return EXE


def write_scenario(path, model, state, settings, dt, steps, packed, actions=None):
    """The scenario file host_step reads (its header comment gives the format)."""
    B, R, J, C = wd.dims(state)
    n = np.asarray(state.bodies.type).shape[0]
    with open(path, "wb") as f:
        f.write(b"GOISCN02")
        f.write(struct.pack("<4i", model.fixture_body.shape[0], model.joint_type.shape[0], model.pair_a.shape[0],
                            0 if model.body_type is None else model.body_type.shape[0]))
        names = [name for name, _ in _abi.GoiModelDesc._fields_[4:]]
        assert sorted(names) == sorted(DESC_DTYPES)
        for name in names:
            a = getattr(model, name)
            if a is None:
                f.write(struct.pack("<q", -1))
                continue
            x = np.ascontiguousarray(np.asarray(a), dtype=DESC_DTYPES[name]).tobytes()
            f.write(struct.pack("<q", len(x)) + x)
        cs = bytes(settings.to_c())
        f.write(struct.pack("<i", len(cs)) + cs)
        f.write(np.float32(dt).tobytes())
        f.write(struct.pack("<9i", steps, n, B, R, J, C, C, int(packed), len(wd.LEAVES)))
        for (group, name, dt, _), leaf in zip(wd.LEAVES, wd.leaves(state)):
            a = np.ascontiguousarray(np.asarray(leaf))
            full = (f"{group}.{name}" if group else name).encode()
            per_world = int(np.prod(a.shape[1:], dtype=np.int64))
            kind = 1 if np.dtype(dt) == np.float32 else 0
            f.write(struct.pack("<i", len(full)) + full + struct.pack("<iqi", a.itemsize, per_world, kind) + a.tobytes())
        if actions is None:
            f.write(struct.pack("<i", -1) + np.float32(0).tobytes() * 2)
        else:
            f.write(struct.pack("<i", b2.scenes.MOTOR_JOINT) + np.float32(b2.scenes.MOTOR_GAIN).tobytes()
                    + np.float32(b2.scenes.MOTOR_TORQUE).tobytes())
            f.write(np.ascontiguousarray(actions, dtype=F32).tobytes())


def run(exe, scenario, mode, plant=False, poison="nan"):
    """host_step on a scenario file. Every launch first fills each block's LDS and the constraint and task rows with
    `poison` (host_shim.hpp): a quiet NaN by default, so that a read of a word the launch did not write shows as a
    mismatch instead of passing on a value an earlier launch left."""
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=1:halt_on_error=1",
               UBSAN_OPTIONS="print_stacktrace=1:halt_on_error=1", GOI_HOST_LAUNCH_LOG="1", GOI_HOST_POISON=poison)
    cmd = [str(exe), str(scenario), mode] + (["plant"] if plant else [])
    return subprocess.run(cmd, capture_output=True, text=True, env=env, timeout=600)


def check(r):
    assert r.returncode == 0 and "PASS" in r.stdout, (
        f"exit {r.returncode}\n{r.stdout[-1500:]}\n{r.stderr[-6000:]}")


def kernels(r):
    """The names of the step kernels a run launched, in order."""
    return [ln.split()[1] for ln in r.stderr.splitlines() if ln.startswith("launch ") and "k_step" in ln]


def config_case(k, n, steps, edges="quad", seed=7):
    s, m, st, cfg = b2.scenes.make_config(k, n, edges=edges)
    rng = np.random.default_rng(seed)
    acts = np.stack([b2.scenes.actions(rng, n) for _ in range(steps)])
    return m, st, s, cfg.dt, acts


@pytest.mark.parametrize("packed", [True, False], ids=["packed-rig", "per-leaf-waves"])
@pytest.mark.parametrize("edges", ["quad", "native"])
def test_config4_sanitized(host_step, tmp_path, packed, edges):
    """The benchmark rig (config 4) with actions: the packed State takes the fixed-dimension rig kernel, the State
    with one buffer per leaf the instance for one world a wave."""
    m, st, s, dt, acts = config_case(4, 256, 60, edges)
    p = tmp_path / "scn.bin"
    write_scenario(p, m, st, s, dt, 60, packed, acts)
    r = run(host_step, p, "step")
    check(r)
    assert "60 steps" in r.stdout
    ran = kernels(r)
    assert len(ran) == 60
    assert all(("k_step_fixed<kRig" if packed else "k_step_waves<kS") in k for k in ran), ran[:2]


@pytest.mark.parametrize("case,mode", [("rig", "step:debug"), ("native", "step_n:3:debug"), ("piles", "step:debug"),
                                       ("joints", "step:debug"), ("joints_v23", "noalloc:2:debug")])
def test_debug_launches_sanitized(host_step, tmp_path, case, mode):
    """Launches with every debug array take the general k_step; the arrays (islands, solve order, TOI traces, status) and
    the State equal the oracle's."""
    acts = None
    if case in ("rig", "native", "piles"):
        k, n, steps = (5, 6, 45) if case == "piles" else (4, 32, 30)
        m, st, s, dt, acts = config_case(k, n, steps, "native" if case == "native" else "quad")
        acts = acts if mode == "step:debug" else None
    else:
        s, m, one = scene_defs.build_test_scene(case, iterations=(8, 3))
        st, dt, steps = perturbed(one, 12), 1.0 / 60.0, 40
    p = tmp_path / "scn.bin"
    write_scenario(p, m, st, s, dt, steps, False, acts)
    r = run(host_step, p, mode)
    check(r)
    ran = kernels(r)
    assert ran and all(k.startswith(("k_step<", "(k_step<")) for k in ran), ran[:2]


@pytest.mark.parametrize("n", [4093, 4500])
def test_block_order_many_chunks(host_step, tmp_path, n):
    """k_group_order with as many chunks a lane as it keeps classes of (16: 4,093 worlds in blocks of one, 512 or 511 to
    an XCD, 32 to a chunk) and more (18), on event counts and then on block times; a block left out or run twice shows."""
    m, st, s, dt, acts = config_case(4, n, 2)
    p = tmp_path / "scn.bin"
    write_scenario(p, m, st, s, dt, 2, True, acts)
    r = run(host_step, p, "step")
    check(r)
    assert "k_group_order" in r.stderr


@pytest.mark.parametrize("poison", ["8", "-1", "0"])
def test_poisoned_scratch_sanitized(host_step, tmp_path, poison):
    """The benchmark rig (packed: the fixed instance), the instance for one world a wave and the general k_step with the
    LDS workspaces and rows filled with small integers instead of NaN before every launch (8 as a body or slot index, -1
    as an empty slot, 0): the same results, so no pass reads a word its launch has not written."""
    m, st, s, dt, acts = config_case(4, 64, 30)
    for packed, mode in ((True, "step"), (False, "step"), (False, "step:debug")):
        p = tmp_path / f"scn{int(packed)}.bin"
        write_scenario(p, m, st, s, dt, 30, packed, acts)
        check(run(host_step, p, mode, poison=poison))


def nonfinite_case(n=64, steps=30, seed=7):
    """Config 4 with non-finite values written into a few worlds (the failure inputs of the reference's bench,
    bench_gpu.py:135-136): a NaN linear velocity (world 3), an infinite angular velocity (5), a NaN position (7), a
    velocity of 1e30 m/s (9: the max-translation clamp scales it by 2 / inf = 0) and a NaN force (11); the other
    worlds are untouched."""
    m, st, s, dt, acts = config_case(4, n, steps, seed=seed)
    bd = st.bodies
    bd.v[3, 1, 0] = np.nan
    bd.w[5, 4] = np.inf
    bd.c[7, 2, 1] = np.nan
    bd.v[9, 3] = (1e30, -1e30)
    bd.force[11, 1, 1] = np.nan
    return m, st, s, dt, acts


def test_nonfinite_worlds_sanitized(host_step, tmp_path):
    """NaN and infinite body values step without an out-of-bounds access or undefined operation in either the
    library's step or the oracle, to the same bits (both run here on the same float hardware), on the rig instance,
    the instance for one world a wave and the general k_step."""
    m, st, s, dt, acts = nonfinite_case()
    for packed, mode in ((True, "step"), (False, "step"), (False, "step:debug")):
        p = tmp_path / f"scn{int(packed)}.bin"
        write_scenario(p, m, st, s, dt, 30, packed, acts)
        check(run(host_step, p, mode))


def nonfinite_islands_case(oracle, n=8, clean=50):
    """Config 5 after `clean` steps on the oracle (its worlds then hold 1 to 11 awake islands), with non-finite values
    written into one island of a few worlds: a NaN linear velocity of a box (world 1), an infinite angular velocity
    (world 3) and a NaN force (world 5). In Box2D's order a non-finite impulse reaches the terrain's velocity
    (v - 0 * P) and from there the world's other islands; the library, whose lanes solve a world's rows side by
    side where they share no moving body, must then solve that world's rows one after another to give the same bits."""
    s, m, st, cfg = b2.scenes.make_config(5, n)
    for _ in range(clean):
        oracle.step_(m, st, s, cfg.dt)
    bd = st.bodies
    bd.v[1, 10, 0] = np.nan
    bd.w[3, 12] = np.inf
    bd.force[5, 8, 1] = np.nan
    return m, st, s, cfg.dt


def test_nonfinite_islands_sanitized(host_step, tmp_path, oracle):
    """Worlds of several islands with non-finite values in one of them step to the oracle's bits, on the island
    instance, the instance for one world a wave and the general k_step."""
    m, st, s, dt = nonfinite_islands_case(oracle)
    for packed, mode in ((True, "step"), (False, "step"), (False, "step:debug")):
        p = tmp_path / f"scn{int(packed)}.bin"
        write_scenario(p, m, st, s, dt, 20, packed)
        check(run(host_step, p, mode))


@pytest.mark.parametrize("k,case", [(4, "negpose"), (5, "negpose"), (5, "negzero")])
def test_static_negative_zero_sanitized(host_step, tmp_path, oracle, k, case):
    """A terrain body whose pose or velocity is -0 (x - 0 * P may turn it into +0, which the rows after it see): the
    velocity or the position phase runs again row after row, on the fixed instances and the one for any State."""
    s, m, st, cfg = b2.scenes.make_config(k, 16)
    for _ in range(40 if k == 5 else 10):
        oracle.step_(m, st, s, cfg.dt)
    st = scene_defs.with_odd_static(st, case)
    for packed in (True, False):
        p = tmp_path / f"scn{int(packed)}.bin"
        write_scenario(p, m, st, s, cfg.dt, 8, packed)
        check(run(host_step, p, "step"))


@pytest.mark.parametrize("v24", [True, False])
@pytest.mark.parametrize("kind,count", [("rigs", 2), ("rigs", 6), ("anchored", 4), ("pairs", 8), ("mixed", 9)])
def test_jointed_islands_sanitized(host_step, tmp_path, oracle, kind, count, v24):
    """Several islands with joints of their own: revolute rows in registers (up to 8 joints on the host's one lane) or the
    islands one by one from the row tiles; then static bodies with -0 velocities or poses, and a NaN."""
    from dataclasses import replace
    s, m, one = scene_defs.jointed_islands(kind, count)
    s, st = replace(s, revolute_v24=v24), perturbed(one, 8)
    p = tmp_path / "scn.bin"
    write_scenario(p, m, st, s, 0.02, 25, False)
    check(run(host_step, p, "step"))
    for _ in range(15):
        oracle.step_(m, st, s, np.float32(0.02))
    for case in ("negzero", "negpose", "nan"):
        write_scenario(p, m, scene_defs.with_odd_static(oracle.copy(st), case), s, 0.02, 6, False)
        check(run(host_step, p, "step"))


@pytest.mark.parametrize("dt", [0.0, -0.02])
def test_non_positive_dt_sanitized(host_step, tmp_path, dt):
    """dt <= 0: Solve still runs (step.py:35-40) and SolveTOI is skipped (toi.py:841); inv_dt0 keeps its value."""
    m, st, s, _, acts = config_case(4, 64, 6)
    p = tmp_path / "scn.bin"
    write_scenario(p, m, st, s, dt, 6, True, acts)
    r = run(host_step, p, "step")
    check(r)
    assert "events 0" in r.stdout


@pytest.mark.parametrize("max_events", [1, 2, 3])
def test_max_events_sanitized(host_step, tmp_path, max_events):
    """SolveTOI stopped after max_events events per step (toi.py:838-842), on the rig instance."""
    from dataclasses import replace
    m, st, s, dt, acts = config_case(4, 64, 30)
    p = tmp_path / "scn.bin"
    write_scenario(p, m, st, replace(s, max_events=max_events), dt, 30, True, acts)
    check(run(host_step, p, "step"))


@pytest.mark.parametrize("capacity", [6, 10])
def test_contact_table_overflow_sanitized(host_step, tmp_path, capacity):
    """Config 4 with 6 or 10 contact slots a world: FindNewContacts drops pairs (overflow > 0 in many worlds) and
    those worlds keep full candidate searches; the instance for any State (the fixed rig instance needs 40 slots)."""
    s, m, st, cfg = b2.scenes.make_config(4, 64, capacity=capacity)
    rng = np.random.default_rng(31)
    acts = np.stack([b2.scenes.actions(rng, 64) for _ in range(40)])
    p = tmp_path / "scn.bin"
    write_scenario(p, m, st, s, cfg.dt, 40, True, acts)
    r = run(host_step, p, "step")
    check(r)
    assert "overflow" in r.stdout and "overflow 0 " not in r.stdout, r.stdout[-500:]


@pytest.mark.parametrize("mode", ["step_n:4", "noalloc:5"])
def test_multi_step_launches_sanitized(host_step, tmp_path, mode):
    """goi_step_n and goi_step_n_noalloc on the rig's packed State (no actions between the steps of a launch)."""
    m, st, s, dt, _ = config_case(4, 64, 24)
    p = tmp_path / "scn.bin"
    write_scenario(p, m, st, s, dt, 24, True)
    check(run(host_step, p, mode))


@pytest.mark.parametrize("packed", [True, False], ids=["packed-island", "per-leaf-waves"])
def test_config5_sanitized(host_step, tmp_path, packed):
    """Config 5's box piles: 128 contact slots a world, large islands. The packed State takes the instance compiled
    for these dimensions, one buffer per leaf the instance for one world a wave."""
    m, st, s, dt, _ = config_case(5, 8, 60)
    p = tmp_path / "scn.bin"
    write_scenario(p, m, st, s, dt, 60, packed)
    r = run(host_step, p, "step")
    check(r)
    ran = kernels(r)
    assert len(ran) == 60 and all(("k_step_fixed<kIsland" if packed else "k_step_waves<kS") in k for k in ran), ran[:2]


@pytest.mark.parametrize("name", ["pile", "joints", "joints_v23", "misc", "hammer_chain", "multi_event",
                                  "island_walk", "toi_tie", "edges", "poly_angles", "ball_wall", "stock_bullets",
                                  "toi_plank_bullet"])
def test_scenes_sanitized(host_step, tmp_path, name):
    """The test scenes, a few perturbed copies each: every shape pair, joint type, TOI path and edge case."""
    s, m, st = scene_defs.build_test_scene(name, iterations=(8, 3))
    p = tmp_path / "scn.bin"
    write_scenario(p, m, perturbed(st, 16), s, 1.0 / 60.0, 90, False)
    check(run(host_step, p, "step"))


def test_negative_zero_kinematic_sanitized(host_step, tmp_path):
    """TOI events against a kinematic wall that starts at x = -0 (a side without mass in the TOI position passes).
    b2Sweep::Advance turns a resting -0 coordinate into +0 (c0 + beta * (c - c0) with c - c0 = +0) before the passes
    see it; the -0 until then, and the +0 after, follow the oracle."""
    s, m, st = scene_defs.build_test_scene("kinematic_wall", iterations=(8, 3))
    st = negative_zero_kinematic(perturbed(st, 16))
    assert np.signbit(st.bodies.c[:, 0, 0]).all()
    p = tmp_path / "scn.bin"
    write_scenario(p, m, st, s, 1.0 / 60.0, 40, False)
    check(run(host_step, p, "step"))


def test_planted_mismatch_is_reported(host_step, tmp_path):
    """One ulp moved in the oracle's input alone must end the run with a mismatch (the comparison is live)."""
    m, st, s, dt, acts = config_case(4, 8, 3)
    p = tmp_path / "scn.bin"
    write_scenario(p, m, st, s, dt, 3, True, acts)
    r = run(host_step, p, "step", plant=True)
    assert r.returncode == 1 and "MISMATCH after step 1" in r.stdout, r.stdout + r.stderr[-3000:]


@pytest.mark.parametrize("case", ["config4", "joints", "circles"])
def test_full_layout_state_sanitized(host_step, tmp_path, case):
    """States in the full fixture layout (a row per fixture, as WorldDef.build returns them) with the compact Model:
    the step addresses the non-static rows at their fixtures' rows and leaves the static rows alone. config4's
    non-static fixtures are the last rows; in "joints" and "circles" static fixtures sit between them."""
    if case == "config4":
        s, m, st, cfg = b2.scenes.make_config(4, 32)
        st, dt, steps = wd.expand_state(m, st), cfg.dt, 40
        rng = np.random.default_rng(5)
        acts = np.stack([b2.scenes.actions(rng, 32) for _ in range(steps)])
    else:
        s, m, st = scene_defs.build_test_scene(case, iterations=(8, 3))
        st, dt, steps, acts = wd.expand_state(m, perturbed(st, 16)), 1.0 / 60.0, 60, None
    B, R, J, C = wd.dims(st)
    assert R == m.fixture_body.shape[0] > int((np.asarray(m.fixture_slot) >= 0).sum())
    p = tmp_path / "scn.bin"
    write_scenario(p, m, st, s, dt, steps, True, acts)
    r = run(host_step, p, "step")
    check(r)
    ran = kernels(r)
    assert ran and all("k_step_waves<kS" in k for k in ran), ran[:2]

"""GPU tests of the sweeps ordered by data: one launch runs all velocity
iterations and one all position iterations, each constraint waiting for its
bodies' earlier updates (b2g_flow.h). Every body sees the same updates in the
same order as with a launch per colour, so every state compares bit for bit:
against a launch per colour (B2G_OPT_SWEEPS 1), and with the launches'
workgroups made to give up their places, so that one workgroup does all
sweeps (2).
"""
import sys

import numpy as np
import pytest

from util import GOLDEN, load_pkg, scene_for

pytestmark = pytest.mark.gpu
S = load_pkg().scenes
sys.path.insert(0, GOLDEN)


def _motors(n=70):
    """Jointed pairs with limits and motors over a kinematic and a static body, some in contact."""
    s = S.small_mixed(seed=3, n=20)
    lift = s.add_body(S.KINEMATIC, 6.0, 2.0, 0.0, 0.3, 0.1, 0.2)
    s.add_box(lift, 1.5, 0.2)
    prev = lift
    for i in range(n):
        b = s.add_body(S.DYNAMIC, 6.0 + 0.4 * i, 3.0 + 0.02 * (i % 3))
        s.add_box(b, 0.25, 0.1)
        s.add_revolute(prev, b, (5.9 + 0.4 * i, 3.0), collide_connected=i % 4 == 0,
                       limit=(-0.3, 0.4) if i % 3 == 0 else None, motor=(2.0, 30.0) if i % 5 == 0 else None)
        prev = b if i % 7 else lift if i % 2 else 0
    return s


def _pendulums(single, double):
    """Pendulums apart from each other, every anchor on the static body 0, the last `double` with a second link."""
    s = S.Scene(name="pendulums", gravity=(0.0, -10.0))
    s.add_body(S.STATIC, 0.0, 0.0)
    at = [(4.0 * (i % 250), 5.0 * (i // 250)) for i in range(single + double)]
    for x, y in at:
        s.add_box(s.add_body(S.DYNAMIC, x + 0.5, y), 0.4, 0.1)
    for x, y in at[single:]:
        s.add_box(s.add_body(S.DYNAMIC, x + 1.5, y), 0.4, 0.1)
    for i, (x, y) in enumerate(at):
        s.add_revolute(0, 1 + i, (x, y))
    for i, (x, y) in enumerate(at[single:]):
        s.add_revolute(1 + single + i, 1 + single + double + i, (x + 1.0, y))
    return s


def _sleepers():
    import make_golden
    return make_golden.sleep_scene()


CASES = {
    # scenes, steps, velocity and position iterations, warm starting, sleeping
    "one_box": ([lambda: S.pyramid(1)], 40, 8, 3, True, False),
    "pyramid": ([lambda: S.pyramid(20)], 60, 8, 3, True, False),
    "pyramid_cold": ([lambda: S.pyramid(12)], 30, 8, 3, False, False),
    "pile": ([lambda: S.random_pile(3001, seed=5, half_w=30.0, height=80.0)], 90, 8, 3, True, False),
    "chain": ([lambda: scene_for("chain")[0]], 60, 8, 3, True, False),
    "motors": ([_motors], 90, 8, 3, True, False),
    "motors_many_iterations": ([_motors], 40, 13, 7, True, False),
    "motors_no_iterations": ([_motors], 10, 0, 0, True, False),
    "gas_chains": ([lambda: S.gas_and_chains(4000, 16, 30, seed=0x5C3, half=80.0)], 30, 8, 3, True, False),
    "worlds_with_joints": ([lambda: S.gas_and_chains(300, 4, 9, seed=1, half=25.0), _motors,
                            lambda: S.random_pile(200, seed=2, half_w=9.0, height=30.0)], 50, 8, 3, True, False),
    # more joints on one static body than a byte counts; the first second link shares a wavefront with its anchor
    "pendulums_two_to_a_wave": ([lambda: _pendulums(1200, 1)], 40, 8, 3, True, False),
    "pendulums_64_to_a_wave": ([lambda: _pendulums(64990, 10)], 10, 8, 3, True, False),
    "sleep": ([_sleepers], 200, 8, 3, True, True),
    "sleep_joints": ([lambda: S.gas_and_chains(300, 6, 12, seed=7, half=40.0)], 120, 8, 3, True, True),
}


@pytest.mark.parametrize("name", list(CASES))
def test_gpu_sweeps_ordered_by_data_equal_a_launch_per_colour(engine, name):
    scenes, steps, vi, pi, warm, sleep = CASES[name]
    made = [f() for f in scenes]
    batches = []
    for mode in (1, 0, 2):
        b = engine.Batch.from_scenes(made)
        b.set_option(engine.OPT_SOLVER, engine.SOLVER_COLOURS)
        b.set_option(engine.OPT_SWEEPS, mode)
        batches.append(b)
    ordered = 0
    for k in range(0, steps, 10):
        for b in batches:
            b.advance(10, vi=vi, pi=pi, warm=[warm] * len(made), sleep=[sleep] * len(made))
        ordered += batches[1].get_option(engine.OPT_LAST_SWEEPS) == 2
        assert batches[0].get_option(engine.OPT_LAST_SWEEPS) == 1
        ref = batches[0]
        for mode, b in ((0, batches[1]), (2, batches[2])):
            assert np.array_equal(ref.bodies().view(np.uint8), b.bodies().view(np.uint8)), (k, mode, "bodies")
            assert np.array_equal(ref.contacts().view(np.uint8), b.contacts().view(np.uint8)), (k, mode, "contacts")
            nj = sum(s.joint_count for s in made)
            assert np.array_equal(ref.joints(nj).view(np.uint8), b.joints(nj).view(np.uint8)), (k, mode, "joints")
    assert ordered == steps // 10  # the default did order its sweeps by data
    for b in batches:
        b.close()


def test_gpu_sweeps_past_the_resident_limit_use_a_launch_per_colour(engine):
    """More constraints than the launch keeps resident: 512 workgroups of 256 lanes."""
    sc = S.gas_and_chains(2000, 9000, 15, seed=4, half=700.0)  # 135,000 joints
    b = engine.Batch.from_scenes([sc]).advance(2)
    assert b.get_option(engine.OPT_LAST_SWEEPS) == 1
    b.close()


def test_gpu_a_jointed_body_that_turns_dynamic_gets_a_place_in_its_joints_order(engine):
    """Which joints of a body must differ in colour, and its joints' ranks, go by the body's type."""
    sc = _motors()
    lift = [i for i, t in enumerate(sc.body_type) if t == S.KINEMATIC][0]
    batches = []
    for mode in (1, 0):
        b = engine.Batch.from_scenes([sc])
        b.set_option(engine.OPT_SOLVER, engine.SOLVER_COLOURS)
        b.set_option(engine.OPT_SWEEPS, mode)
        b.advance(10)
        rec = b.bodies()
        rec["type"][lift], rec["mass"][lift], rec["inv_mass"][lift], rec["inv_i"][lift] = S.DYNAMIC, 2.0, 0.5, 0.3
        b.upload_bodies(0, rec)
        b.advance(30)
        batches.append(b)
    ref, b = batches
    assert b.get_option(engine.OPT_LAST_SWEEPS) == 2
    assert np.array_equal(ref.bodies().view(np.uint8), b.bodies().view(np.uint8))
    assert np.array_equal(ref.joints(sc.joint_count).view(np.uint8), b.joints(sc.joint_count).view(np.uint8))


def test_gpu_steps_after_a_withdrawn_launch_take_a_launch_per_colour(engine):
    """A launch without room for its workgroups costs a millisecond and one workgroup's sweeps: the steps after
    it do without, and try again later. The states are a launch per colour's all the way."""
    scenes = [S.gas_and_chains(300, 6, 12, seed=7, half=40.0)]
    ref, b = engine.Batch.from_scenes(scenes), engine.Batch.from_scenes(scenes)
    ref.set_option(engine.OPT_SWEEPS, 1)
    took = []
    for k in range(300):
        b.set_option(engine.OPT_SWEEPS, 2 if k == 5 else 0)  # (2: the workgroups give up their places)
        ref.advance(1)
        b.advance(1)
        took.append(b.get_option(engine.OPT_LAST_SWEEPS))
    assert took == [2] * 6 + [1] * 256 + [2] * 38
    assert np.array_equal(ref.bodies().view(np.uint8), b.bodies().view(np.uint8))


def test_gpu_a_phase_of_many_seconds_is_no_stall(engine):
    """Twenty spokes on one hub, their sweeps a chain of twenty updates an iteration, for so many iterations that
    the launch takes seconds and the bodies' update counts wrap their 16 bits many times."""
    s = S.Scene(name="star", gravity=(0.0, -10.0))
    s.add_body(S.STATIC, 0.0, 0.0)
    hub = s.add_body(S.DYNAMIC, 0.0, 0.0)
    s.add_circle(hub, 0.3)
    for i in range(20):
        x, y = np.cos(0.31 * i), np.sin(0.31 * i)
        arm = s.add_body(S.DYNAMIC, 2.0 * x, 2.0 * y)
        s.add_box(arm, 0.1, 0.05)
        s.add_revolute(hub, arm, (x, y))
    batches = []
    for mode in (0, 2):
        b = engine.Batch.from_scenes([s])
        b.set_option(engine.OPT_SWEEPS, mode)
        b.advance(1, vi=120000, pi=20)
        assert b.get_option(engine.OPT_LAST_SWEEPS) == 2
        batches.append(b)
    assert np.array_equal(batches[0].bodies().view(np.uint8), batches[1].bodies().view(np.uint8))
    assert np.isfinite(batches[0].bodies()["v"]).all()


def test_gpu_a_world_solved_in_a_workgroup_keeps_no_flow_states(engine):
    """A single world that fits a workgroup does without the bodies' flow states (256 bytes each, and their
    stores in every step): the step in which it outgrows the workgroup takes a launch per colour."""
    b = engine.Batch.from_scenes([S.random_pile(1700, seed=7, half_w=24.0, height=130.0)])
    paths = []
    while len(paths) < 400 and paths[-2:] != [(1, 2)] * 2:
        b.advance(1)
        paths.append((b.get_option(engine.OPT_LAST_SOLVER), b.get_option(engine.OPT_LAST_SWEEPS)))
    out = [k for k, p in enumerate(paths) if p[0] == 1]
    assert paths[0][0] == 2 and out and paths[out[0]] == (1, 1) and paths[-1] == (1, 2)

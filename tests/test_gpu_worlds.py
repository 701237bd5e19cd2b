"""GPU tests of the one-workgroup solves by class (b2g_worlds.h): worlds of
sizes around the classes' limits, past every class, empty of contacts, with
and without warm starting, idle in some steps, in eager and captured steps.
Each compares bit for bit with the colour sweeps, a launch per colour."""
import numpy as np
import pytest

from util import load_pkg

pytestmark = pytest.mark.gpu
S = load_pkg().scenes


def _sized():
    """Solved contacts from none to past the largest class's 2048, bodies past its 4096 and past the smaller ones'."""
    out = [S.pyramid(r) for r in (1, 5, 6, 7, 8, 9, 10, 11, 15, 16, 21, 22, 30, 31, 32, 40, 44, 45)]
    out += [S.random_pile(n, seed=40 + n, half_w=max(6.0, 0.55 * n ** 0.5), height=20.0 + n ** 0.5)
            for n in (3, 40, 90, 200, 500, 1100, 2500)]
    out += [S.random_pile(5200, seed=3, half_w=120.0, height=400.0)]  # few contacts, too many bodies
    fall = S.pyramid(3)  # nothing touches anything
    fall.body_pos = [(x, y + 30.0 * i) for i, (x, y) in enumerate(fall.body_pos)]
    return out + [fall]


def _same(a, b, what):
    assert np.array_equal(a.bodies().view(np.uint8), b.bodies().view(np.uint8)), (what, "bodies")
    assert np.array_equal(a.contacts().view(np.uint8), b.contacts().view(np.uint8)), (what, "contacts")


def _pair(engine, scenes):
    a, b = engine.Batch.from_scenes(scenes), engine.Batch.from_scenes(scenes)
    b.set_option(engine.OPT_SOLVER, engine.SOLVER_COLOURS)
    b.set_option(engine.OPT_SWEEPS, 1)
    return a, b


@pytest.mark.parametrize("warm", [True, False])
def test_gpu_worlds_by_class_equal_colour_sweeps(engine, warm):
    scenes = _sized()
    a, b = _pair(engine, scenes)
    flags = [warm or k % 2 == 0 for k in range(len(scenes))]
    for steps in (1, 1, 18, 40, 60):
        a.advance(steps, warm=flags)
        b.advance(steps, warm=flags)
        assert a.get_option(engine.OPT_LAST_SOLVER) == 2 and b.get_option(engine.OPT_LAST_SOLVER) == 1
        _same(a, b, steps)
    assert np.array_equal(a.contact_colours(len(a.contacts())), b.contact_colours(len(b.contacts())))
    # captured steps of the same batch, on from here
    g = engine.Batch.from_scenes(scenes).advance(120, warm=flags)
    for _ in range(12):
        a.step(8, 3, 0)
        g.step(8, 3, engine.STEP_GRAPH | engine.STEP_ASYNC)
    assert g.counts().graph_steps == 12
    _same(a, g, "captured")


@pytest.mark.parametrize("vi,pi", [(0, 0), (1, 1), (5, 9)])
def test_gpu_worlds_by_class_iteration_counts(engine, vi, pi):
    scenes = [S.pyramid(4), S.random_pile(300, seed=9, half_w=9.0, height=30.0), S.pyramid(30)]
    a, b = _pair(engine, scenes)
    a.advance(30, vi=vi, pi=pi)
    b.advance(30, vi=vi, pi=pi)
    _same(a, b, (vi, pi))


@pytest.mark.parametrize("make", [lambda: S.pyramid(2), lambda: S.pyramid(20), lambda: S.pyramid(43),
                                  lambda: S.random_pile(400, seed=6, half_w=11.0, height=50.0),
                                  lambda: S.random_pile(1700, seed=7, half_w=24.0, height=130.0)])
def test_gpu_single_world_in_one_launch_equals_colour_sweeps(engine, make):
    """A world that outgrows the largest class on the way (the last scene) goes over to the sweeps."""
    a, b = _pair(engine, [make()])
    paths = set()
    for _ in range(20):
        a.advance(20)
        b.advance(20)
        paths.add(a.get_option(engine.OPT_LAST_SOLVER))
        _same(a, b, paths)
    assert 2 in paths


def test_gpu_worlds_by_class_with_idle_worlds(engine):
    scenes = [S.batch_world(i, 30 + 60 * i) for i in range(14)]
    a, b = _pair(engine, scenes)
    a.advance(20)
    b.advance(20)
    rng = np.random.default_rng(5)
    dt = np.float32(1.0 / 60.0)
    for k in range(12):
        on = rng.random(len(scenes)) < (0.0 if k == 5 else 0.4)
        for x in (a, b):
            x.set_world_params(0, [engine.WorldParams(g, dt, 1.0, 1, int(on[w])) for w, g in enumerate(x.gravity)])
            x.step(8, 3, 0)
        _same(a, b, k)


def test_gpu_worlds_past_the_largest_class_keep_the_claim_rounds(engine):
    """One launch of a step moves the claim-round base on, also where the largest worlds' launches run beside
    the classes': with a base that lags, old claims win and colours change. Colours of every step."""
    big = S.random_pile(2600, seed=8, half_w=26.0, height=60.0)
    a, b = _pair(engine, [big] + [S.batch_world(i, 20 + 25 * i) for i in range(12)])
    a.advance(100)
    b.advance(100)
    for k in range(60):
        a.advance(1)
        b.advance(1)
        n = len(a.contacts())
        assert np.array_equal(a.contact_colours(n), b.contact_colours(n)), k
    _same(a, b, "end")
    assert a.counts().touching > 2048  # (the large world is past the largest class by far)


def test_gpu_worlds_of_the_last_classes_share_a_launch_while_both_are_active(engine):
    """A world of 1025 to 2048 contacts is solved in its own class's launch, or with the worlds past it where the
    step before had one: both come and go here."""
    scenes = [S.pyramid(30), S.pyramid(44), S.pyramid(34)] + [S.batch_world(i, 40 + 50 * i) for i in range(6)]
    a, b = _pair(engine, scenes)
    a.advance(3)
    b.advance(3)
    dt = np.float32(1.0 / 60.0)
    for k, off in enumerate([(), (1,), (1,), (0, 2), (), (0, 1, 2), (), (3, 4, 5, 6, 7, 8), (), (1,), ()]):
        for x in (a, b):
            x.set_world_params(0, [engine.WorldParams(g, dt, 1.0, 1, int(w not in off))
                                   for w, g in enumerate(x.gravity)])
            x.step(8, 3, 0)
        assert a.get_option(engine.OPT_LAST_SOLVER) == 2
        _same(a, b, (k, off))
    n = len(a.contacts())
    assert np.array_equal(a.contact_colours(n), b.contact_colours(n))


def test_gpu_a_single_world_has_sweeps_to_time(engine):
    """A small world is solved in one launch, which has no sweeps; a caller who times them gets them, with the
    same states."""
    a, b = (engine.Batch.from_scenes([S.pyramid(12)]).advance(30) for _ in range(2))
    assert a.get_option(engine.OPT_LAST_SOLVER) == 2
    for kernel in (engine.KERNEL_WARM_START, engine.KERNEL_CONTACT_VELOCITY, engine.KERNEL_CONTACT_POSITION,
                   engine.KERNEL_NARROWPHASE, engine.KERNEL_SOLVER):
        a.time_kernel(kernel)
        for x in (a, b):
            for _ in range(5):
                x.step(8, 3, 0)
        ms, launches, items = a.kernel_time()
        assert launches >= 5 and ms > 0 and items > 0, kernel
        a.time_kernel(-1)
        _same(a, b, kernel)
    a.step(8, 3, 0)
    assert a.get_option(engine.OPT_LAST_SOLVER) == 2

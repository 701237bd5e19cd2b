"""Query lists (hits packed one query after the other) and the spread of rays
over wavefronts, against the slot entries run query by query."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def batch(engine, pkg):
    b = engine.Batch.from_scenes([pkg.scenes.random_pile(160, seed=3, half_w=20.0), pkg.scenes.pyramid(9)])
    b.step(8, 3)
    yield b
    b.close()


def _one_by_one(engine, batch, entry, dtype, worlds, boxes):
    """Each query alone, with slots for every shape."""
    room, got = batch.counts().shapes, []
    cnt = np.zeros(1, np.int32)
    for w, q in zip(worlds, boxes):
        out = np.zeros(room, dtype)
        w1, q1 = np.array([w], np.int32), np.ascontiguousarray(q, np.float32)
        engine.check(entry(batch.h, 1, engine._ptr(w1), engine._ptr(q1), room, engine._ptr(out), engine._ptr(cnt)))
        got.append(out[:cnt[0]].copy())
    return got


# (2047 and 2048 rays: one per wavefront; 4099: two, the last wavefront with one)
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 2047, 2048, 4099])
@pytest.mark.parametrize("capacity", [0, 1, 64])
def test_gpu_query_lists_equal_single_queries(engine, batch, n, capacity):
    rng = np.random.default_rng(n)
    few = min(n, 65)  # distinct queries; more of them repeat these in order
    lo = rng.uniform([-25, -2], [20, 12], (few, 2))
    box = np.concatenate([lo, lo + rng.uniform(0, 30, (few, 2))], 1).astype(np.float32)
    seg = rng.uniform([-30, -3, -30, -3], [30, 30, 30, 30], (few, 4)).astype(np.float32)
    box[0], seg[0] = (500, 500, 501, 501), (500, 500, 501, 501)  # a query without results
    worlds = rng.integers(0, 2, few).astype(np.int32)
    pick = np.arange(n) % few
    for run, entry, dtype, q in ((batch.query_aabbs, batch.L.b2g_query_aabbs, np.int32, box),
                                 (batch.raycast, batch.L.b2g_raycast, engine.RAY_HIT_DTYPE, seg)):
        want = _one_by_one(engine, batch, entry, dtype, worlds, q)
        got = run(worlds[pick], q[pick], capacity)
        assert len(got) == n
        for i in range(n):
            assert got[i].dtype == dtype and got[i].tobytes() == want[pick[i]].tobytes(), i
    assert n < 3 or sum(map(len, want)) > 0


def test_gpu_query_list_without_queries_or_results(engine, batch):
    assert batch.raycast([], np.zeros((0, 4), np.float32)) == []
    assert [len(h) for h in batch.query_aabbs([0], [[500, 500, 501, 501]])] == [0]
    out = np.zeros(1, engine.RAY_HIT_DTYPE)
    with pytest.raises(engine.B2GError):  # nothing is waiting to be fetched
        engine.check(batch.L.b2g_query_results(batch.h, engine._ptr(out)))
    with pytest.raises(engine.B2GError):
        batch.raycast([2], np.zeros((1, 4), np.float32))


def test_gpu_query_slots_of_several_queries(engine, batch):
    """The slot entry counts what does not fit and fills what does."""
    w = np.zeros(3, np.int32)
    box = np.tile(np.array([-1e4, -1e4, 1e4, 1e4], np.float32), (3, 1))
    full = batch.query_aabbs(w, box)
    out, cnt = np.full((3, 5), -1, np.int32), np.zeros(3, np.int32)
    engine.check(batch.L.b2g_query_aabbs(batch.h, 3, engine._ptr(w), engine._ptr(box), 5, engine._ptr(out),
                                         engine._ptr(cnt)))
    for i in range(3):
        assert cnt[i] == len(full[i]) and np.array_equal(out[i], full[i][:5])

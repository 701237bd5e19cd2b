"""Query lists (hits packed one query after the other) and the spread of rays
over wavefronts, against the slot entries run query by query, and both queries
against the shapes' geometry in 64 bits."""
import numpy as np
import pytest

from util import load_pkg

pytestmark = pytest.mark.gpu
S = load_pkg().scenes


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


# --- against the geometry in 64 bits ------------------------------------------
# Coordinates are below 64, so a float's spacing is at most 4e-6 and a sum of a
# few products of distances and unit vectors is off by some 1e-5: NEAR is ten
# times that. Where moving every surface by NEAR changes whether there is a hit,
# either answer is right.
NEAR = 1e-4


def _near(shape, centre, radius, p1, p2):
    """A circle's hit is the difference of two squares, (s.d)^2 - d.d (s.s - r^2) with s from its centre to the
    ray's start: four roundings of either, over d.d, move the squared radius, and so the radius by its 2r-th part."""
    if shape["type"] != 0:
        return NEAR
    s, d = p1 - centre, p2 - p1
    squared = 4 * 2.0 ** -24 * ((s @ d) ** 2 / (d @ d) + abs(s @ s - radius * radius))
    return NEAR + squared / (2 * radius)


def _geometry(shapes, bodies):
    """Vertices (world, 64 bits), their number, the circles' centre and every shape's radius."""
    x = bodies["xf"].astype(np.float64)[shapes["body"]]
    turn = lambda v: np.stack([x[:, None, 3] * v[..., 0] - x[:, None, 2] * v[..., 1],  # noqa: E731
                               x[:, None, 2] * v[..., 0] + x[:, None, 3] * v[..., 1]], -1) + x[:, None, :2]
    return (turn(shapes["vertices"].astype(np.float64).reshape(-1, 8, 2)),
            turn(shapes["centroid"].astype(np.float64)[:, None])[:, 0], shapes["radius"].astype(np.float64))


def _ray_hits(shape, verts, centre, radius, p1, p2, off):
    """(fraction, is it a hit) of one shape whose surface is moved outwards by `off`."""
    d = p2 - p1
    slack = off / np.hypot(*d)
    if shape["type"] == 0:
        s, rr, r = p1 - centre, d @ d, radius + off
        sigma = (s @ d) ** 2 - rr * (s @ s - r * r)
        if sigma < 0:
            return 0.0, False
        t = -(s @ d + np.sqrt(sigma)) / rr
        return t, 0 <= t <= 1
    if shape["type"] == 1:
        v1, e = verts[1], verts[2] - verts[1]
        n = np.array([e[1], -e[0]]) / np.hypot(*e)
        num, den = n @ (v1 - p1), n @ d
        if den == 0 or (shape["count"] and num > off):
            return 0.0, False
        t, end = num / den, off / np.hypot(*e)
        u = (p1 + t * d - v1) @ e / (e @ e)
        return t, -slack <= t <= 1 + slack and -end <= u <= 1 + end
    v = verts[:shape["count"]]
    e = np.roll(v, -1, 0) - v
    n = np.stack([e[:, 1], -e[:, 0]], 1) / np.hypot(e[:, 0], e[:, 1])[:, None]
    num, den = ((v - p1) * n).sum(1) + off, n @ d
    if ((den == 0) & (num < 0)).any() or not (num < 0).any():
        return 0.0, False
    t = np.max(num[den < 0] / den[den < 0], initial=0.0)
    return t, 0 < t <= np.min(num[den > 0] / den[den > 0], initial=1.0)


def test_gpu_ray_casts_and_box_queries_against_the_geometry_in_64_bits(engine):
    sc = S.random_pile(300, seed=71, half_w=12.0, height=30.0)
    sc.add_edge(0, (-10.0, 5.0), (0.0, 2.0), v0=(-15.0, 6.0), v3=(5.0, 2.0))  # a one-sided edge
    scenes = [sc, S.pyramid(6), S.gas_and_chains(150, 4, 5, seed=4, half=14.0)]
    b = engine.Batch.from_scenes(scenes).advance(40)
    shapes = np.concatenate([engine.scene_records(s, world=i, body_offset=int(b.world_bodies[i]))[1]
                             for i, s in enumerate(scenes)])
    assert set(shapes["type"]) == {0, 1, 2}
    verts, centre, radius = _geometry(shapes, b.bodies())
    world = np.repeat(np.arange(3), np.diff(b.world_shapes))
    rng = np.random.default_rng(9)
    n = 300
    worlds = rng.integers(0, 3, n).astype(np.int32)
    seg = rng.uniform([-16, -15, -16, -15], [16, 18, 16, 18], (n, 4)).astype(np.float32)
    lo = rng.uniform([-16, -15], [14, 16], (n, 2))
    box = np.concatenate([lo, lo + rng.uniform(0, 8, (n, 2))], 1).astype(np.float32)
    rays, found = b.raycast(worlds, seg), b.query_aabbs(worlds, box)
    hits = unsure = 0
    for k in range(n):
        p1, p2 = seg[k, :2].astype(np.float64), seg[k, 2:].astype(np.float64)
        have = {int(h["shape"]): h for h in rays[k]}
        assert len(have) == len(rays[k]) and all(world[j] == worlds[k] for j in have)
        for j in np.flatnonzero(world == worlds[k]):
            near = _near(shapes[j], centre[j], radius[j], p1, p2)
            want = [_ray_hits(shapes[j], verts[j], centre[j], radius[j], p1, p2, off)[1] for off in (-near, 0.0, near)]
            if len(set(want)) > 1:
                unsure += 1
                continue
            assert want[0] == (j in have), (k, j)
            if not want[0]:
                continue
            hits += 1
            at = p1 + float(have[j]["fraction"]) * (p2 - p1)  # on the surface, where the ray enters
            nrm = have[j]["normal"].astype(np.float64)
            assert abs(np.hypot(*nrm) - 1) < 1e-5 and nrm @ (p2 - p1) < NEAR
            if shapes[j]["type"] == 0:
                assert abs(np.hypot(*(at - centre[j])) - radius[j]) < near
                assert np.abs(nrm * radius[j] - (at - centre[j])).max() < near
            else:
                v = verts[j][1:3] if shapes[j]["type"] == 1 else verts[j][:shapes[j]["count"]]
                away = np.abs((v - at) @ nrm)
                assert np.sort(away)[1] < NEAR, (k, j)  # both ends of the side that it hits lie in its plane
        for j in np.flatnonzero(world == worlds[k]):
            v = centre[j][None] if shapes[j]["type"] == 0 else (verts[j][1:3] if shapes[j]["type"] == 1 else
                                                                verts[j][:shapes[j]["count"]])
            gap = np.max([box[k, :2] - (v.max(0) + radius[j]), (v.min(0) - radius[j]) - box[k, 2:]])
            if abs(gap) > NEAR:
                assert (gap < 0) == (j in found[k]), (k, j)
    print("hits", hits, "unsure", unsure, flush=True)
    assert hits > 500 and unsure < 0.02 * hits

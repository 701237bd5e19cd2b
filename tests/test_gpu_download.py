"""GPU tests of the packed body reads: records and states as the device lays
them out for the host (256 bodies to a block, chunks of at most two staging
buffers), against the field-by-field values of the uploaded records and of the
drop-in world's getters."""
import numpy as np
import pytest

from util import load_pkg

pytestmark = pytest.mark.gpu
S = load_pkg().scenes


@pytest.mark.parametrize("n", [1, 63, 255, 256, 257, 1000, 20971, 20972, 52429, 60001])
def test_gpu_body_records_come_back_as_uploaded(engine, n):
    """Every field of every record, whole and in ranges; 20,971 records fill one staging buffer."""
    rng = np.random.default_rng(n)
    rec = np.zeros(n, engine.BODY_DTYPE)
    raw = rng.standard_normal((n, 25)).astype(np.float32)
    rec[:] = np.frombuffer(raw.tobytes(), engine.BODY_DTYPE)
    rec["type"], rec["world"] = rng.integers(1, 3, n), rng.integers(0, 3, n)
    rec["flags"] = rng.integers(0, 4, n)
    b = engine.Batch(worlds=3, bodies=n, shapes=4, joints=1, contacts=64)
    b.set_worlds([engine.WorldParams((0.0, 0.0), 0.1, 0.0, 1, 1, 0)] * 3)
    b.upload_bodies(0, rec)
    assert np.array_equal(b.bodies(0, n).view(np.uint8), rec.view(np.uint8))
    for first, count in ((0, 1), (n - 1, 1), (n // 3, n - n // 3)):
        assert np.array_equal(b.bodies(first, count).view(np.uint8), rec[first:first + count].view(np.uint8))
    st = np.zeros((n, 10), np.float32)
    engine.check(b.L.b2g_download_states(b.h, 0, n, engine._ptr(st)))
    want = np.concatenate([rec["c"], rec["a"][:, None], rec["v"], rec["w"][:, None], rec["xf"]], axis=1)
    assert np.array_equal(st.view(np.uint32), want.view(np.uint32))
    assert b.L.b2g_download_states(b.h, 0, n + 1, engine._ptr(st)) == engine.ERR_INVALID
    b.close()


def test_gpu_world_states_equal_its_batch_records(engine):
    w = engine.World(S.random_pile(700, seed=8, half_w=15.0, height=40.0))
    w.step(30)
    for _ in range(3):
        w.step(1)
        got = w.bodies()
        r = w.batch().bodies(0, w.nb)
        want = np.concatenate([r["c"], r["a"][:, None], r["v"], r["w"][:, None], r["xf"]], axis=1)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        assert np.array_equal(got, w.bodies())
    w.destroy_body(5)
    assert len(w.bodies()) == 700 and np.array_equal(w.bodies(), np.delete(got, 5, axis=0))
    w.close()

"""Host ray queries (query_kernel) against the device-pointer queries' kernel, at the edges of its blocks,
launches and threads, for records and for separate arrays with one bound or one per ray."""
import ctypes

import numpy as np
import pytest

from jarabotransientrendering_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def worlds():
    from jarabotransientrendering_amd import renderer as R
    # 16-bit stack entries, and more than 65,536 nodes: 32-bit ones
    return {level: R.setup_scene(scenes.icosphere_box(level=level, width=4, height=4))[0] for level in (2, 8)}


def _rays(n, seed):
    rng = np.random.default_rng(seed)
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0:3] = rng.random((n, 3))
    d = rng.normal(size=(n, 3))
    rays[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    rays[:, 3] = rng.uniform(-0.2, 0.3, n)
    rays[:, 7] = rng.uniform(0.1, 1.0, n)
    odd = rng.random(n)
    rays[odd < 0.05, 7] = np.inf
    rays[odd < 0.03, 7] = np.uint32(0xFFFFFFFF).view(np.float32)  # NaN of all ones
    rays[odd < 0.02, 3] = np.nan
    rays[odd > 0.97, 5] = 0.0
    return rays


def _device(world, rays):
    """tr_intersect_batch_noalloc, in calls of at most TR_NOALLOC_MAX_RAYS rays."""
    from jarabotransientrendering_amd import renderer as R
    nat, hits = R.nat, np.zeros((len(rays), 4), np.uint32)
    for a in range(0, len(rays), nat.TR_NOALLOC_MAX_RAYS):
        r, h = np.ascontiguousarray(rays[a:a + nat.TR_NOALLOC_MAX_RAYS]), hits[a:a + nat.TR_NOALLOC_MAX_RAYS]
        nat.check(nat.lib().tr_intersect_batch_noalloc(world.handle, nat.as_ptr(r), len(r), ctypes.c_void_p(h.ctypes.data)))
    return hits


@pytest.mark.parametrize("level", [2, 8])
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 127, 128, 129, 4097, 16384, 16385, 100003])
def test_host_queries_match_the_device_query(worlds, level, n):
    from jarabotransientrendering_amd import renderer as R
    nat, w, rays = R.nat, worlds[level], _rays(n, n)
    ref = _device(w, rays)
    hit = ref[:, 3] != 0xFFFFFFFF
    # records
    hits, occ = np.zeros((n, 4), np.uint32), np.zeros(n, np.uint8)
    nat.check(nat.lib().tr_intersect_batch(w.handle, nat.as_ptr(rays), n, nat.as_ptr(hits)))
    nat.check(nat.lib().tr_occluded_batch(w.handle, nat.as_ptr(rays), n, nat.as_ptr(occ)))
    assert np.array_equal(hits, ref) and np.array_equal(occ, hit)
    # arrays, a bound per ray
    t, geom, prim, tri = w.first_intersection(rays[:, 0:3], rays[:, 4:7], rays[:, 3], rays[:, 7])
    assert np.array_equal(np.stack([t.view(np.uint32), geom, prim, tri], 1), ref)
    # arrays, one bound for all: positive (packed entry distances), zero, negative
    for tnear in (1e-5, 0.25, 0.0, -0.1):
        one = rays.copy()
        one[:, 3], one[:, 7] = tnear, 0.9
        ref1 = _device(w, one)
        t, geom, prim, tri = w.first_intersection(rays[:, 0:3], rays[:, 4:7], tnear, 0.9)
        assert np.array_equal(np.stack([t.view(np.uint32), geom, prim, tri], 1), ref1)
        occ = w.intersects(rays[:, 0:3], rays[:, 4:7], 0.9 + tnear, tnear)
        one[:, 7] = np.float32(np.float64(0.9 + tnear) - tnear)
        assert occ.dtype == bool and np.array_equal(occ, _device(w, one)[:, 3] != 0xFFFFFFFF)
        length = rays[:, 7]  # 32-bit lengths, one per ray
        one[:, 7] = length.astype(np.float64) - tnear
        assert np.array_equal(w.intersects(rays[:, 0:3], rays[:, 4:7], length, tnear), _device(w, one)[:, 3] != 0xFFFFFFFF)


def test_shapes_that_broadcast(worlds):
    w, rays = worlds[2], _rays(33, 1)
    one = rays[0, 4:7]
    a = w.first_intersection(rays[:, 0:3], one, np.full((1, 33), 1e-4), [2.0])
    b = w.first_intersection(rays[:, 0:3], np.tile(one, (33, 1)), 1e-4, 2.0)
    assert all(np.array_equal(x, y) for x, y in zip(a, b))
    assert len(w.first_intersection(np.zeros((0, 3)), np.zeros((0, 3)))[0]) == 0
    with pytest.raises(ValueError):
        w.first_intersection(rays[:, 0:3], rays[:5, 4:7])

"""Wavefronts whose bounces run in one launch (path_kernel) against the same renders through the ray and
shadow queues, at the edges of its GPU wavefronts, of the film kernel's groups of segments and of the sizes
that take it."""
import numpy as np
import pytest

from jarabotransientrendering_amd import scenes

pytestmark = pytest.mark.gpu

QUEUES = 64  # TR_RENDER_STACK_KEYED: closest hits with keyed stack entries, which path_kernel does not have


def _scene(name, paths):
    """One pixel with `paths` incoming samples, or a streak row of 8 pixels with a multiple of 8."""
    film = dict(width=1, height=1) if paths % 8 else dict(width=8, height=1)
    n_inc = paths // film["width"]
    if name.startswith("media"):
        return scenes.media_box(scanline=0, time_bins=50, exposure=0.2, sqrt_spp=1, n_incoming=n_inc, max_bounces=7, seed=3, **film)
    if name == "multibounce":
        s = scenes.smooth_scene(level=1, time_bins=64, exposure=0.1, sqrt_spp=1, max_bounces=5, seed=4, **film)
        s.render.n_incoming = n_inc
        s.film.bounce_layers, s.film.camera_unwarp = 3, True
        return s
    return scenes.icosphere_box(level=2, time_bins=90, exposure=0.1, sqrt_spp=1, n_incoming=n_inc, max_bounces=6, seed=5, **film)


def _render(R, scene, flags):
    w, cam, sampler, film, integ = R.setup_scene(scene)
    eng = R.TransientRenderer()
    eng.extra_flags = flags
    st = eng.render(None, w, integ, cam, film, sampler, seed=7)
    return st, *film.read_sums()


@pytest.mark.parametrize("paths", [1, 15, 17, 63, 64, 65, 129, 8 * 64, 8 * 64 + 1, (1 << 15) + 1, (1 << 16) + 1, 1 << 20, (1 << 20) + 1])
@pytest.mark.parametrize("name", ["icosphere", "media", "media_time", "multibounce"])
def test_path_launch_against_the_queues(name, paths):
    from jarabotransientrendering_amd import renderer as R
    s = _scene(name, paths)
    extra = 16 if name == "media_time" else 0  # TR_RENDER_TIME_SAMPLING
    st, sums, weight = _render(R, s, extra)
    st_q, sums_q, weight_q = _render(R, s, extra | QUEUES)
    medium = name.startswith("media")
    # (the media scene's tree is shallow)
    assert st["kernel_launches"]["shade"] == (0 if medium or paths <= 1 << 20 else s.render.max_bounces)
    assert st_q["kernel_launches"]["shade"] == s.render.max_bounces
    for key in ("paths", "extension_rays", "shadow_rays", "contributions"):
        assert st[key] == st_q[key]
    assert np.array_equal(weight, weight_q)
    # the same contributions in another order: within the film's 2 u of their (non-negative) sum on each side
    assert (np.abs(sums - sums_q) <= 2.0 ** -21 * np.abs(sums_q)).all()


@pytest.mark.parametrize("paths", [(1 << 21) + 8, (1 << 23) - 1, 1 << 23, (1 << 23) + 8])
def test_large_path_launch_over_a_shallow_tree(paths):
    """More paths than lanes: wavefronts begin new paths as others end."""
    from jarabotransientrendering_amd import renderer as R
    s = _scene("media", paths)
    st, sums, weight = _render(R, s, 0)
    st_q, sums_q, weight_q = _render(R, s, QUEUES)
    assert st["kernel_launches"]["shade"] == (0 if paths <= 1 << 23 else s.render.max_bounces)
    for key in ("paths", "extension_rays", "shadow_rays", "contributions"):
        assert st[key] == st_q[key]
    assert np.array_equal(weight, weight_q)
    assert (np.abs(sums - sums_q) <= 2.0 ** -21 * np.abs(sums_q)).all()


@pytest.mark.parametrize("sizes", [(3,), (8, 5), (64, 33, 1, 17)])
def test_batch_path_launch_against_the_queues(sizes):
    from jarabotransientrendering_amd import renderer as R
    out = []
    for flags in (0, QUEUES):
        batch, films = R.Batch(), []
        for k, n in enumerate(sizes):
            w, cam, sampler, film, integ = R.setup_scene(scenes.icosphere_box(
                level=1 + k % 3, width=n, height=n, time_bins=40, exposure=0.2, sqrt_spp=2, n_incoming=1, max_bounces=2 + k, seed=k))
            batch.add(w, integ, cam, film, sampler, seed=k)
            films.append(film)
        st = batch.render({"flags": flags})
        out.append((st, [f.read_sums() for f in films]))
    (st, a), (st_q, b) = out
    assert st["kernel_launches"]["shade"] == 0 < st_q["kernel_launches"]["shade"]
    for key in ("paths", "extension_rays", "shadow_rays", "contributions"):
        assert st[key] == st_q[key]
    for (sums, weight), (sums_q, weight_q) in zip(a, b):
        assert np.array_equal(weight, weight_q)
        assert (np.abs(sums - sums_q) <= 2.0 ** -21 * np.abs(sums_q)).all()

"""Wavefronts that trace and deposit the shadow rays of several bounces together: the film does not
depend on how a render is cut into wavefronts and groups of bounces."""
import numpy as np
import pytest

from jarabotransientrendering_amd import scenes

pytestmark = pytest.mark.gpu


def _scene(name):
    if name == "media":
        return scenes.media_box(width=24, height=24, scanline=5, time_bins=128, exposure=0.08, sqrt_spp=5, max_bounces=9, seed=3)
    if name == "unwarp":
        s = scenes.smooth_scene(level=2, width=15, height=11, time_bins=64, exposure=0.1, sqrt_spp=3, max_bounces=5, seed=4)
        s.film.camera_unwarp = True
        return s
    s = scenes.icosphere_box(level=2, width=17, height=13, time_bins=90, exposure=0.1, sqrt_spp=3, n_incoming=2, max_bounces=7, seed=5)
    if name == "multibounce":
        s.film.bounce_layers = 3
    return s


@pytest.mark.parametrize("flags", [0, 2, 8, 32, 64, 1024])  # defaults, binary BVH, graph, stack formats, no packets
@pytest.mark.parametrize("name", ["media", "unwarp", "icosphere", "multibounce"])
def test_film_does_not_depend_on_the_wavefronts(name, flags):
    from jarabotransientrendering_amd import renderer
    s = _scene(name)
    out = []
    for wave in (0, 64, 2 * 501):  # one wavefront, many of one size, many with a partial last one
        w, cam, sampler, film, integ = renderer.setup_scene(s)
        eng = renderer.TransientRenderer()
        eng.wave_paths, eng.extra_flags = wave, flags
        st = eng.render(None, w, integ, cam, film, sampler, seed=7)
        out.append((st, *film.read_sums()))
    for st, sums, weight in out[1:]:
        for key in ("paths", "extension_rays", "shadow_rays", "contributions"):
            assert st[key] == out[0][0][key]
        assert np.array_equal(weight, out[0][2])
        # the same contributions in another order: within the film's 2 u of their (non-negative) sum on each side
        assert (np.abs(sums - out[0][1]) <= 2.0 ** -21 * np.abs(sums)).all()

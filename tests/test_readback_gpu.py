"""Film read-back through pinned staging (csrc/tr_readback.h): whole films, rows at any alignment and
the compensated sums, at sizes around a chunk (2 MiB) and beyond the staging block (16 MiB)."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# values in the film: 315 (one partial group of four), half a chunk of floats, just below one, one value
# more than one, 2.3 chunks, and more than the 8 chunks of a staging block
SIZES = [(3, 5, 7), (32, 32, 256 // 3), (64, 64, 128 // 3), (1, 1, 174763), (61, 43, 150), (100, 101, 150)]


def _film(size, weights):
    from jarabotransientrendering_amd import renderer, scenes
    w, h, t = size
    if weights == "same":
        s = scenes.cornell_box(width=w, height=h, time_bins=t, exposure=4.0 / t, sqrt_spp=2, max_bounces=2)
        world, cam, sampler, film, integ = renderer.setup_scene(s)
        renderer.TransientRenderer().render(None, world, integ, cam, film, sampler, seed=1)
        return film
    film = renderer.StreakCameraFilm(w, h, t, 1.0)
    rng = np.random.default_rng(w * h)
    a = np.zeros(20000, renderer.nat.FILM_SAMPLE_DTYPE)
    a["x"], a["y"] = rng.integers(0, w, len(a)), rng.integers(0, h, len(a))
    a["time"], a["rgb"], a["weight"] = rng.uniform(0, t, len(a)), rng.exponential(1.0, (len(a), 3)), rng.random(len(a))
    film.add_samples(a)
    return film


def _check(film):
    sums, weight = film.read_sums()
    with np.errstate(divide="ignore", invalid="ignore"):
        v = sums / weight[..., None, None]
    expect = np.where(np.isfinite(v), v, 0.0).astype(np.float32)
    img, steady = film.read(steady=True)
    assert np.array_equal(img, expect)
    # the steady image sums the pixel's values in double (up to 174,763 of them) and rounds once
    total = np.where(np.isfinite(v), v, 0.0).sum(axis=2)
    np.testing.assert_allclose(steady, total, rtol=2.0 ** -23, atol=0)
    for a, n in ((0, 1), (film.rows // 2, film.rows - film.rows // 2), (film.rows - 1, 1)):
        assert np.array_equal(film.read_rows(a, n), expect[a:a + n])


@pytest.mark.parametrize("weights", ["same", "per pixel"])
@pytest.mark.parametrize("size", SIZES)
def test_read_is_the_normalised_sums(size, weights):
    _check(_film(size, weights))


def test_reads_of_several_threads():
    films = [_film(s, "per pixel") for s in SIZES[2:] * 2]
    with ThreadPoolExecutor(4) as pool:
        list(pool.map(_check, films))


def test_multibounce_read_is_the_normalised_sums():
    from jarabotransientrendering_amd import renderer, scenes
    s = scenes.cornell_box(width=41, height=31, time_bins=100, exposure=0.05, sqrt_spp=2, max_bounces=4)
    s.film.bounce_layers = 3
    img, _, film = renderer.render_scene(s)
    sums, weight = film.read_sums()
    with np.errstate(divide="ignore", invalid="ignore"):
        v = sums / weight[..., None, None]
    assert np.array_equal(img, np.where(np.isfinite(v), v, 0.0).astype(np.float32))

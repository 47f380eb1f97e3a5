"""Renders through the ray and shadow queues where a small wavefront would take one launch for all its bounces:
groups of fewer bounces than a render has, stack formats, camera-ray packets, graph replay, batches, and the
oracle's rows of a full-size film, and the largest renders of one launch."""
import numpy as np
import pytest

from jarabotransientrendering_amd import _native as nat, scenes

pytestmark = pytest.mark.gpu

QUEUES, GROUP = nat.TR_RENDER_QUEUES, nat.TR_RENDER_SHADOW_GROUP
COUNTS = ("paths", "extension_rays", "shadow_rays", "contributions")


@pytest.fixture(scope="module")
def R():
    from jarabotransientrendering_amd import renderer
    return renderer


def _scene(name):
    if name == "media":
        return scenes.media_box(width=24, height=24, scanline=5, time_bins=128, exposure=0.08, sqrt_spp=5, max_bounces=7, seed=3)
    if name == "unwarp":
        s = scenes.smooth_scene(level=2, width=15, height=11, time_bins=64, exposure=0.1, sqrt_spp=3, max_bounces=7, seed=4)
        s.film.camera_unwarp = True
        return s
    s = scenes.icosphere_box(level=2, width=17, height=13, time_bins=90, exposure=0.1, sqrt_spp=3, n_incoming=2, max_bounces=7, seed=5)
    if name == "multibounce":
        s.film.bounce_layers = 3
    return s


def _render(R, s, flags, wave=0, guide=None):
    w, cam, sampler, film, integ = R.setup_scene(s)
    eng = R.TransientRenderer()
    eng.wave_paths, eng.extra_flags = wave, flags
    st = eng.render(None, w, integ, cam, film, sampler, seed=7, guide=guide)
    return st, *film.read_sums()


def _same(a, b):
    for key in COUNTS:
        assert a[0][key] == b[0][key]
    assert np.array_equal(a[2], b[2])
    # the same contributions in another order: within the film's 2 u of their (non-negative) sum on each side
    assert (np.abs(a[1] - b[1]) <= 2.0 ** -21 * np.abs(b[1])).all()


@pytest.mark.parametrize("flags", [0, nat.TR_RENDER_BINARY_BVH, nat.TR_RENDER_GRAPH, nat.TR_RENDER_STACK32,
                                   nat.TR_RENDER_STACK_KEYED, nat.TR_RENDER_NO_CAMERA_PACKETS])
@pytest.mark.parametrize("name", ["media", "unwarp", "icosphere", "multibounce", "guided"])
def test_film_does_not_depend_on_groups_of_bounces(R, name, flags):
    """All seven bounces' shadow rays together, or every 1, 2, 3 (a shorter last group) or 6 of them, in one
    wavefront and in several with a partial last one."""
    s = _scene("media" if name == "guided" else name)
    guide = None
    if name == "guided":
        guide = R.PathGuide(steps_per_wave=0, init_seed=2)
    base = _render(R, s, 0, guide=guide)
    for wave in (0, 2 * 151):
        for group in (0, 1, 2, 3, 6):
            out = _render(R, s, flags | QUEUES | GROUP(group), wave, guide)
            launches, waves = out[0]["kernel_launches"], out[0]["waves"]
            assert launches["extend"] == launches["shade"] == 7 * waves
            assert launches["shadow"] == -(-7 // (group or 7)) * waves
            assert (waves > 1) == (wave != 0)
            _same(out, base)


def test_a_batch_does_not_depend_on_groups_of_bounces(R):
    """Jobs of 2 to 5 bounces in shared wavefronts."""
    def render(flags, wave=0):
        batch, films = R.Batch(), []
        for k, n in enumerate((21, 9, 1, 17)):
            w, cam, sampler, film, integ = R.setup_scene(scenes.icosphere_box(
                level=1 + k % 3, width=n, height=n, time_bins=40, exposure=0.2, sqrt_spp=2, n_incoming=1, max_bounces=2 + k, seed=k))
            batch.add(w, integ, cam, film, sampler, seed=k)
            films.append(film)
        st = batch.render({"flags": flags, "wave_paths": wave})
        return st, [f.read_sums() for f in films]
    st0, films0 = render(0)
    assert st0["kernel_launches"]["shade"] == 0
    for flags in (QUEUES, QUEUES | nat.TR_RENDER_GRAPH, QUEUES | nat.TR_RENDER_STACK32, QUEUES | GROUP(1), GROUP(2), GROUP(4)):
        for wave in (0, 1000):
            st, films = render(flags, wave)
            group = flags >> 24 or 5
            assert st["kernel_launches"]["shade"] == 5 * st["waves"]
            assert st["kernel_launches"]["shadow"] == -(-5 // group) * st["waves"]
            for (sums, weight), (sums0, weight0) in zip(films, films0):
                _same((st, sums, weight), (st0, sums0, weight0))


@pytest.mark.parametrize("spp", [1, 3, 8])  # packets over 64 pixels, over seven, of one
@pytest.mark.parametrize("flags", [nat.TR_RENDER_STACK32, nat.TR_RENDER_NO_CAMERA_PACKETS, nat.TR_RENDER_BINARY_BVH,
                                   nat.TR_RENDER_STACK32 | nat.TR_RENDER_NO_CAMERA_PACKETS])
def test_stack_formats_and_packets(R, flags, spp):
    """An odd film around the camera's axis, where the rays of a packet go up and down each axis."""
    s = scenes.icosphere_box(level=4, width=15, height=15, time_bins=128, exposure=0.1, sqrt_spp=spp, n_incoming=1, max_bounces=5, seed=23)
    a, b = _render(R, s, QUEUES), _render(R, s, QUEUES | flags)
    assert a[0]["kernel_launches"]["shade"] == b[0]["kernel_launches"]["shade"] == 5
    _same(a, b)
    _same(a, _render(R, s, flags & ~nat.TR_RENDER_NO_CAMERA_PACKETS))


def test_graph_replay_of_the_queues(R):
    for name in ("media", "icosphere"):
        s = _scene(name)
        a = _render(R, s, QUEUES, 2 * 151)
        for _ in range(3):
            b = _render(R, s, QUEUES | nat.TR_RENDER_GRAPH, 2 * 151)
            assert a[0]["waves"] == b[0]["waves"] >= 2 and a[0]["kernel_launches"] == b[0]["kernel_launches"]
            _same(a, b)


@pytest.mark.parametrize("flags", [QUEUES, QUEUES | GROUP(3), QUEUES | nat.TR_RENDER_STACK32])
def test_full_size_rows_match_the_oracle(R, oracle, flags):
    """Three rows of a 256 x 256 pixel, 1024 bin film over 81,920 triangles, by the kernels of large frames."""
    s = scenes.icosphere_box(level=6, width=256, height=256, time_bins=1024, exposure=0.01, sqrt_spp=4,
                             n_incoming=1, max_bounces=8, seed=9)
    w, cam, sampler, film, integ = R.setup_scene(s)
    eng = R.TransientRenderer()
    eng.extra_flags = flags
    st = eng.render(None, w, integ, cam, film, sampler, seed=9)
    assert st["kernel_launches"]["shade"] == 8
    part = film.read_rows(120, 3)
    f, wt, _ = oracle.render(s, oracle.RNG_PER_PATH, rows=(120, 123), seed=9)
    ref = oracle.normalize(f, wt)
    # a path whose hit or bin is decided otherwise by a rounding goes another way: few pixels, little of the sum
    per_pix = np.abs(part - ref).sum(axis=(2, 3)) / np.maximum(np.abs(ref).sum(axis=(2, 3)), 1e-4)
    assert (per_pix < 1e-4).mean() >= 0.95
    assert abs(part.sum() / ref.sum() - 1) < 5e-3


def _cubes(n):
    """A box shell with n cubes in it: 4-wide trees of 2, 4, 6, 8, 11, 13 and 16 nodes for n from 0 to 6."""
    rng = np.random.default_rng(n)
    tris = [scenes.box_shell(inner_box=False)[0]]
    for _ in range(n):
        c, size = rng.uniform(0.1, 0.7, 3), rng.uniform(0.08, 0.25, 3)
        v = np.array([[x, y, z] for x in (0, 1) for y in (0, 1) for z in (0, 1)]) * size + c
        for a, b, d, e in ((0, 1, 3, 2), (4, 6, 7, 5), (0, 4, 5, 1), (2, 3, 7, 6), (0, 2, 6, 4), (1, 5, 7, 3)):
            tris.append(np.array([[v[a], v[b], v[d]], [v[a], v[d], v[e]]], np.float32))
    return np.concatenate(tris).astype(np.float32)


@pytest.mark.parametrize("cubes,paths,flags,one_launch", [
    (4, 1 << 23, 0, True), (4, (1 << 23) + 8, 0, False),      # the largest of a tree of eleven nodes
    (6, 1 << 20, 0, True), (6, (1 << 20) + 8, 0, False),      # of more
    (6, 1 << 19, nat.TR_RENDER_STACK32, True), (6, (1 << 19) + 8, nat.TR_RENDER_STACK32, False),  # with 32-bit stacks
    (1, (1 << 10) + 8, 0, True), (1, (1 << 16) + 8, 0, True)])  # wavefronts of 16 and 64 paths
def test_the_largest_path_launches(R, cubes, paths, flags, one_launch):
    w = R.World()
    w.add_triangles(_cubes(cubes), R.Lambertian((0.7, 0.6, 0.5)))
    w.add_light(R.PointLightSource((0.5, 0.95, 0.5), (10, 10, 10)))
    w.freeze()
    camera = R.PinholeCamera((0.5, 0.5, -1.2), (0.5, 0.5, 0.5), (0.0, 1.0, 0.0), 45.0)
    out = []
    for queues in (0, QUEUES):
        film = R.StreakCameraFilm(8, 1, 50, 0.1)
        integ = R.BidirectionalPathTracing(w, paths // 8, None, film)
        integ.set_max_path_size(4)
        eng = R.TransientRenderer()
        eng.extra_flags = flags | queues
        st = eng.render(None, w, integ, camera, film, R.StratifiedSampler(8, 1, 1), seed=2)
        assert (st["kernel_launches"]["shade"] == 0) == (one_launch and not queues)
        out.append((st, *film.read_sums()))
    _same(*out)

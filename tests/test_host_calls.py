"""The library's host code over a HIP runtime that launches nothing (fake_hip.cpp): what a call does when memory
runs out, and which kernels it launches. Each program runs in a process of its own."""
import os
import subprocess
import sys

import pytest

from tests.conftest import ROOT
from jarabotransientrendering_amd.build import LIB

pytestmark = pytest.mark.skipif(not os.path.exists(LIB), reason="HIP library not built")

HEAD = """
import ctypes, sys
sys.path.insert(0, {root!r})
fake = ctypes.CDLL({fake!r}, mode=ctypes.RTLD_GLOBAL)
fake.fake_log.restype, fake.fake_used.restype = ctypes.c_char_p, ctypes.c_size_t
fake.fake_pinned_live.restype = fake.fake_pinned_made.restype = ctypes.c_size_t
fake.fake_budget.argtypes = [ctypes.c_size_t]
fake.fake_mallocs_left.argtypes = [ctypes.c_long]
import numpy as np
from jarabotransientrendering_amd import _native as nat, renderer as R, scenes
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    so = os.path.join(tmp_path_factory.mktemp("hip"), "libamdhip64.so.7")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-w", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__",
                           "-I/opt/rocm/include", "-Wl,-soname,libamdhip64.so.7",
                           os.path.join(ROOT, "tests", "fake_hip.cpp"), "-o", so])

    def program(text):
        r = subprocess.run([sys.executable, "-c", HEAD.format(root=ROOT, fake=so) + text], capture_output=True, text=True,
                           timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout
    return program


@pytest.mark.parametrize("n", [1000, 20000])
def test_samples_need_no_pinned_memory(run, n):
    """Once a call has added its radiance nothing is left that can run out of memory: the weights are in too."""
    run(f"""
film = R.StreakCameraFilm(13, 7, 20, 0.1)
a = np.zeros({n}, nat.FILM_SAMPLE_DTYPE)
a["x"], a["y"], a["weight"] = np.arange({n}) % 13, np.arange({n}) // 13 % 7, 1.0
film.handle
fake.fake_pinned_fails(1)
film.add_samples(a)
weights = np.empty((7, 13))
nat.check(nat.lib().tr_film_read_sums(film.handle, None, nat.as_ptr(weights)))
assert np.array_equal(weights.ravel(), np.bincount(a["y"] * 13 + a["x"], minlength=91)), weights
""")


@pytest.mark.parametrize("n", [100, 16384, 16385, 131072])
@pytest.mark.parametrize("width,height", [(13, 7), (300, 100)])
def test_sample_weights_are_summed_in_order(run, n, width, height):
    """Weights of any magnitudes: each call's are summed in the order of the samples and then added to the
    film's, in double, so that the same calls give the same bits."""
    run(f"""
rng = np.random.default_rng(5)
film = R.StreakCameraFilm({width}, {height}, 8, 0.1)
expect = np.zeros({width * height})
for call in range(3):
    a = np.zeros({n}, nat.FILM_SAMPLE_DTYPE)
    pix = rng.integers(0, min(40, {width * height}), {n})
    a["x"], a["y"] = pix % {width}, pix // {width}
    a["weight"] = np.exp(rng.normal(0.0, 12.0, {n}))
    film.add_samples(a)
    added = np.zeros({width * height})
    for p, w in zip(pix, a["weight"].astype(np.float64)):
        added[p] += w
    expect += added
got = np.empty(({height}, {width}))
nat.check(nat.lib().tr_film_read_sums(film.handle, None, nat.as_ptr(got)))
assert np.array_equal(got.ravel(), expect), np.abs(got.ravel() - expect).max()
# a sample outside the film: no weight is added, then or by the next call
a["y"][{n} - 1] = {height}
try:
    film.add_samples(a)
    raise SystemExit("accepted")
except nat.TrError as e:
    assert "sample {n - 1} lies outside the film" in str(e), e
nat.check(nat.lib().tr_film_read_sums(film.handle, None, nat.as_ptr(got)))
assert np.array_equal(got.ravel(), expect)
a["y"][{n} - 1] = 0
a["weight"] = 1.0
film.add_samples(a)
nat.check(nat.lib().tr_film_read_sums(film.handle, None, nat.as_ptr(got)))
pix[{n} - 1] = a["x"][{n} - 1]
assert np.array_equal(got.ravel(), expect + np.bincount(pix, minlength={width * height}))
""")


@pytest.mark.parametrize("threads", [8, 40])
def test_concurrent_reads_share_the_pinned_chunks(run, threads):
    """Films of 6 MB read by several threads at once, again and again: at most 32 chunks of 2 MiB are kept, and
    no more are made than those and one for each thread that finds none."""
    run(f"""
import threading
films = [R.StreakCameraFilm(45, 45, 256, 0.1) for _ in range({threads})]
for f in films:
    f.handle
fake.fake_event_us(300)
def go(f):
    for _ in range(6):
        f.read()
ts = [threading.Thread(target=go, args=(f,)) for f in films]
[t.start() for t in ts]
[t.join() for t in ts]
assert fake.fake_pinned_live() <= 64 << 20, fake.fake_pinned_live()
if {threads} <= 32:
    assert fake.fake_pinned_made() <= 64 << 20, fake.fake_pinned_made()
""")


def test_a_read_without_pinned_memory_says_so(run):
    run("""
film = R.StreakCameraFilm(4, 4, 8, 0.1)
film.handle
fake.fake_pinned_fails(1)
try:
    film.read()
    raise SystemExit("read")
except nat.TrError as e:
    assert e.code == nat.TR_ERR_NOMEM, e
fake.fake_pinned_fails(0)
film.read()
""")


FRAME = """
def frame(size, spp, bounces, layers=0, unwarp=False, n_inc=1):
    s = scenes.icosphere_box(level=0, width=size, height=size, time_bins=4, exposure=1.0, sqrt_spp=spp, n_incoming=n_inc,
                             max_bounces=bounces, seed=1)
    s.film.bounce_layers, s.film.camera_unwarp = layers, unwarp
    w, cam, sampler, film, integ = R.setup_scene(s)
    return lambda **k: R.TransientRenderer().render(None, w, integ, cam, film, sampler, seed=1, **k)
"""


def test_a_process_may_hold_many_rendered_scenes(run):
    """Frames of 67 M paths in as many scenes, all kept: a few take the large shape (25 GB), the others stay at
    6.7 GB while there is memory, and then idle ones give theirs back."""
    run(FRAME + """
frames = [frame(256, 32, 8) for _ in range(60)]
used = []
for f in frames:
    assert f()["paths"] == 1 << 26
    used.append(fake.fake_used())
assert used[0] > 20 << 30 and used[9] < 130 << 30, [u >> 30 for u in used]
assert frames[0]()["paths"] == 1 << 26
assert not fake.fake_freed()
""")


@pytest.mark.parametrize("budget", [1, 3, 5, 9, 20, 40])
def test_renders_shrink_to_the_memory_there_is(run, budget):
    """Whatever is left by the time buffers are made: fewer bounces per group, then fewer paths per wavefront, and
    no error left behind for the next launch to report."""
    run(FRAME + f"""
fs = [frame(256, 32, 8), frame(128, 8, 255), frame(256, 16, 16, layers=3, unwarp=True, n_inc=3)]
fake.fake_budget(({budget} << 30) + fake.fake_used())
for f in fs + fs[::-1]:
    f()
assert not fake.fake_freed()
""")


def test_an_allocation_that_fails_leaves_a_scene_that_renders(run):
    """hipMalloc failing at any point of a first, a larger and a multibounce render."""
    run(FRAME + """
for kind in (dict(size=16, spp=2, bounces=5), dict(size=16, spp=2, bounces=5, layers=2, unwarp=True)):
    done = False
    for k in range(60):
        small, f = frame(size=4, spp=1, bounces=2, layers=kind.get("layers", 0)), frame(**kind)
        small()
        fake.fake_mallocs_left(k)
        try:
            f()
            done = True
        except nat.TrError as e:
            assert e.code == nat.TR_ERR_NOMEM, e
        fake.fake_mallocs_left(-1)
        f()
        small()
    assert done and not fake.fake_freed()
""")


def test_idle_buffers_are_given_back_while_others_render(run):
    """Threads that render in turn in more scenes than memory holds: no render loses its buffers."""
    run(FRAME + """
import threading
fake.fake_budget((9 << 30) + fake.fake_used())
wrong = []
def go(k):
    fs = [frame(64, 16, 4 + k) for _ in range(4)]
    for _ in range(5):
        for f in fs:
            try:
                assert f()["paths"] == 1 << 20
            except nat.TrError as e:
                if e.code != nat.TR_ERR_NOMEM:  # (the other threads may hold all there is)
                    wrong.append(str(e))
fake.fake_event_us(200)
ts = [threading.Thread(target=go, args=(k,)) for k in range(8)]
[t.start() for t in ts]
[t.join() for t in ts]
assert not wrong and not fake.fake_freed(), wrong[:3]
""")


@pytest.mark.parametrize("bounces,group", [(1, 1), (5, 1), (5, 2), (7, 3), (7, 6), (7, 7), (9, 0)])
def test_launches_of_groups_of_bounces(run, bounces, group):
    """Closest hits of a bounce carry the shadow queue over (flag 4) unless it begins a group; a group's shadow and
    film launches follow its last bounce."""
    out = run(FRAME + f"""
for flags in (nat.TR_RENDER_QUEUES | nat.TR_RENDER_SHADOW_GROUP({group}), 1024 | nat.TR_RENDER_QUEUES | nat.TR_RENDER_SHADOW_GROUP({group})):
    s = scenes.icosphere_box(level=0, width=4, height=4, time_bins=4, sqrt_spp=1, n_incoming=1, max_bounces={bounces}, seed=1)
    w, cam, sampler, film, integ = R.setup_scene(s)
    e = R.TransientRenderer()
    e.extra_flags = flags
    fake.fake_clear()
    e.render(None, w, integ, cam, film, sampler, seed=1)
    print("\\n".join(l for l in fake.fake_log().decode().split("\\n") if "extend" in l or "shadow_k" in l or "film_k" in l))
    print("end")
""")
    first, second = out.split("end\n")[:2]
    for lines, packets in ((first, True), (second, False)):
        expect = []
        for b in range(bounces):
            flags = (b & 1) | (2 if b == 0 else 0) | (4 if b % (group or bounces) else 0)
            expect.append("extend_camera" if packets and b == 0 else f"extend {flags}")
            if (b + 1) % (group or bounces) == 0 or b + 1 == bounces:
                expect += ["shadow", "film"]
        got = []
        for line in lines.strip().split("\n"):
            kind = next(k for k in ("extend_camera", "extend", "shadow", "film") if k in line)
            got.append(kind + (" " + line.split()[-1] if kind == "extend" else ""))
        assert got == expect


@pytest.mark.parametrize("meshes", ["s", "sf", "fs", "sfs", "ss", "fsfs", "f"])
def test_corner_normals_of_every_mesh_reach_the_device(run, meshes):
    """Smooth (s) and flat (f) meshes in any order: a slot's shading frame holds its triangle's corners and normals,
    zeros for a flat one; a scene of flat meshes alone has none."""
    run(f"""
rng = np.random.default_rng(3)
w, tris, normals = R.World(), [], []
for kind in {meshes!r}:
    t = rng.normal(size=(5, 3, 3)).astype(np.float32)
    n = rng.normal(size=(5, 3, 3)).astype(np.float32) if kind == "s" else None
    w.add_triangles(t, R.Lambertian((0.5, 0.5, 0.5)), n)
    tris.append(t)
    normals.append(np.zeros((5, 3, 3), np.float32) if n is None else n)
tris, normals = np.concatenate(tris), np.concatenate(normals)
w.add_light(R.PointLightSource((0, 0, 5), (1, 1, 1)))
w.freeze()
film = R.StreakCameraFilm(4, 4, 4, 1.0)
integ = R.BidirectionalPathTracing(w, 1, None, film)
R.TransientRenderer().render(None, w, integ, R.PinholeCamera((0, 0, 4), (0, 0, 0), (0, 1, 0)), film, R.StratifiedSampler(4, 4, 1))
fake.fake_shading_normals.restype = ctypes.c_void_p
p = fake.fake_shading_normals()
if "s" not in {meshes!r}:
    assert not p
else:
    assert p
    v = np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_float)), (len(tris), 6, 4))[:, :, :3]
    for k in range(len(tris)):
        slot = np.flatnonzero((v[:, 0] == tris[k, 0]).all(axis=1))
        assert len(slot) == 1
        assert np.array_equal(v[slot[0], 1:3], tris[k, 1:] - tris[k, 0])
        assert np.array_equal(v[slot[0], 3:], normals[k]), k
""")

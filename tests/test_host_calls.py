"""The library's host code over a HIP runtime that launches nothing (fake_hip.cpp): what a call does when memory
runs out, and which kernels it launches. Each program runs in a process of its own."""
import functools
import os
import subprocess
import sys
import tempfile

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


@functools.lru_cache(maxsize=None)
def _fake():
    d = tempfile.mkdtemp()
    so = os.path.join(d, "libamdhip64.so.7")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-w", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__",
                           "-I/opt/rocm/include", "-Wl,-soname,libamdhip64.so.7",
                           os.path.join(ROOT, "tests", "fake_hip.cpp"), "-o", so])
    return so


def run(program):
    r = subprocess.run([sys.executable, "-c", HEAD.format(root=ROOT, fake=_fake()) + program], capture_output=True,
                       text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


@pytest.mark.parametrize("n", [1000, 20000])
def test_samples_need_no_pinned_memory(n):
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
def test_sample_weights_are_summed_in_order(n, width, height):
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
def test_concurrent_reads_share_the_pinned_chunks(threads):
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


def test_a_read_without_pinned_memory_says_so():
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

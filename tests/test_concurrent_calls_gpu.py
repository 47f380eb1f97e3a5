"""Reads, queries and sample calls from many threads at once, over the pinned chunks that they share: every thread
gets the answers that it gets alone."""
import threading

import numpy as np
import pytest

from jarabotransientrendering_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("threads", [2, 9, 34])  # chunks for all, a share each, more threads than chunks
def test_threads_get_their_own_answers(threads):
    from jarabotransientrendering_amd import _native as nat, renderer as R
    rng = np.random.default_rng(threads)
    w = R.setup_scene(scenes.icosphere_box(level=3, width=4, height=4))[0]
    jobs = []
    for k in range(threads):
        film = R.StreakCameraFilm(40 + k % 5, 41, 257, 0.1)  # 5 MB, in part rounded chunks
        a = np.zeros(20000, nat.FILM_SAMPLE_DTYPE)
        a["x"], a["y"] = rng.integers(0, film.width, len(a)), rng.integers(0, film.height, len(a))
        a["time"], a["rgb"], a["weight"] = rng.uniform(0, 26, len(a)), rng.random((len(a), 3)), 1.0
        film.add_samples(a)
        n = 40000 + 1000 * k
        o, d = rng.random((n, 3), np.float32), rng.normal(size=(n, 3)).astype(np.float32)
        jobs.append((film, o, d))

    def answers(job):
        film, o, d = job
        return [film.read(), film.read_sums()[0], *w.first_intersection(o, d), w.intersects(o, d, 0.5)]

    alone = [answers(j) for j in jobs]
    wrong, start = [], threading.Barrier(threads)

    def go(k):
        start.wait()
        for _ in range(3):
            if not all(np.array_equal(x, y) for x, y in zip(answers(jobs[k]), alone[k])):
                wrong.append(k)

    ts = [threading.Thread(target=go, args=(k,)) for k in range(threads)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not wrong

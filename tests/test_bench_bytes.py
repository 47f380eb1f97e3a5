"""The benchmark's byte accounting: what each stage's kernels write and read, with renders of one launch under their
own name."""
import importlib.util
import os

from tests.conftest import ROOT


def test_stage_bytes_follow_the_launches():
    spec = importlib.util.spec_from_file_location("bench", os.path.join(ROOT, "bench.py"))
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    queues = {"camera": 1, "extend": 4, "shade": 4, "shadow": 1, "film": 1}
    one = {"camera": 0, "extend": 1, "shade": 0, "shadow": 0, "film": 1}
    b = bench.stage_bytes(1000, 3000, 2000, 1500, queues)
    assert b["camera"] == 16 * 1000  # a float4 per camera ray (camera_kernel)
    assert set(b) == {"camera", "extend", "shade", "shadow", "film"}
    b1 = bench.stage_bytes(1000, 3000, 2000, 1500, one)
    assert set(b1) == {"path", "film"} and b1["film"] == b["film"]
    assert b1["path"] == 2000 * 81
    assert bench.stage_names({"extend": 1.5, "film": 2.0}, one) == {"path": 1.5, "film": 2.0}
    assert bench.stage_names({"extend": 1.5, "film": 2.0}, queues) == {"extend": 1.5, "film": 2.0}

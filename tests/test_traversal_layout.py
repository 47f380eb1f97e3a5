"""The device layout of the 4-wide BVH (device_bvh4, csrc/tr_bvh.cpp) and the slab test that reads it
(ray_pre / slabs4, csrc/tr_device.h)."""
import os
import subprocess

import numpy as np
import pytest

from jarabotransientrendering_amd import scenes
from tests.conftest import ROOT

CSRC = os.path.join(ROOT, "jarabotransientrendering_amd", "csrc")

PROG = r"""
#include "tr_internal.h"
#include <cmath>
#include <cstdio>
#include <cstring>
#include <vector>
int main(int argc, char** argv) {
    std::vector<float> T;
    FILE* f = std::fopen(argv[1], "rb");
    float x;
    while (std::fread(&x, 4, 1, f) == 1) T.push_back(x);
    std::fclose(f);
    const uint32_t n = uint32_t(T.size() / 9);
    std::vector<int32_t> mat(n, 0);
    const BvhBuildResult br = build_bvh(T.data(), mat.data(), n);
    const std::vector<Bvh4QNodeHost> q = quantize_bvh4(collapse_bvh4(br));
    const Bvh4Device d = device_bvh4(q, br.tris.size());
    // walk both trees together: same boxes, same triangles, children matched by their box bytes
    int bad = d.nodes.size() != q.size() || d.tri_order.size() != n || d.tri_slot.size() != n;
    std::vector<int> seen(n, 0), node_seen(q.size(), 0);
    std::vector<std::pair<uint32_t, uint32_t>> todo{{0u, 0u}};
    while (!todo.empty()) {
        const auto t = todo.back();
        todo.pop_back();
        const Bvh4QNodeHost& a = q[t.first];
        const Bvh4DevNode& b = d.nodes[t.second];
        node_seen[t.second]++;
        bad += std::memcmp(a.origin, b.origin, 12) != 0;
        const float st[3] = {a.step_x, a.step_y, a.step_z};
        for (int k = 0; k < 3; ++k) bad += std::ldexp(b.step24[k], -24) != st[k];
        int inner = 0, m = 0, order[4];
        for (int pass = 0; pass < 3; ++pass)
            for (int k = 0; k < 4; ++k) {
                const uint32_t c = a.ref[k] >> 29;
                if (pass == (c == 0 ? 0 : c == kQEmpty ? 2 : 1)) order[m++] = k;
            }
        for (int i = 0; i < 4; ++i) {
            const int k = order[i];
            const uint32_t c = a.ref[k] >> 29, index = a.ref[k] & 0x1FFFFFFFu, mask = (b.tri_masks >> (8 * i)) & 0xFFu;
            for (int w = 0; w < 6; ++w) bad += a.q[4 * w + k] != b.q[4 * w + i];
            if (c == 0) {
                bad += mask != 0 || i != inner;
                todo.push_back({index, b.child0 + uint32_t(inner)});
                ++inner;
            } else if (c == kQEmpty) {
                bad += mask != 0;
            } else {
                bad += __builtin_popcount(mask) != int(c);
                for (int j = 0; j < 8; ++j)
                    if (mask >> j & 1u) {
                        const uint32_t slot = b.tri0 + uint32_t(j), from = d.tri_order[slot];
                        seen[from]++;
                        bad += from < index || from >= index + c || d.tri_slot[from] != slot;
                    }
            }
        }
        bad += b.n_inner != uint32_t(inner);
    }
    for (int s : seen) bad += s != 1;
    for (int s : node_seen) bad += s != 1;
    std::printf("%d %d\n", bad, int(d.scaled));
    return 0;
}
"""


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    d = tmp_path_factory.mktemp("layout")
    src, exe = d / "c.cpp", d / "c"
    src.write_text(PROG)
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-I", CSRC, str(src), os.path.join(CSRC, "tr_bvh.cpp"), "-o", str(exe)])

    def run(tris):
        path = d / "t.f32"
        np.ascontiguousarray(tris, dtype=np.float32).tofile(path)
        return [int(v) for v in subprocess.check_output([str(exe), str(path)], text=True).split()]
    return run


@pytest.mark.parametrize("n", [0, 1, 2, 3, 4, 5, 8, 9, 17, 22, 333, 5130])
def test_device_layout_holds_the_quantized_tree(walk, n):
    tris = np.concatenate([scenes.box_shell(True)[0], scenes.displaced_icosphere(4)])[:n]
    assert walk(tris) == [0, 1]


def test_grid_steps_that_cannot_be_scaled_are_reported(walk):
    """Scaled by 2^24 the steps of a scene 2^45 across leave the range that the largest reciprocal
    (1e20) allows: such a scene is traversed through its binary BVH."""
    tris = scenes.box_shell(True)[0].astype(np.float64)
    assert walk(tris * 2.0 ** 20) == [0, 1]
    assert walk(tris * 2.0 ** 45) == [0, 0]


def test_widened_slab_contains_exact_plane_distance():
    """Entry planes are evaluated as fma(q, step inv, fma(origin, inv, c0)) with c0 = fma(-k, |inv|,
    -(o inv)), exit planes with c1 = fma(k, |inv|, -(o inv)), k = 1e-6 (C + |o|). The exact distances
    of the planes as the host rounds them lie between; the exit plane also lies the three ulp
    further by which the far bound of a hit is moved. Without the margin neither holds."""
    F = np.float32
    rng = np.random.default_rng(5)
    n = 400_000
    origin = rng.uniform(-2.0, 2.0, n).astype(F)
    step = np.ldexp(F(1.0), rng.integers(-20, -2, n)).astype(F)
    q = rng.integers(0, 256, n).astype(F)
    o = (origin + rng.uniform(-1.0, 1.0, n) * rng.choice([1e-6, 1e-3, 1.0], n)).astype(F)
    d = (rng.normal(size=n) * rng.choice([1.0, 1e-3, 1e-7, 0.0], n, p=[0.7, 0.1, 0.1, 0.1])).astype(F)
    inv = (F(1.0) / np.where(np.abs(d) < F(1e-20), np.copysign(F(1e-20), d), d)).astype(F)
    C = np.nextafter((np.abs(origin).astype(np.float64) + 255.0 * step).astype(F), F(np.inf))

    def fma(a, b, c):  # rounded once in float64, once to float32: at most an ulp from a fused one
        return (a.astype(np.float64) * b.astype(np.float64) + c.astype(np.float64)).astype(F)
    exact = ((origin.astype(np.float64) + q.astype(np.float64) * step).astype(F).astype(np.float64) - o) * inv.astype(np.float64)

    def planes(scale):
        k = (F(1e-6) * F(scale) * (C + np.abs(o)).astype(F)).astype(F)
        a, c = (step * inv).astype(F), (-(o * inv).astype(F)).astype(F)
        entry = fma(q, a, fma(origin, inv, fma(-k, np.abs(inv), c))).astype(np.float64)
        exit_ = fma(q, a, fma(origin, inv, fma(k, np.abs(inv), c))).astype(np.float64)
        slack = np.spacing(np.abs(entry).astype(F)).astype(np.float64)
        return entry - slack, exit_ + slack
    entry, exit_ = planes(1.0)
    assert (entry <= exact).all()
    assert (exit_ >= exact + 3.6e-7 * np.abs(exact)).all()
    entry, exit_ = planes(0.0)
    assert (entry > exact).any() and (exit_ < exact + 3.6e-7 * np.abs(exact)).any()


@pytest.mark.gpu
@pytest.mark.parametrize("level", [None, 2, 6])
@pytest.mark.parametrize("tnear", [0.0, 1e-5, 0.3])
def test_queries_from_any_near_bound_match_the_oracle(oracle, level, tnear):
    """Bit-exact ids and distances against the oracle's brute-force watertight test; the public
    queries take a near bound of zero too, whose entry distances do not order like their bits (-0)."""
    from jarabotransientrendering_amd import renderer
    s = scenes.cornell_box() if level is None else scenes.icosphere_box(level=level)
    w, *_ = renderer.setup_scene(s)
    rng = np.random.default_rng(3)
    n = 300 if level == 6 else 3000
    o = rng.uniform(0.02, 0.98, (n, 3)).astype(np.float32)
    d = rng.normal(size=(n, 3))
    d = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    t, _, _, tri = w.first_intersection(o, d, tnear=tnear)
    ids, ref_t = oracle.intersect(s, np.concatenate([o, d], 1), tnear=tnear, method=oracle.ISECT_WATERTIGHT, use_bvh=False)
    assert np.array_equal(np.where(tri == 0xFFFFFFFF, -1, tri.astype(np.int64)), ids)
    assert np.array_equal(t[ids >= 0], ref_t[ids >= 0])

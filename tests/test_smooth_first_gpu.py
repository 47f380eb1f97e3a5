"""A scene whose first mesh has corner normals (as an OBJ with "vn" records is loaded), against the oracle and against
the same triangles with the flat ones first."""
import numpy as np
import pytest

from jarabotransientrendering_amd import _native as nat, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flags", [0, nat.TR_RENDER_QUEUES])
def test_smooth_mesh_first(oracle, flags):
    from jarabotransientrendering_amd import renderer as R

    def render(s):
        w, cam, sampler, film, integ = R.setup_scene(s)
        eng = R.TransientRenderer()
        eng.extra_flags = flags
        return eng.render(None, w, integ, cam, film, sampler, seed=5), film.read()

    s = scenes.smooth_scene(level=2, width=16, height=16, time_bins=128, exposure=0.05, sqrt_spp=2, n_incoming=2, max_bounces=5, seed=5)
    st, img = render(s)
    smooth = np.any(s.vertex_normals != 0, axis=(1, 2))
    order = np.concatenate([np.flatnonzero(smooth), np.flatnonzero(~smooth)])
    s.tris, s.tri_mat, s.vertex_normals = s.tris[order], s.tri_mat[order], s.vertex_normals[order]
    st1, img1 = render(s)
    f, wt, _ = oracle.render(s, oracle.RNG_PER_PATH, seed=5)
    # paths whose hit is decided otherwise (by a rounding, or by the order of triangles at equal distance) go
    # another way: few pixels, little of the sum
    for ref, got in ((oracle.normalize(f, wt), img1), (img, img1)):
        per_pix = np.abs(got - ref).sum(axis=(2, 3)) / np.maximum(np.abs(ref).sum(axis=(2, 3)), 1e-4)
        assert (per_pix < 1e-4).mean() >= 0.95
        assert abs(got.sum() / ref.sum() - 1) < 5e-3
    assert abs(st1["contributions"] / st["contributions"] - 1) < 5e-3

"""The device-side sum of a gradient call (grad_kernel, csrc/tr_guide.hip) at the edges of its thread rows."""
import numpy as np
import pytest

from oracle import guide_ref as G
from tests.test_guide_gpu import _records

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 64, 65, 16 * 64, 16 * 64 + 1, 17 * 64 + 5, 40 * 64 - 1])
def test_gradient_is_the_mean_of_its_tiles(n):
    """With unit weights (whose mean is 1 for any batch) a tile of 64 records gives the same partial
    alone and in a larger batch, so the gradient over n records is the mean of the tiles' sums: both
    are rounded to float once (2^-24 of the value, and of each tile's share). Record j of a call is
    read at (j (2^31 - 1)) mod n, so a tile alone is laid out to be read in the batch's order."""
    from jarabotransientrendering_amd import renderer
    g = renderer.PathGuide(init_seed=3, batch_size=4096)
    g.params = G.initial_like(seed=8, out_scale=1.0)
    rec = _records(np.random.default_rng(n), n)
    rec[:, 11] = 1.0
    grad, loss = g.gradient(rec)
    step = 2 ** 31 - 1
    order = rec[np.arange(n) * step % n]
    tiles = []
    for k in range(0, n, 64):
        tile = order[k:k + 64]
        alone = np.empty_like(tile)
        alone[np.arange(len(tile)) * step % len(tile)] = tile
        tiles.append((len(tile), *g.gradient(alone)))
    expect = sum(m * t.astype(np.float64) for m, t, _ in tiles) / n
    bound = 2.0 ** -23 * sum(m * np.abs(t.astype(np.float64)) for m, t, _ in tiles) / n
    assert (np.abs(grad - expect) <= bound + 1e-30).all()
    assert abs(loss - sum(m * l for m, _, l in tiles) / n) <= 2.0 ** -22 * max(abs(l) for _, _, l in tiles)

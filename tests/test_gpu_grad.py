"""Weight gradients at batch sizes where the splits and the waves of a split run out of tiles (16 samples a tile, 56
splits, 8 waves): a batch's gradient is the mean of its parts' gradients, taken over parts of one wave's single tile
and added up in float64.  A sample's forward and backward do not depend on its batch, so only float32 sums differ:
up to n / 448 + 60 additions in a row, 2^-24 each, over terms that partly cancel."""
import numpy as np
import pytest

from test_gpu_cache import layer_errors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [16, 16 * 56 - 5, 16 * 56 + 1, 16 * 56 * 8, 16 * 56 * 8 + 3])
def test_gradient_is_mean_of_parts(ctx, vtapi, n):
    rng = np.random.default_rng(n)
    cache = vtapi.RadianceCache(ctx, seed=3)
    raw = rng.uniform(0, 1, (n, 12)).astype(np.float32)
    tgt = rng.uniform(0, 3, (n, 3)).astype(np.float32)
    g, loss = cache.gradient(raw, tgt)
    want, lwant = np.zeros(len(g)), 0.0
    for i in range(0, n, 16):
        gi, li = cache.gradient(raw[i:i + 16], tgt[i:i + 16])
        k = len(raw[i:i + 16]) / n
        want += k * gi.astype(np.float64)
        lwant += k * float(li)
    cache.close()
    assert abs(loss - lwant) <= 1e-5 * lwant
    err = layer_errors(g, want)
    assert np.all(err <= 2e-5), err

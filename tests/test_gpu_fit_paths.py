"""Fits of narrow blocks on both sides of the lines between streamed sums and lists of members, and between blocks of their
own width and padded ones: centroids against the CPU oracle, bit for bit."""
import numpy as np
import pytest

from oracle import oracle as O
from tests import data

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.mark.parametrize("n,m,sd,k", [
    (40_000, 40, 8, 75), (66_000, 48, 8, 40), (66_000, 48, 8, 24), (70_000, 16, 8, 16), (120_000, 20, 8, 40), (120_000, 26, 8, 20),
    (110_000, 33, 7, 46), (110_000, 33, 7, 4), (60_000, 12, 6, 24), (60_000, 12, 6, 60), (90_000, 5, 3, 90), (200_000, 5, 2, 200),
    (50_000, 4, 12, 39), (50_000, 4, 12, 40), (30_000, 3, 10, 20), (30_000, 4, 10, 20), (26_000, 2, 25, 35), (26_000, 2, 25, 36),
    (66_000, 40, 8, 40), (70_000, 40, 8, 40), (72_000, 40, 8, 40), (61_440, 49, 8, 40), (61_441, 49, 8, 40), (61_440, 55, 8, 30), (61_441, 55, 8, 30), (90_000, 32, 3, 20), (90_000, 33, 3, 100)])
def test_fit(n, m, sd, k):
    import vq_amd
    ctx = vq_amd.Context(0)
    x = np.random.default_rng(n + sd + k).random((n, m * sd), dtype=F)
    init, reseed = data.index_streams(n, m, k, 2, seed=3)
    cb = ctx.empty((m, k, sd), F)
    ctx.lbg_fit(ctx.to_device(x), n, m * sd, m, sd, k, 2, init, reseed, cb)
    want = O.pq_fit(x, m, k, 2, init, reseed)["codebooks"]
    assert np.array_equal(cb.download().view(np.uint32), want.view(np.uint32))
    ctx.close()

"""Leaf sums by a workgroup per leaf and tile of components: widths around the pieces and the tiles of 32, leaves of one
member to whole parts of 4096, both sides of the sizes from which a lane takes a component, spaced and unaligned rows."""
import numpy as np
import pytest

from oracle import oracle as O
from tests import data

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.mark.parametrize("n,m,sd,k,extra,skew", [
    (14_000, 3, 1, 5, 0, 0), (14_000, 3, 2, 40, 1, 0), (14_000, 2, 3, 17, 0, 0), (14_000, 3, 5, 16, 0, 0), (14_000, 2, 7, 30, 3, 0),
    (14_000, 1, 31, 9, 0, 0), (14_000, 2, 33, 20, 1, 0), (14_000, 1, 36, 20, 0, 0), (14_000, 1, 65, 64, 2, 0), (14_000, 1, 300, 22, 0, 0),
    (3000, 1, 1025, 20, 0, 0), (2500, 1, 1057, 130, 1, 0), (20_000, 1, 24, 3, 0, 1), (20_000, 2, 6, 8, 0, 1), (70_000, 1, 40, 66, 0, 0), (70_000, 1, 4, 65, 0, 0), (300_000, 1, 20, 256, 0, 0),
    (270_000, 4, 16, 256, 0, 0), (262_145, 1, 5, 250, 2, 0)])
def test_fit(n, m, sd, k, extra, skew):
    import vq_amd
    ctx = vq_amd.Context(0)
    rng = np.random.default_rng(n + sd)
    ld = m * sd + extra
    buf = rng.random((n, ld)).astype(F)
    if skew:  # most rows in one cluster: leaves of whole parts
        buf[rng.random(n) < 0.95] *= F(1e-2)
    init, reseed = data.index_streams(n, m, k, 3, seed=7)
    cb = ctx.empty((m, k, sd), F)
    dx = ctx.to_device(buf)
    ctx.lbg_fit(dx, n, ld, m, sd, k, 3, init, reseed, cb)
    want = O.pq_fit(np.ascontiguousarray(buf[:, :m * sd]), m, k, 3, init, reseed)["codebooks"]
    assert np.array_equal(cb.download().view(np.uint32), want.view(np.uint32))
    ctx.close()

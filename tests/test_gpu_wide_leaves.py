"""Sums of wide column blocks: leaves of every length class (short, long, very long, empty), several column blocks,
widths at the edges of a workgroup, rows shuffled and in the order of their clusters; bit for bit.  The leaves are taken in
an order of their own (k_lbg_leafsum_wide) from 300,000 rows and 100 million floats on, in block order below that."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module")
def ctx():
    import vq_amd
    c = vq_amd.Context(0)
    yield c
    c.close()


SIZES = [1, 15, 16, 17, 64, 65, 127, 128, 129, 511, 512, 1024, 1025, 2500, 8000, 12_300]


ORDERED = [(1, 64, 1_570_000, "shuffled"), (2, 161, 311_000, "shuffled"), (1, 333, 302_000, "sorted"), (1, 257, 390_000, "reversed"),
           (1, 100, 1_001_000, "sorted"), (1, 128, 790_000, "shuffled"), (1, 128, 790_000, "sorted"), (1, 512, 300_100, "shuffled"),
           (1, 512, 300_100, "reversed"), (3, 100, 340_000, "shuffled"), (3, 128, 301_000, "reversed"), (2, 256, 300_001, "shuffled")]


@pytest.mark.parametrize("m,sd,n,order", [(m, sd, 0, order) for order in ("shuffled", "sorted", "reversed") for m, sd in
                                          [(1, 64), (2, 65), (1, 128), (1, 256), (1, 257), (3, 100), (1, 512)]] + ORDERED)
def test_leaves(ctx, m, sd, n, order):
    rng = np.random.default_rng(sd)
    sizes = SIZES + ([n // 3, n - sum(SIZES) - n // 3] if n else [])
    label = np.repeat(np.arange(len(sizes)), sizes)
    label = label if order == "sorted" else label[::-1] if order == "reversed" else rng.permutation(label)
    assert not n or (n >= 300_000 and n * m * sd >= 100_000_000)  # in an order of their own
    n, k = len(label), len(sizes)
    x = rng.standard_normal((n, m * sd), dtype=F)
    x += (50 * label[:, None]).astype(F)
    init = np.tile(np.array([np.flatnonzero(label == j)[0] for j in range(k)], np.uint32), (m, 1))
    reseed = rng.integers(0, n, (m, 3 * k), dtype=np.uint32)
    want = O.pq_fit(x, m, k, 3, init, reseed)
    cb = ctx.empty((m, k, sd), F)
    it, _ = ctx.lbg_fit(ctx.to_device(x), n, m * sd, m, sd, k, 3, init, reseed, cb)
    assert np.array_equal(it, want["iters"])
    assert np.array_equal(cb.download().view(np.uint32), want["codebooks"].view(np.uint32))

"""Tree builds over rows that are copied with zeros behind them (widths that are no multiple of 8): both sides of the
numbers of rows from which they are, data whose variances are all zero, ties, infinities, spaced and unaligned rows."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.test_gpu_tsvq import assert_same_tree, bfs_order

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.mark.parametrize("n,dim,extra,depth,kind", [
    (2048, 50, 0, 4, "normal"), (2049, 50, 0, 4, "normal"), (2049, 1, 0, 3, "normal"), (3000, 7, 2, 12, "grid"), (8192, 100, 0, 3, "normal"),
    (8193, 100, 0, 3, "normal"), (8200, 100, 1, 3, "normal"), (20_000, 50, 0, 9, "normal"), (2600, 9, 0, 3, "same"), (40_000, 3, 0, 2, "same"),
    (140_000, 5, 0, 3, "normal"), (2500, 33, 0, 3, "inf"), (5000, 30, 0, 13, "normal")])
def test_build(n, dim, extra, depth, kind):
    import vq_amd
    ctx = vq_amd.Context(0)
    rng = np.random.default_rng(n + dim)
    buf = rng.standard_normal((n, dim + extra)).astype(F)
    if kind == "grid":
        buf = np.round(buf * 2).astype(F)
    elif kind == "same":
        buf[:] = np.arange(dim + extra, dtype=F)
    elif kind == "inf":
        buf[::501, 3] = F(1e30)
        buf[1::503, 7] = F(-np.inf)
    got = ctx.tsvq_build(ctx.to_device(buf), n, dim + extra, dim, depth).download()
    want, _ = bfs_order(O.tsvq_fit(np.ascontiguousarray(buf[:, :dim]), depth))
    if kind == "inf":  # means and variances of a column with infinities are no numbers: the same ones, whatever their sign bit
        nan = np.isnan(want["centroids"])
        assert np.array_equal(np.isnan(got["centroids"]), nan)
        got["centroids"][nan] = want["centroids"][nan] = F(0)
    assert_same_tree(got, want)
    ctx.close()

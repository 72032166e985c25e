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
    (140_000, 5, 0, 3, "normal"), (2500, 33, 0, 3, "inf"), (5000, 30, 0, 13, "normal"),
    (8192, 50, 0, 4, "normal"), (8193, 50, 2, 4, "normal"), (8193, 1, 0, 3, "normal"), (9000, 7, 2, 12, "grid"), (8193, 87, 0, 3, "normal"), (16_384, 100, 0, 3, "normal"),
    (16_385, 100, 1, 3, "normal"), (16_385, 95, 0, 3, "normal"), (9000, 9, 0, 3, "same"), (9000, 33, 0, 3, "inf")])
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


@pytest.mark.parametrize("n,dim,depth", [(8193, 262_133, 1), (8193, 262_139, 1), (8193, 262_144, 1), (5, 1_048_603, 2)])
def test_widths_around_the_grids_limit(n, dim, depth):
    """Rows whose columns, four or sixteen to a workgroup, pass 65,535 workgroups: all zeros but eight columns, so that the tree is
    the one of those columns."""
    import vq_amd
    ctx = vq_amd.Context(0)
    rng = np.random.default_rng(dim)
    cols = np.concatenate([[0], np.sort(rng.choice(np.arange(1, dim - 1), 6, replace=False)), [dim - 1]])
    part = rng.standard_normal((n, 8)).astype(F)
    x = np.zeros((n, dim), F)
    x[:, cols] = part
    got = ctx.tsvq_build(ctx.to_device(x), n, dim, dim, depth).download()
    want, _ = bfs_order(O.tsvq_fit(part, depth))
    rest = np.ones(dim, bool)
    rest[cols] = False
    assert not got["centroids"][:, rest].any()
    got["centroids"] = np.ascontiguousarray(got["centroids"][:, cols])
    want["split_dim"] = np.where(want["split_dim"] < 0, -1, cols[want["split_dim"]]).astype(want["split_dim"].dtype)
    assert_same_tree(got, want)
    ctx.close()


@pytest.mark.parametrize("dim", [262_133, 262_139, 262_144])
def test_composed_maps_around_the_grids_limit(dim):
    """The same widths with more rows than a node that is taken by tiles: the composed maps up to 262,140 columns (65,535 workgroups
    of four), the tiles beyond and, where the padded width is above it, for 262,139."""
    import vq_amd
    ctx = vq_amd.Context(0)
    n = 16_385
    rng = np.random.default_rng(dim)
    cols = np.concatenate([[0], np.sort(rng.choice(np.arange(1, dim - 1), 6, replace=False)), [dim - 1]])
    part = rng.standard_normal((n, 8)).astype(F)
    x = np.zeros((n, dim), F)  # (17 GB, of which the host holds the pages written)
    x[:, cols] = part
    got = ctx.tsvq_build(ctx.to_device(x), n, dim, dim, 1).download()
    want, _ = bfs_order(O.tsvq_fit(part, 1))
    rest = np.ones(dim, bool)
    rest[cols] = False
    assert not got["centroids"][:, rest].any()
    got["centroids"] = np.ascontiguousarray(got["centroids"][:, cols])
    want["split_dim"] = np.where(want["split_dim"] < 0, -1, cols[want["split_dim"]]).astype(want["split_dim"].dtype)
    assert_same_tree(got, want)
    ctx.close()

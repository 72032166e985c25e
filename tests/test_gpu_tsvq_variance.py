"""Variances by a workgroup per node and tile of columns: widths around the pieces and the tiles of 16, spaced and unaligned rows,
both sides of the node sizes from which the composed maps are taken (8192 rows, 16,384 from 89 columns on).  Shorter nodes
are k_node_stats' by default and k_seg_variance_tile's where the levels are the host's."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.test_gpu_tsvq import assert_same_tree, bfs_order

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.mark.parametrize("n,dim,extra,depth", [
    (1, 5, 0, 2), (2, 1, 0, 2), (300, 1, 0, 5), (300, 2, 1, 5), (513, 3, 0, 4), (1025, 4, 3, 4), (700, 15, 0, 6), (700, 17, 0, 6), (700, 33, 2, 9),
    (4096, 20, 0, 3), (4097, 20, 0, 3), (4096, 16, 0, 8), (4097, 16, 0, 2), (8192, 96, 0, 3), (8193, 96, 0, 3), (8192, 99, 0, 2), (8193, 99, 1, 2),
    (1500, 1100, 0, 3), (12_000, 8, 0, 12),
    (8192, 20, 0, 3), (8193, 20, 0, 3), (8193, 16, 0, 2), (16_384, 96, 0, 3), (16_385, 96, 0, 3), (16_384, 99, 0, 2), (16_385, 99, 1, 2),
    (8193, 88, 0, 2), (16_384, 88, 0, 3), (8193, 89, 0, 2), (16_384, 89, 1, 3), (16_385, 89, 0, 2), (16_384, 95, 0, 3)])
def test_build(n, dim, extra, depth):
    import vq_amd
    ctx = vq_amd.Context(0)
    rng = np.random.default_rng(n + dim)
    buf = (rng.standard_normal((n, dim + extra)) * 10.0 ** rng.integers(-3, 4, dim + extra)).astype(F)
    got = ctx.tsvq_build(ctx.to_device(buf), n, dim + extra, dim, depth).download()
    want, _ = bfs_order(O.tsvq_fit(np.ascontiguousarray(buf[:, :dim]), depth))
    assert_same_tree(got, want)
    ctx.close()


@pytest.mark.parametrize("n,dim,extra,depth,kind", [
    # by chains: chunks of 336 members, one to three components, a last tile that overlaps
    (335, 13, 0, 1, "normal"), (337, 13, 0, 1, "normal"), (673, 13, 0, 1, "normal"), (2000, 1, 0, 4, "normal"), (2000, 3, 1, 5, "integers"), (3001, 50, 0, 4, "normal"),
    (8192, 50, 0, 4, "normal"), (16_384, 99, 0, 3, "normal"), (1000, 1100 + 3, 0, 2, "normal"), (4097, 20 + 2, 0, 4, "zeros"), (4097, 22, 0, 4, "tiny"),
    # more workgroups than three to a compute unit in the lower levels: tiles of up to 32 components
    (8192, 50, 1, 10, "normal"), (6000, 99, 0, 9, "integers"), (4000, 3, 0, 12, "normal"), (5000, 33, 0, 10, "huge"), (3000, 300 + 1, 0, 7, "normal")])
def test_tiles_of_levels_by_the_host(n, dim, extra, depth, kind):
    import vq_amd
    ctx = vq_amd.Context(0)
    ctx.set_tsvq_variance_path(1)  # (widths that are no multiple of 8 and not padded: k_seg_variance_tile)
    rng = np.random.default_rng(n + dim)
    buf = rng.standard_normal((n, dim + extra)).astype(F)
    if kind == "integers":
        buf = np.round(buf * 3).astype(F)
    elif kind == "zeros":
        buf[:] = 0
    elif kind in ("tiny", "huge"):
        buf = (buf * F(1e-22 if kind == "tiny" else 1e15)).astype(F)
    got = ctx.tsvq_build(ctx.to_device(buf), n, dim + extra, dim, depth).download()
    want, _ = bfs_order(O.tsvq_fit(np.ascontiguousarray(buf[:, :dim]), depth))
    assert_same_tree(got, want)
    ctx.close()


@pytest.mark.parametrize("n,dim,depth", [
    (9000, 4100, 13),   # the deepest tree's means above 256 MB: no level on the device
    (5000, 4000, 12)])  # a level of more than 500 such nodes: the host's again below levels on the device
def test_levels_that_return_to_the_host(n, dim, depth):
    import vq_amd
    ctx = vq_amd.Context(0)
    x = np.random.default_rng(n).standard_normal((n, dim), dtype=F)
    got = ctx.tsvq_build(ctx.to_device(x), n, dim, dim, depth).download()
    want, _ = bfs_order(O.tsvq_fit(x, depth))
    assert_same_tree(got, want)
    ctx.close()

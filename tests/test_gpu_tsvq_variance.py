"""Variances by a workgroup per node and tile of columns: widths around the pieces and the tiles of 16, spaced and unaligned rows,
both sides of the node sizes from which the composed maps are taken."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.test_gpu_tsvq import assert_same_tree, bfs_order

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.mark.parametrize("n,dim,extra,depth", [
    (1, 5, 0, 2), (2, 1, 0, 2), (300, 1, 0, 5), (300, 2, 1, 5), (513, 3, 0, 4), (1025, 4, 3, 4), (700, 15, 0, 6), (700, 17, 0, 6), (700, 33, 2, 9),
    (4096, 20, 0, 3), (4097, 20, 0, 3), (4096, 16, 0, 8), (4097, 16, 0, 2), (8192, 96, 0, 3), (8193, 96, 0, 3), (8192, 99, 0, 2), (8193, 99, 1, 2),
    (1500, 1100, 0, 3), (12_000, 8, 0, 12)])
def test_build(n, dim, extra, depth):
    import vq_amd
    ctx = vq_amd.Context(0)
    rng = np.random.default_rng(n + dim)
    buf = (rng.standard_normal((n, dim + extra)) * 10.0 ** rng.integers(-3, 4, dim + extra)).astype(F)
    got = ctx.tsvq_build(ctx.to_device(buf), n, dim + extra, dim, depth).download()
    want, _ = bfs_order(O.tsvq_fit(np.ascontiguousarray(buf[:, :dim]), depth))
    assert_same_tree(got, want)
    ctx.close()

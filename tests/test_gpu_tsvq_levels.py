"""TSVQ levels built without the host between them (k_node_leafsum, k_node_stats, k_node_split): trees that are not
balanced, so that nodes are longer than a launch expects (their keys in memory, their leaves summed in rounds), slots
without a node, levels by the host above them, more levels than one table holds, few components; against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.test_gpu_tsvq import assert_same_tree, bfs_order

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module")
def ctx():
    import vq_amd
    c = vq_amd.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("n,dim,depth,kind", [
    (4096, 10, 6, "lopsided"), (8192, 100, 7, "lopsided"), (8000, 97, 5, "lopsided"), (3000, 3, 8, "normal"),
    (20000, 8, 8, "lopsided"), (30000, 96, 7, "lopsided"), (700, 1, 10, "normal"), (40, 6, 13, "normal"), (2100, 4, 14, "lopsided"),
    (6000, 17, 12, "copies"), (257, 20, 1, "normal"), (5, 2, 3, "copies"), (9000, 33, 9, "copies"),
    # a chain's chunks of 336 members (16 components) and the ends of its two stages, three components, a last tile that overlaps
    (335, 16, 1, "normal"), (336, 16, 1, "normal"), (337, 16, 1, "normal"), (672, 16, 1, "normal"), (1009, 20, 1, "normal"), (900, 3, 1, "normal"),
    # the longest nodes: sixteen leaves, 68 KB of LDS for the split
    (16_384, 100, 6, "normal"), (16_385, 100, 4, "normal"), (16_384, 96, 5, "lopsided"), (8193, 50, 5, "lopsided"),
    # more workgroups than a round: tiles of up to 32 components, nodes of some hundred rows and of two leaves
    (30_000, 256, 7, "normal"), (40_000, 100, 8, "normal"), (26_000, 250, 6, "lopsided"), (90_000, 130, 6, "normal"),
    # levels that end because a node is longer than three times a balanced tree's: once and again, at the last level of the tree,
    # one above it, an odd and an even number of levels early, many nodes above them, three components
    (16_384, 100, 9, "one of fifty"), (9000, 100, 2, "one of fifty"), (9000, 100, 3, "one of fifty"), (8000, 96, 4, "one of fifty"), (5000, 17, 5, "one of fifty"),
    (8192, 3, 10, "one of fifty"), (60_000, 130, 8, "one of fifty"), (6000, 24, 7, "even above"), (6001, 24, 8, "even above"),
])
def test_levels_on_device(ctx, n, dim, depth, kind):
    rng = np.random.default_rng(17 * n + dim)
    x = rng.standard_normal((n, dim)).astype(F)
    if kind == "lopsided":  # every column: four rows of five share the least value, which is the median
        x = np.where(rng.random((n, dim)) < 0.8, F(0.0), np.abs(x) * F(10) + F(1)).astype(F) * np.arange(1, dim + 1, dtype=F)
    elif kind == "one of fifty":  # a node loses one row in fifty per level
        x = np.where(rng.random((n, dim)) < 0.98, F(0.0), np.abs(x) + F(1)).astype(F)
    elif kind == "even above":  # three balanced levels, then equal values
        x = np.where(rng.random((n, dim)) < 0.9, F(0.0), F(1.0)).astype(F) * np.arange(1, dim + 1, dtype=F) * F(0.01)
        x[:, :3] = rng.standard_normal((n, 3)) * [400, 200, 100]
    elif kind == "copies":  # few distinct rows: nodes of equal rows have no children
        x = x[rng.integers(0, min(n, 9), n)]
    got = ctx.tsvq_build(ctx.to_device(x), n, dim, dim, depth).download()
    want, _ = bfs_order(O.tsvq_fit(x, depth))
    assert_same_tree(got, want)

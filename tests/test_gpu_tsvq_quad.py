"""Descents by four lanes per row: widths around the pieces of 4 and 16 components, spaced and unaligned rows, trees
whose nodes are in LDS, in the table beyond it and beyond the table, numbers of rows around a wave's 16, rows and
centroids that the margins cannot decide."""
from types import SimpleNamespace

import numpy as np
import pytest

from oracle import oracle as O
from tests.test_gpu_tsvq import _hand_tree

pytestmark = pytest.mark.gpu
F = np.float32
METRICS = [O.SQEUCLIDEAN, O.EUCLIDEAN, O.COSINE, O.MANHATTAN]


@pytest.fixture(scope="module")
def ctx():
    import vq_amd
    c = vq_amd.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("metric", METRICS)
@pytest.mark.parametrize("n,dim,extra,offset,depth", [
    (1, 1, 0, 0, 3), (15, 3, 0, 0, 4), (17, 5, 2, 1, 4), (129, 15, 0, 0, 5), (700, 16, 1, 3, 6), (700, 17, 0, 0, 6),
    (700, 31, 0, 2, 9), (3000, 50, 0, 0, 10), (700, 64, 0, 0, 10), (700, 100, 0, 0, 8), (700, 112, 3, 0, 5),
    (5000, 128, 0, 0, 9), (700, 129, 0, 0, 5), (700, 161, 0, 0, 7), (700, 208, 0, 0, 6), (2500, 248, 0, 0, 11),
    (700, 256, 4, 0, 8), (700, 257, 0, 0, 4), (70_000, 9, 0, 0, 12),
    # a lane per row, and the first that are not
    (700, 1, 1, 0, 10), (70_000, 2, 0, 1, 6), (700, 3, 2, 0, 8), (700, 3, 0, 1, 9), (700, 4, 0, 0, 3), (700, 4, 1, 1, 4), (3000, 7, 0, 0, 2), (600, 15, 0, 0, 1),
    (600, 16, 0, 0, 1), (100_001, 5, 0, 0, 4), (600, 32, 0, 0, 0)])
def test_widths_and_depths(ctx, metric, n, dim, extra, offset, depth):
    rng = np.random.default_rng(n + dim)
    nn = 2 ** (depth + 1) - 1
    cen = rng.standard_normal((nn, dim)).astype(F)
    ld = dim + extra
    buf = rng.standard_normal(n * ld + offset).astype(F)
    q = np.lib.stride_tricks.as_strided(buf[offset:], (n, dim), (4 * ld, 4))
    tree, otree = _hand_tree(ctx, cen, depth)
    dbuf = ctx.to_device(buf)
    leaf = ctx.empty(n, np.int32)
    ctx.tsvq_descend(metric, SimpleNamespace(ptr=dbuf.ptr + 4 * offset), n, ld, tree, leaf)
    assert np.array_equal(leaf.download(), O.tsvq_descend(metric, np.ascontiguousarray(q), otree))


@pytest.mark.parametrize("metric", METRICS)
@pytest.mark.parametrize("dim,depth", [(20, 5), (100, 11), (250, 9)])
@pytest.mark.parametrize("kind", ["grid", "scales", "zeros", "non_finite", "far", "same"])
def test_undecided_rows(ctx, metric, dim, depth, kind):
    """Ties of whole numbers, lengths from 1e-20 to 1e18, zero vectors, infinities and NaN, rows whose differences are
    near the last bit, children that are equal: at every level, in LDS or not."""
    rng = np.random.default_rng(dim)
    nn, n = 2 ** (depth + 1) - 1, 700
    cen = rng.standard_normal((nn, dim)).astype(F)
    q = rng.standard_normal((n, dim)).astype(F)
    if kind == "grid":
        cen, q = np.round(cen).astype(F), np.round(q).astype(F)
    elif kind == "scales":
        q = (q * np.exp(rng.uniform(np.log(1e-20), np.log(1e18), (n, 1)))).astype(F)
        cen = (cen * np.exp(rng.uniform(np.log(1e-18), np.log(1e16), (nn, 1)))).astype(F)
    elif kind == "zeros":
        q[::5] = 0.0
        cen[rng.integers(0, nn, nn // 4)] = 0.0
    elif kind == "non_finite":
        q[::11, 3] = np.nan
        q[5::13, 7] = np.inf
        q[6::17, 2] = -np.inf
        cen[6::31, 1] = np.nan
        cen[11::37, 0] = np.inf
    elif kind == "far":
        cen, q = (1000.0 + cen * 1e-3).astype(F), (1000.0 + q * 1e-3).astype(F)
    else:
        cen[2::2] = cen[1::2]
    tree, otree = _hand_tree(ctx, cen, depth)
    with np.errstate(all="ignore"):
        want = O.tsvq_descend(metric, q, otree)
    leaf = ctx.empty(n, np.int32)
    ctx.tsvq_descend(metric, ctx.to_device(q), n, dim, tree, leaf)
    assert np.array_equal(leaf.download(), want)


@pytest.mark.parametrize("metric", METRICS)
@pytest.mark.parametrize("dim", [32, 64, 96, 128])
def test_many_rows_of_register_widths(ctx, metric, dim):
    """Beyond 65,536 rows and up to 255 inner nodes rows are held by one lane each: the same leaves as two distances per node."""
    rng = np.random.default_rng(dim)
    cen, q = np.round(rng.standard_normal((511, dim)) * 2).astype(F), np.round(rng.standard_normal((66_000, dim)) * 2).astype(F)
    q[::501] = 0.0
    q[::499, 1] = np.inf
    tree, otree = _hand_tree(ctx, cen, 8)
    dq = ctx.to_device(q)
    with np.errstate(all="ignore"):
        want = O.tsvq_descend(metric, q, otree)
    for n in (65_536, 65_537, len(q)):
        leaf = ctx.to_device(np.full(len(q), -1, np.int32))
        ctx.tsvq_descend(metric, dq, n, dim, tree, leaf)
        assert np.array_equal(leaf.download(), np.where(np.arange(len(q)) < n, want, -1)), n

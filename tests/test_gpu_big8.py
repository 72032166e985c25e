"""Column blocks of 8 and 16 floats (and of widths padded to them) with 257 to 2048 and 1024 centroids in one pass: codes against the
CPU oracle at the edges of the centroid tiles, of the two workgroup sizes and of the row tiles, for badly scaled,
tied and non-finite input."""
import numpy as np
import pytest

from oracle import oracle as O
from tests import data
from tests.test_gpu_wide_bound import _case

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module")
def ctx():
    import vq_amd
    c = vq_amd.Context(0)
    c.set_few_path(1)
    yield c
    c.close()


def _check(ctx, x, cb, metric, ld=None):
    m, k, sd = cb.shape
    n, dim = x.shape
    rows = np.full((n, ld or dim), np.nan, F)
    rows[:, :dim] = x
    codes = ctx.empty((n, m), np.uint16)
    ctx.assign_u16(metric, ctx.to_device(rows), n, rows.shape[1], m, sd, k, ctx.to_device(cb), codes)
    with np.errstate(all="ignore"):
        want = O.pq_encode(metric, x, cb)
    assert np.array_equal(codes.download(), want.astype(np.uint16))


@pytest.mark.parametrize("kind", ["normal", "collapsed", "near_ties", "grid", "spread", "overflow", "tiny", "offset", "edges"])
@pytest.mark.parametrize("metric", [O.SQEUCLIDEAN, O.EUCLIDEAN, O.COSINE])
@pytest.mark.parametrize("n,m,k,sd", [(700, 3, 257, 8), (1300, 2, 1000, 8), (333, 2, 2048, 8), (700, 2, 300, 16), (300, 2, 1024, 16)])
def test_codes(ctx, n, m, k, sd, metric, kind):
    x, cb = _case(kind, n, m, sd, k)
    _check(ctx, x, cb, metric)


@pytest.mark.parametrize("k", [300, 320, 321, 511, 513, 1024, 1216, 1217, 1985, 2047])
@pytest.mark.parametrize("n,m,sd", [(1, 600, 8), (33, 20, 8), (5000, 1, 8), (2049, 3, 7), (900, 2, 5), (2049, 2, 16), (700, 3, 11)])
def test_sizes(ctx, n, m, sd, k):
    rng = np.random.default_rng(k + n)
    x, cb = rng.random((n, m * sd), dtype=F), rng.random((m, k, sd), dtype=F)
    if sd > 8 and k > 1024:
        pytest.skip("chunk by chunk: test_gpu_big_k.py")
    cb[:, k - 1] = cb[:, 3]  # a tie of the last centroid with an early one
    cb[:, k // 2] = cb[:, k // 2 - 1]  # and of neighbours
    x[: n // 3] = cb[np.arange(m), :][:, rng.integers(0, k, n // 3)].transpose(1, 0, 2).reshape(n // 3, m * sd)
    _check(ctx, x, cb, O.EUCLIDEAN, ld=m * sd + 3)


def test_codebook_off_alignment(ctx):
    """A codebook that starts at any float goes chunk by chunk, as a codebook above 2048 does."""
    rng = np.random.default_rng(1)
    x, cb = rng.standard_normal((600, 16)).astype(F), rng.standard_normal((2, 400, 8)).astype(F)
    raw = ctx.to_device(np.concatenate([np.zeros(1, F), cb.ravel()]))
    codes = ctx.empty((600, 2), np.uint16)
    ctx.assign_u16(O.SQEUCLIDEAN, ctx.to_device(x).ptr, 600, 16, 2, 8, 400, raw.ptr + 4, codes.ptr)
    assert np.array_equal(codes.download(), O.pq_encode(O.SQEUCLIDEAN, x, cb).astype(np.uint16))
    big = rng.standard_normal((1, 2100, 8)).astype(F)
    _check(ctx, x[:, :8].copy(), big, O.SQEUCLIDEAN)


@pytest.mark.parametrize("metric", [O.SQEUCLIDEAN, O.EUCLIDEAN])
@pytest.mark.parametrize("sd,k", [(16, 35), (16, 63), (16, 319), (16, 1023), (8, 319), (8, 2047)])  # one padding centroid in the last set
def test_block_around_the_padding(ctx, sd, k, metric):
    """A block far from the origin, by any place that padding centroids could be given: none of them is ever chosen."""
    rng = np.random.default_rng(k)
    for off in (1e18, -1e18, 1e15, 0.0):
        x = (F(off) + F(3e12) * rng.standard_normal((4000, 2 * sd)).astype(F)).astype(F)
        cb = (F(off) + F(1e13) * rng.standard_normal((2, k, sd)).astype(F)).astype(F)
        if k > 256:
            _check(ctx, x, cb, metric)
            continue
        codes = ctx.empty((4000, 2), np.uint8)
        ctx.assign(metric, ctx.to_device(x), 4000, 2 * sd, 2, sd, k, ctx.to_device(cb), codes)
        assert np.array_equal(codes.download(), O.pq_encode(metric, x, cb).astype(np.uint8))


def test_fit_around_the_padding(ctx):
    n, m, sd, k = 5000, 2, 16, 35
    rng = np.random.default_rng(3)
    x = (F(1e18) + F(1e13) * rng.standard_normal((n, m * sd)).astype(F)).astype(F)
    init, reseed = data.index_streams(n, m, k, 4, seed=k)
    cb = ctx.empty((m, k, sd), F)
    ctx.lbg_fit(ctx.to_device(x), n, sd * m, m, sd, k, 4, init, reseed, cb)
    assert np.array_equal(cb.download().view(np.uint32), O.pq_fit(x, m, k, 4, init, reseed)["codebooks"].view(np.uint32))

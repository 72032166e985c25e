"""Column blocks of widths that the register kernel holds with zeros behind them, on both sides of the number of
centroids from which rows are padded for the matrix-core kernels: codes and centroids against the CPU oracle, bit for bit."""
import numpy as np
import pytest

from oracle import oracle as O
from tests import data

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module")
def ctx():
    import vq_amd
    c = vq_amd.Context(0)
    c.set_few_path(1)  # short calls, too, by the kernels named here
    yield c
    c.close()


# n, m, sub_dim, k, extra columns of the row buffer: the first and last width of every register width, tiles of 256
# rows and their neighbours, two and four blocks per lane, k below and above each line
CASES = [(255, 4, 7, 2, 0), (256, 2, 7, 31, 1), (257, 3, 7, 47, 0), (513, 4, 7, 48, 0), (300, 2, 9, 3, 0), (1000, 4, 11, 39, 2), (257, 1, 10, 59, 0),
         (700, 2, 10, 60, 0), (300, 2, 13, 40, 1), (511, 3, 15, 59, 0), (513, 1, 17, 5, 0), (400, 3, 20, 60, 0), (300, 1, 23, 59, 0),
         (129, 2, 24, 17, 1), (600, 2, 25, 31, 0), (257, 1, 31, 60, 0), (300, 2, 33, 16, 0), (65, 1, 47, 256, 3), (260, 1, 48, 31, 1),
         (300, 1, 49, 17, 0), (257, 1, 100, 30, 1), (500, 2, 5, 31, 0), (1, 1, 20, 1, 0)]


@pytest.mark.parametrize("n,m,sd,k,extra", CASES)
def test_encode(ctx, n, m, sd, k, extra):
    import vq_amd
    rng = np.random.default_rng(100 * n + sd)
    dim, ld = m * sd, m * sd + extra
    buf = rng.standard_normal((n, ld)).astype(F)
    cb = rng.standard_normal((m, k, sd)).astype(F)
    buf[n // 2, :sd] = 0.0        # a zero row and a zero centroid (cosine), equal centroids (ties), values that are no numbers
    cb[0, k // 2] = 0.0
    cb[m - 1, k - 1] = cb[m - 1, 0]
    buf[n // 3, dim - 1] = np.inf
    buf[n // 5, 0] = np.nan
    x = np.ascontiguousarray(buf[:, :dim])
    dx, dcb, codes = ctx.to_device(buf), ctx.to_device(cb), ctx.empty((n, m), np.uint8)
    for metric, om in ((vq_amd.SQEUCLIDEAN, O.SQEUCLIDEAN), (vq_amd.EUCLIDEAN, O.EUCLIDEAN), (vq_amd.COSINE, O.COSINE),
                       (vq_amd.MANHATTAN, O.MANHATTAN)):
        ctx.assign(metric, dx, n, ld, m, sd, k, dcb, codes)
        assert np.array_equal(codes.download(), O.pq_encode(om, x, cb).astype(np.uint8)), metric


# with a small update behind it (the rows are padded) and without
@pytest.mark.parametrize("n,m,sd,k", [(900, 4, 7, 2), (5000, 3, 10, 30), (3000, 2, 20, 16), (30_000, 2, 15, 24), (700, 1, 100, 17), (1200, 2, 3, 20),
                                      (9000, 1, 25, 59)])
def test_fit(ctx, n, m, sd, k):
    rng = np.random.default_rng(n + sd)
    x = rng.random((n, m * sd), dtype=F)
    init, reseed = data.index_streams(n, m, k, 4, seed=n)
    dcb = ctx.empty((m, k, sd), F)
    ctx.lbg_fit(ctx.to_device(x), n, m * sd, m, sd, k, 4, init, reseed, dcb)
    ref = O.pq_fit(x, m, k, 4, init, reseed)
    assert np.array_equal(dcb.download().view(np.uint32), ref["codebooks"].view(np.uint32))


def test_encode_in_slices(ctx):
    """More rows than one padded slice holds (96 MiB), from the number of centroids on where rows are padded."""
    import vq_amd
    n, m, sd, k = 800_003, 3, 10, 64
    rng = np.random.default_rng(4)
    x, cb = rng.random((n, m * sd), dtype=F), rng.random((m, k, sd), dtype=F)
    codes = ctx.empty((n, m), np.uint8)
    ctx.assign(vq_amd.EUCLIDEAN, ctx.to_device(x), n, m * sd, m, sd, k, ctx.to_device(cb), codes)
    at = np.concatenate([np.arange(500), rng.integers(0, n, 3000), np.arange(n - 500, n), 520_000 + np.arange(10_000)])
    assert np.array_equal(codes.download()[at], O.pq_encode(O.EUCLIDEAN, x[at], cb).astype(np.uint8))


@pytest.mark.parametrize("n,m,sd,k", [(65_281, 4, 3, 6), (65_280, 4, 5, 9), (65_281, 8, 7, 17), (65_281, 2, 12, 9), (65_300, 2, 15, 5), (65_281, 4, 4, 2), (44_000, 6, 10, 3)])
def test_encode_with_several_blocks_per_lane(ctx, n, m, sd, k):
    """Two or four blocks per lane: only where that leaves a workgroup per compute unit (65,281 rows x 4 by fours)."""
    import vq_amd
    rng = np.random.default_rng(n + sd)
    x, cb = np.round(rng.standard_normal((n, m * sd)) * 3).astype(F), np.round(rng.standard_normal((m, k, sd)) * 3).astype(F)
    x[n // 3, 1] = np.inf
    dx, dcb = ctx.to_device(x), ctx.to_device(cb)
    for metric, om in ((vq_amd.SQEUCLIDEAN, O.SQEUCLIDEAN), (vq_amd.EUCLIDEAN, O.EUCLIDEAN), (vq_amd.COSINE, O.COSINE), (vq_amd.MANHATTAN, O.MANHATTAN)):
        codes = ctx.to_device(np.full((n, m), 255, np.uint8))
        ctx.assign(metric, dx, n, m * sd, m, sd, k, dcb, codes)
        assert np.array_equal(codes.download(), O.pq_encode(om, x, cb).astype(np.uint8)), metric


@pytest.mark.parametrize("n,m,sd,k", [(300, 3, 24, 256), (7000, 3, 24, 60), (300, 2, 25, 200), (300, 4, 28, 100), (9000, 4, 28, 100), (513, 1, 33, 256), (3000, 16, 33, 90),
                                      (260, 2, 47, 256), (257, 4, 48, 130), (20_000, 3, 48, 40)])
def test_manhattan_by_waves_and_by_lanes(ctx, n, m, sd, k):
    """Blocks of 24 to 48 floats, few and many rows, short and long codebooks: whichever kernel takes them, also chunk by chunk."""
    import vq_amd
    rng = np.random.default_rng(n + sd)
    x, cb = np.round(rng.standard_normal((n, m * sd)) * 2).astype(F), np.round(rng.standard_normal((m, k + 256, sd)) * 2).astype(F)
    dx = ctx.to_device(x)
    codes, wide = ctx.to_device(np.full((n, m), 255, np.uint8)), ctx.to_device(np.full((n, m), 65535, np.uint16))
    ctx.assign(vq_amd.MANHATTAN, dx, n, m * sd, m, sd, k, ctx.to_device(np.ascontiguousarray(cb[:, :k])), codes)
    assert np.array_equal(codes.download(), O.pq_encode(O.MANHATTAN, x, np.ascontiguousarray(cb[:, :k])).astype(np.uint8))
    ctx.assign_u16(vq_amd.MANHATTAN, dx, n, m * sd, m, sd, k + 256, ctx.to_device(cb), wide)
    assert np.array_equal(wide.download(), O.pq_encode(O.MANHATTAN, x, cb).astype(np.uint16))

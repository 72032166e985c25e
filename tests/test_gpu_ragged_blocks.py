"""Column blocks whose width is no multiple of 8, or whose rows are not 16-byte aligned, on the
matrix-core kernels through padded copies: training and encode against the CPU oracle, bit for bit."""
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
    c.set_few_path(1)  # short calls, too, by the kernels named here (test_gpu_few_rows.py has the others)
    yield c
    c.close()


# n, m, sub_dim, k, extra columns of the row buffer
CASES = [(33, 1, 1, 32, 0), (300, 5, 2, 40, 0), (1025, 4, 3, 256, 0), (4097, 8, 4, 64, 3), (129, 4, 7, 33, 1),
         (2000, 3, 9, 200, 0), (6007, 10, 10, 200, 0), (700, 2, 15, 32, 5), (513, 1, 25, 256, 0), (400, 1, 100, 50, 0), (66_001, 5, 8, 33, 0),
         (1500, 2, 16, 96, 1), (260, 1, 300, 256, 0), (70_000, 6, 3, 40, 0)]


@pytest.mark.parametrize("n,m,sd,k,extra", CASES)
def test_fit_and_encode(ctx, n, m, sd, k, extra):
    import vq_amd
    rng = np.random.default_rng(n + sd)
    dim, ld = m * sd, m * sd + extra
    buf = rng.standard_normal((n, ld)).astype(F)
    x = np.ascontiguousarray(buf[:, :dim])
    init, reseed = data.index_streams(n, m, k, 3, seed=n)
    dx, dcb = ctx.to_device(buf), ctx.empty((m, k, sd), F)
    it, _ = ctx.lbg_fit(dx, n, ld, m, sd, k, 3, init, reseed, dcb)
    ref = O.pq_fit(x, m, k, 3, init, reseed)
    assert np.array_equal(dcb.download().view(np.uint32), ref["codebooks"].view(np.uint32))
    codes = ctx.empty((n, m), np.uint8)
    for metric, om in ((vq_amd.SQEUCLIDEAN, O.SQEUCLIDEAN), (vq_amd.EUCLIDEAN, O.EUCLIDEAN)):
        ctx.assign(metric, dx, n, ld, m, sd, k, dcb, codes)
        assert np.array_equal(codes.download(), O.pq_encode(om, x, ref["codebooks"]).astype(np.uint8))


def test_encode_in_slices(ctx):
    """More rows than one padded slice holds (96 MiB)."""
    import vq_amd
    n, m, sd, k = 800_003, 3, 10, 32
    rng = np.random.default_rng(4)
    x, cb = rng.random((n, m * sd), dtype=F), rng.random((m, k, sd), dtype=F)
    codes = ctx.empty((n, m), np.uint8)
    ctx.assign(vq_amd.EUCLIDEAN, ctx.to_device(x), n, m * sd, m, sd, k, ctx.to_device(cb), codes)
    at = np.concatenate([np.arange(500), rng.integers(0, n, 3000), np.arange(n - 500, n), 520_000 + np.arange(10_000)])
    assert np.array_equal(codes.download()[at], O.pq_encode(O.EUCLIDEAN, x[at], cb).astype(np.uint8))

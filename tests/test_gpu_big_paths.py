"""More than 256 centroids chunk by chunk: blocks padded before the chunks, winners' distances from the assignment kernel or
from the merge, whole pieces and remainders of its sums; fits on rows padded once, both means kernels: against the oracle, bit for bit."""
import numpy as np
import pytest

from oracle import oracle as O
from tests import data

pytestmark = pytest.mark.gpu
F = np.float32
METRICS = [O.SQEUCLIDEAN, O.EUCLIDEAN, O.COSINE, O.MANHATTAN]


@pytest.mark.parametrize("metric", METRICS)
@pytest.mark.parametrize("n,m,sd,k,extra", [(700, 3, 10, 1030, 0), (600, 4, 20, 300, 1), (520, 4, 5, 2060, 0), (513, 4, 8, 2305, 0), (600, 1, 47, 258, 0),
                                            (300, 2, 51, 513, 0), (257, 8, 2, 600, 0), (600, 2, 16, 1281, 2)])
def test_encode(metric, n, m, sd, k, extra):
    import vq_amd
    ctx = vq_amd.Context(0)
    ctx.set_few_path(1)
    rng = np.random.default_rng(n + sd + k)
    buf = np.round(rng.standard_normal((n, m * sd + extra)) * 4).astype(F)  # ties inside and between chunks
    cb = np.round(rng.standard_normal((m, k, sd)) * 4).astype(F)
    buf[::9] = rng.standard_normal((len(buf[::9]), m * sd + extra))
    buf[5] = 0.0
    buf[7, 0] = np.nan
    buf[11, -1 - extra] = np.inf
    cb[0, 256, 0] = np.nan  # a chunk whose first distance is no number
    cb[0, 3] = 0.0
    codes = ctx.empty((n, m), np.uint16)
    ctx.assign_u16(metric, ctx.to_device(buf), n, m * sd + extra, m, sd, k, ctx.to_device(cb), codes)
    with np.errstate(all="ignore"):
        want = O.pq_encode(metric, np.ascontiguousarray(buf[:, :m * sd]), cb)
    assert np.array_equal(codes.download(), want.astype(np.uint16))
    ctx.close()


@pytest.mark.parametrize("n,m,sd,k", [(9000, 9, 3, 280), (8959, 3, 9, 280), (12_000, 2, 33, 260), (3000, 17, 10, 1100), (20_000, 1, 2, 300), (40_000, 2, 20, 300)])
def test_fit(n, m, sd, k):
    import vq_amd
    ctx = vq_amd.Context(0)
    x = np.random.default_rng(n + sd).random((n, m * sd), dtype=F)
    x[: n // 4] *= F(0.01)  # clusters of more than 1024 members
    init, reseed = data.index_streams(n, m, k, 2, seed=5)
    cb = ctx.empty((m, k, sd), F)
    ctx.lbg_fit(ctx.to_device(x), n, m * sd, m, sd, k, 2, init, reseed, cb)
    want = O.pq_fit(x, m, k, 2, init, reseed)["codebooks"]
    assert np.array_equal(cb.download().view(np.uint32), want.view(np.uint32))
    ctx.close()


@pytest.mark.parametrize("iters", [1, 3])  # (ends with the last iteration, ends when no code changed)
@pytest.mark.parametrize("sd", [31, 32])
def test_fit_is_done_on_return(sd, iters):
    """The codebooks are in place when the call returns: nothing of it is left on the stream, whether the rows were padded or not."""
    import ctypes
    import vq_amd
    from vq_amd._ffi import lib
    ctx = vq_amd.Context(0)
    hip = ctypes.CDLL("libamdhip64.so")
    n, m, k = 4096, 64, 2048  # 4 MB of codebooks: tens of microseconds for what follows the last update
    rng = np.random.default_rng(sd)
    x = rng.random((n, m * sd), dtype=F) if iters == 1 else np.tile(rng.random((k, m * sd), dtype=F), (n // k, 1))
    init = np.stack([rng.permutation(n)[:k] if iters == 1 else np.arange(k) for _ in range(m)]).astype(np.uint32)
    reseed = rng.integers(0, n, (m, k * iters)).astype(np.uint32)
    ran = np.zeros(m, np.int32)
    dx, cb = ctx.to_device(x), ctx.empty((m, k, sd), F)
    for _ in range(2):
        ctx.sync()
        ctx._check(lib().vq_lbg_fit(ctx._h, dx.ptr, n, m * sd, m, sd, k, iters, init.ctypes.data, reseed.ctypes.data, k * iters, cb.ptr,
                                    ran.ctypes.data, None))
        assert hip.hipStreamQuery(ctypes.c_void_p(lib().vq_ctx_stream(ctx._h))) == 0
        assert ran.max() < 3  # (rows that are their own centroids: the first or second pass changes nothing)
    want = O.pq_fit(np.ascontiguousarray(x[:, :sd]), 1, k, iters, init[:1], reseed[:1])["codebooks"]
    assert np.array_equal(cb.download()[:1].view(np.uint32), want.view(np.uint32))
    ctx.close()


def test_fit_keeps_the_copy_of_other_calls():
    """A fit whose rows need no copy leaves the one that a padded residual encode has made with the context."""
    import ctypes
    import vq_amd
    ctx = vq_amd.Context(0)
    hip = ctypes.CDLL("libamdhip64.so")

    def free_bytes():
        ctx.sync()
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value
    rng = np.random.default_rng(1)
    n, dim, k = 50_000, 300, 300
    dx, dcb = ctx.to_device(rng.random((n, dim), dtype=F)), ctx.to_device(rng.random((2, 64, dim), dtype=F))
    codes = ctx.empty((n, 2), np.uint8)
    init, reseed = data.index_streams(4096, 2, k, 1, seed=5)
    x8, cb8 = ctx.to_device(rng.random((4096, 16), dtype=F)), ctx.empty((2, k, 8), F)
    ctx.lbg_fit(x8, 4096, 16, 2, 8, k, 1, init, reseed, cb8)
    ctx.rvq_encode(O.EUCLIDEAN, dx, n, dim, dim, 2, 64, dcb, 0.0, codes)
    before = free_bytes()
    ctx.lbg_fit(x8, 4096, 16, 2, 8, k, 1, init, reseed, cb8)
    assert abs(free_bytes() - before) < 16 << 20
    ctx.close()

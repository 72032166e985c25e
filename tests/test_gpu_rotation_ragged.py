"""Rotation and cross-covariance of dimensions that are no multiple of the matrix-core tiles: against 64-bit products, with
the bound of a chain of fused multiply-adds, rows spaced and unaligned, and what is not finite in the components behind a row."""
from types import SimpleNamespace

import numpy as np
import pytest

from tests import np_ref

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.mark.parametrize("n,dim,extra,offset", [
    (2, 1, 0, 0), (257, 2, 1, 1), (300, 3, 0, 0), (130, 4, 0, 2), (127, 5, 0, 0), (33, 8, 0, 0), (31, 9, 0, 1), (1, 16, 0, 0), (129, 17, 1, 0), (500, 24, 0, 0), (64, 25, 0, 0), (40, 32, 0, 1), (128, 31, 0, 1), (129, 33, 2, 0), (300, 50, 0, 0), (65, 64, 1, 0), (64, 96, 0, 2), (257, 100, 0, 0), (700, 130, 0, 0),
    (1000, 180, 0, 0), (33, 250, 5, 3), (200, 300, 0, 0), (40, 639, 0, 0)])
def test_rotate(n, dim, extra, offset):
    import vq_amd
    ctx = vq_amd.Context(0)
    rng = np.random.default_rng(dim)
    ld = dim + extra
    buf = np.full(n * ld + offset, np.nan, F)  # what lies between the rows is no number
    x = np.lib.stride_tricks.as_strided(buf[offset:], (n, dim), (4 * ld, 4))
    x[:] = rng.standard_normal((n, dim))
    x[n // 2, dim // 2] = np.inf
    R = rng.standard_normal((dim, dim)).astype(F)
    y = ctx.empty((n, dim), F)
    dx = ctx.to_device(buf)
    ctx.rotate(SimpleNamespace(ptr=dx.ptr + 4 * offset), n, ld, dim, ctx.to_device(R), y)
    got = y.download()
    X, R64 = x.astype(np.float64), R.astype(np.float64)
    rest = np.arange(n) != n // 2
    want, size = X @ R64.T, np.abs(X) @ np.abs(R64).T
    if dim % 32 or extra or offset:
        assert np.array_equal(got[rest].view(np.uint32), np_ref.rotate_chain(x[rest], R).view(np.uint32))
    with np.errstate(invalid="ignore"):
        err = np.abs(got - want)
    assert np.all(err[rest] <= (dim + 1) * 2.0 ** -24 * size[rest])
    assert np.array_equal(got[n // 2], want[n // 2].astype(F))  # infinities, not NaN
    with pytest.raises(Exception):
        ctx.rotate(dx, 1, 700, 640 + 3, ctx.to_device(R), y)
    ctx.close()


@pytest.mark.parametrize("n,dim", [(1, 1), (3, 15), (130, 7), (129, 17), (131, 18), (1, 33), (4, 33), (700, 50), (1025, 100), (514, 130), (2050, 180), (520, 250), (516, 300)])
def test_cross_cov(n, dim):
    import vq_amd
    ctx = vq_amd.Context(0)
    rng = np.random.default_rng(n + dim)
    y, x = rng.standard_normal((n, dim)).astype(F), rng.standard_normal((n, dim)).astype(F)
    got = ctx.cross_cov(ctx.to_device(y), ctx.to_device(x), n, dim)
    Y, X = y.astype(np.float64), x.astype(np.float64)
    assert np.all(np.abs(got - Y.T @ X) <= 2 * n * 2.0 ** -53 * (np.abs(Y).T @ np.abs(X)) + 1e-300)
    ctx.close()


@pytest.mark.parametrize("n,dim", [(700, 3), (40_000, 20), (300, 50), (40_000, 50), (300, 180), (70_000, 130), (5, 250)])
def test_rotate_in_place(n, dim):
    import vq_amd
    ctx = vq_amd.Context(0)
    rng = np.random.default_rng(dim)
    x, R = rng.standard_normal((n, dim)).astype(F), ctx.to_device(rng.standard_normal((dim, dim)).astype(F))
    dx, y = ctx.to_device(x), ctx.empty((n, dim), F)
    ctx.rotate(dx, n, dim, dim, R, y)
    want = y.download()
    ctx.rotate(dx, n, dim, dim, R, dx)
    assert np.array_equal(dx.download().view(np.uint32), want.view(np.uint32))
    ctx.close()


@pytest.mark.parametrize("n,dim,extra", [(70, 1, 0), (70, 5, 0), (70, 16, 3), (40, 23, 0), (70, 31, 0), (40, 32, 1), (70, 33, 0), (100, 50, 0), (33, 100, 0), (40, 250, 2)])
@pytest.mark.parametrize("kind", ["rows", "matrix", "products", "sums", "minus_zero"])
def test_rotate_below_the_smallest_normal_number(n, dim, extra, kind):
    """Rows, matrices, products and partial sums without a normal exponent, and sums that come down to -0: the bits of the
    chain of fused multiply-adds, also behind the last component."""
    import vq_amd
    ctx = vq_amd.Context(0)
    rng = np.random.default_rng(dim)
    x, R = rng.standard_normal((n, dim + extra)), rng.standard_normal((dim, dim))
    if kind == "rows":
        x *= 1e-41
    elif kind == "matrix":
        R *= 1e-41
    elif kind == "products":
        x, R = x * 1e-20, R * 1e-21
    elif kind == "sums":
        x, R = x * np.exp2(rng.integers(-75, -60, x.shape)), R * np.exp2(rng.integers(-75, -60, R.shape))
    else:  # zeros, then one product below the smallest number
        x[:, :dim - 1] = 0.0
        x[:, dim - 1], R[:, dim - 1] = -1e-30, 1e-30
    x, R = x.astype(F), R.astype(F)
    y = ctx.empty((n, dim), F)
    ctx.rotate(ctx.to_device(x), n, dim + extra, dim, ctx.to_device(R), y)
    want = np_ref.rotate_chain(np.ascontiguousarray(x[:, :dim]), R)
    assert kind != "minus_zero" or np.all(np.signbit(want) & (want == 0))
    assert np.array_equal(y.download().view(np.uint32), want.view(np.uint32))
    ctx.close()


@pytest.mark.parametrize("dim,extra", [(2, 1), (20, 3), (50, 2), (64, 1), (64, 4), (160, 32), (180, 1)])
@pytest.mark.parametrize("shift", [0, 4, -52])  # of the output against the rows, in floats (multiples of 16 bytes)
def test_rotate_over_the_rows(dim, extra, shift):
    """An output that lies over rows of other waves, spaced or shifted: as into a buffer of its own."""
    import vq_amd
    ctx = vq_amd.Context(0)
    n, ld = 100_000, dim + (extra if shift >= 0 else 0)
    rng = np.random.default_rng(dim)
    front = max(0, -shift)
    buf = rng.standard_normal(front + n * ld + max(0, shift)).astype(F)
    dx, R, y = ctx.to_device(buf), ctx.to_device(rng.standard_normal((dim, dim)).astype(F)), ctx.empty((n, dim), F)
    rows = SimpleNamespace(ptr=dx.ptr + 4 * front)
    ctx.rotate(rows, n, ld, dim, R, y)
    want = y.download().view(np.uint32).ravel()
    for _ in range(6):
        dx.upload(buf)
        ctx.rotate(rows, n, ld, dim, R, SimpleNamespace(ptr=rows.ptr + 4 * shift))
        got = dx.download()[front + shift:front + shift + n * dim]
        assert np.array_equal(got.view(np.uint32), want)
    ctx.close()


def test_rotate_over_many_rows():
    """More rows than one copy takes: the same rows, in slices where the output begins no later than they do, whole where it begins
    later (the one that exceeds the bound is given back)."""
    import ctypes
    import vq_amd
    ctx = vq_amd.Context(0)
    hip = ctypes.CDLL("libamdhip64.so")

    def free_bytes():
        ctx.sync()
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value
    n, dim, slack = 1_300_000, 500, 1000  # 2.6 GB
    x = np.random.default_rng(1).standard_normal((1300, dim)).astype(F)
    R = ctx.to_device(np.random.default_rng(2).standard_normal((dim, dim)).astype(F))
    y, dx = ctx.empty((1300, dim), F), ctx.empty(n * dim + slack, F)
    ctx.rotate(ctx.to_device(x), 1300, dim, dim, R, y)
    want = y.download().view(np.uint32)
    rows = np.tile(x, (n // 1300, 1)).ravel()
    for at, to in ((0, 0), (slack, 0), (0, slack)):
        host = np.zeros(n * dim + slack, F)
        host[at:at + n * dim] = rows
        dx.upload(host)
        before = free_bytes()
        ctx.rotate(SimpleNamespace(ptr=dx.ptr + 4 * at), n, dim, dim, R, SimpleNamespace(ptr=dx.ptr + 4 * to))
        assert before - free_bytes() < 128 << 20
        got = dx.download()[to:to + n * dim].view(np.uint32).reshape(-1, *want.shape)
        assert np.array_equal(got, np.broadcast_to(want, got.shape))
    ctx.close()

"""What the context keeps after a call: a fit of padded column blocks gives its copy of the rows back, and
the workspace of an assignment above 256 centroids does not grow with the number of rows."""
import ctypes
import time

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu
F = np.float32
MB = 1 << 20


@pytest.fixture
def ctx():
    import vq_amd
    c = vq_amd.Context(0)
    yield c
    c.close()


def _free():
    """Free bytes of the GPU, from the runtime that the library has loaded."""
    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL(path).hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def _held_at_most(before, limit):
    """Memory that was freed comes back a little later: the driver clears up behind the call."""
    for _ in range(40):
        if before - _free() < limit:
            return True
        time.sleep(0.05)
    return False


def test_padded_rows_of_a_fit_are_given_back(ctx):
    n, m, sd, k, iters = 1_200_000, 64, 2, 64, 2  # 2.5 GB of padded copy for 614 MB of rows
    rng = np.random.default_rng(1)
    x = rng.random((n, m * sd), dtype=F)
    init = np.stack([rng.permutation(n)[:k] for _ in range(m)]).astype(np.uint32)
    reseed = rng.integers(0, n, (m, k * iters), dtype=np.uint32)
    dx, out = ctx.to_device(x), []
    for path in (0, 1):  # by the padded copy; by the kernels that take the rows as they are
        cb = ctx.empty((m, k, sd), F)
        ctx.set_assign_path(path)
        before = _free()
        ctx.lbg_fit(dx, n, m * sd, m, sd, k, iters, init, reseed, cb)
        ctx.sync()
        if path == 0:
            # member lists, codes, part sums: 11 bytes per (row, block) pair at most
            assert _held_at_most(before, 11 * n * m + 64 * MB)
        out.append(cb.download())
    assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))


def test_rows_in_slices_above_256_centroids(ctx):
    n, m, sd, k = 280_001, 64, 2, 1300  # 18 million pairs, slices of 16 Mi; six chunks: two merges each
    rng = np.random.default_rng(2)
    x, cb = np.round(rng.standard_normal((n, m * sd)) * 9).astype(F), np.round(rng.standard_normal((m, k, sd)) * 9).astype(F)
    dx, dcb, codes = ctx.to_device(x), ctx.to_device(cb), ctx.empty((n, m), np.uint16)
    before = _free()
    ctx.assign_u16(O.EUCLIDEAN, dx, n, m * sd, m, sd, k, dcb, codes)
    ctx.sync()
    assert _held_at_most(before, 600 * MB)
    got = codes.download()
    at = np.unique(np.concatenate([np.arange(200), rng.integers(0, n, 300), np.arange(262_100, 262_200), np.arange(n - 200, n)]))
    assert np.array_equal(got[at], O.pq_encode(O.EUCLIDEAN, x[at], cb).astype(np.uint16))
    # the rows of both slices on their own
    for lo, hi in ((0, 262_144), (262_144, n)):
        part = ctx.to_device(x[lo:hi])
        ctx.assign_u16(O.EUCLIDEAN, part, hi - lo, m * sd, m, sd, k, dcb, codes)
        assert np.array_equal(got[lo:hi], codes.download()[:hi - lo])

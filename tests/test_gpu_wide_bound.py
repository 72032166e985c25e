"""Wide column blocks on the matrix cores: a score's error bound depends on the centroid, so codebooks whose
norms lie far apart, near-ties among the small ones, and values at the ends of the range are compared with the
CPU oracle code for code."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module")
def ctx():
    import vq_amd
    c = vq_amd.Context(0)
    yield c
    c.close()


def _case(kind, n, m, sd, k):
    rng = np.random.default_rng(sd * 11 + k)
    x, cb = rng.standard_normal((n, m, sd)).astype(F), rng.standard_normal((m, k, sd)).astype(F)
    if kind == "collapsed":  # a few centroids of small norm take most rows, the others are rows
        cb[:, : max(2, k // 4)] *= F(0.02)
    elif kind == "near_ties":
        cb[:, 1::2] = cb[:, 0::2][:, : cb[:, 1::2].shape[1]] * F(1 + 2e-6)
        x[::2] = cb[0, rng.integers(0, k, x[::2].shape[0])][:, None] + F(1e-3) * x[::2]
    elif kind == "grid":  # exact ties, duplicates, zero rows
        x, cb = np.round(x), np.round(cb)
        cb[:, k // 2] = cb[:, 0]
        x[:3] = 0.0
    elif kind == "spread":  # norms of rows and centroids over twelve decades
        x *= (10.0 ** rng.uniform(-6, 6, (n, 1, 1))).astype(F)
        cb *= (10.0 ** rng.uniform(-6, 6, (m, k, 1))).astype(F)
    elif kind == "overflow":  # beside centroids of norm one, rows past the range of binary16 and far below it
        x *= (10.0 ** rng.uniform(-9, 6, (n, 1, 1))).astype(F)
        x[:, :, 1::3] *= F(1e-6)
        cb[:, :, 2::3] *= F(1e-7)
    elif kind == "tiny":
        x, cb = x * F(1e-18), cb * F(1e-18)
        cb[:, 0] *= F(1e15)
    elif kind == "offset":  # far from the origin: the scores are relative to the centre
        x, cb = x * F(0.01) + F(30), cb * F(0.01) + F(30)
    elif kind == "edges":
        x *= (10.0 ** rng.uniform(-18, 18, (n, 1, 1))).astype(F)
        x[3], x[5, 0, 0], x[7, -1, -1] = 0.0, np.nan, np.inf
        cb[-1, k // 2] = 0.0
        cb[0, 1, 0] = np.inf
    return np.ascontiguousarray(x.reshape(n, m * sd)), cb


@pytest.mark.parametrize("kind", ["normal", "collapsed", "near_ties", "grid", "spread", "overflow", "tiny", "offset", "edges"])
@pytest.mark.parametrize("metric", [O.SQEUCLIDEAN, O.EUCLIDEAN])
@pytest.mark.parametrize("n,m,sd,k", [(1300, 3, 16, 256), (700, 2, 24, 33), (900, 1, 64, 200), (300, 2, 104, 256),
                                      (1000, 1, 128, 100), (2049, 1, 256, 256), (130, 1, 264, 31), (333, 1, 264, 61),
                                      (200, 2, 72, 225), (200, 1, 1000, 256)])
def test_wide_codes(ctx, n, m, sd, k, metric, kind):
    x, cb = _case(kind, n, m, sd, k)
    codes = ctx.empty((n, m), np.uint8)
    with np.errstate(all="ignore"):
        ctx.assign(metric, ctx.to_device(x), n, m * sd, m, sd, k, ctx.to_device(cb), codes)
        want = O.pq_encode(metric, x, cb).astype(np.uint8)
    assert np.array_equal(codes.download(), want)

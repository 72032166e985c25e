"""More than 256 centroids: the chunks' winners merged four to a launch.  Numbers of chunks around that, a last
chunk of one centroid, chunks whose first distance is NaN, ties across chunks, against the CPU oracle."""
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


@pytest.mark.parametrize("kind", ["normal", "grid", "nan"])
@pytest.mark.parametrize("metric", [O.SQEUCLIDEAN, O.EUCLIDEAN, O.COSINE, O.MANHATTAN])
@pytest.mark.parametrize("n,m,sd,k", [(700, 2, 8, 1024), (601, 1, 8, 1025), (650, 3, 5, 1281), (520, 1, 64, 2050), (900, 4, 8, 769)])
def test_merge(ctx, n, m, sd, k, metric, kind):
    rng = np.random.default_rng(k + sd)
    x, cb = rng.standard_normal((n, m * sd)).astype(F), rng.standard_normal((m, k, sd)).astype(F)
    if kind == "grid":  # the same centroids in several chunks: the first one wins
        x, cb = np.round(x), np.round(cb)
        cb[:, 256:512] = cb[:, :256]
    elif kind == "nan":
        cb[0, 256, 0] = np.nan
        cb[-1, 512] = np.nan
        x[7, 0] = np.nan
    codes = ctx.empty((n, m), np.uint16)
    with np.errstate(all="ignore"):
        ctx.assign_u16(metric, ctx.to_device(x), n, m * sd, m, sd, k, ctx.to_device(cb), codes)
        want = O.pq_encode(metric, x, cb).astype(np.uint16)
    assert np.array_equal(codes.download(), want)

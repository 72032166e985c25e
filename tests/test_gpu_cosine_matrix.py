"""Cosine encode on the matrix cores (scores against normalised centroids, exact re-check) against the CPU
oracle: every width class, ties, norms at the edges of the range the scores decide, non-finite values."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module")
def ctx():
    import vq_amd
    c = vq_amd.Context(0)
    c.set_few_path(1)  # short calls, too, by the kernels named here (test_gpu_few_rows.py has the others)
    yield c
    c.close()


@pytest.mark.parametrize("kind", ["normal", "unit", "same_direction", "grid", "edges", "scaled"])
@pytest.mark.parametrize("n,m,sd,k", [(2049, 4, 8, 256), (1500, 3, 8, 33), (40_000, 4, 8, 200), (1000, 2, 5, 64), (800, 2, 16, 256),
                                      (700, 1, 40, 100), (600, 1, 100, 256), (1200, 1, 256, 31)])
def test_cosine(ctx, n, m, sd, k, kind):
    import vq_amd
    rng = np.random.default_rng(sd * 7 + k)
    x, cb = rng.standard_normal((n, m * sd)).astype(F), rng.standard_normal((m, k, sd)).astype(F)
    if kind == "unit":
        x /= np.linalg.norm(x, axis=1, keepdims=True)
    elif kind == "same_direction":  # every centroid nearly parallel
        cb = (1.0 + 1e-4 * cb).astype(F)
        x = (2.0 + 1e-3 * x).astype(F)
    elif kind == "grid":  # exact ties, zero vectors
        x, cb = np.round(x), np.round(cb)
        cb[:, -1] = 0.0
    elif kind == "edges":
        x *= (10.0 ** rng.uniform(-22, 22, (n, 1))).astype(F)
        x[3], x[5, 0], x[7, -1] = 0.0, np.nan, np.inf
        cb[0, 0] *= F(1e-17)
        cb[-1, k // 2] = 0.0
    elif kind == "scaled":
        cb *= (10.0 ** rng.uniform(-6, 6, (m, k, 1))).astype(F)
    codes = ctx.empty((n * m + 3,), np.uint8)
    ctx.assign(vq_amd.COSINE, ctx.to_device(x), n, m * sd, m, sd, k, ctx.to_device(cb), codes)
    assert np.array_equal(codes.download()[:n * m].reshape(n, m), O.pq_encode(O.COSINE, x, cb).astype(np.uint8))

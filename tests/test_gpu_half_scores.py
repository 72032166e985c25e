"""Column blocks of 8 and 16 floats: scores from operands rounded to binary16, scaled per column block.  Codebooks and rows
whose norms lie far apart, past the range of binary16 or far below it, near-ties and exact ties are compared with the
CPU oracle code for code, with the tables made by a launch of their own and by the waves themselves, and a fit on
badly scaled rows bit for bit."""
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


@pytest.mark.parametrize("kind", ["collapsed", "near_ties", "grid", "spread", "overflow", "tiny", "offset", "edges", "outlier", "same"])
@pytest.mark.parametrize("metric", [O.SQEUCLIDEAN, O.EUCLIDEAN, O.COSINE])
@pytest.mark.parametrize("n,m,k,sd", [(1300, 4, 256, 8), (900, 3, 33, 8), (70, 8, 255, 8), (330, 1, 2, 8), (210_000, 4, 37, 8),  # tables by a launch
                                      (1300, 3, 256, 16), (900, 2, 33, 16), (70, 40, 65, 16), (330, 1, 2, 16)])
def test_codes(ctx, n, m, k, sd, metric, kind):
    x, cb = _case("normal" if kind in ("outlier", "same") else kind, n, m, sd, k)
    if kind == "outlier":  # one centroid as long as the scale allows for, rows near it and past the range
        cb[:, k // 2] *= F(1e5)
        x[::3, :sd] = cb[0, k // 2] * F(1.0001)
        x[1::3] *= F(3e4)
    elif kind == "same":
        cb[:] = cb[:, :1]
    codes = ctx.empty((n, m), np.uint8)
    ctx.assign(metric, ctx.to_device(x), n, sd * m, m, sd, k, ctx.to_device(cb), codes)
    with np.errstate(all="ignore"):
        assert np.array_equal(codes.download(), O.pq_encode(metric, x, cb).astype(np.uint8))


@pytest.mark.parametrize("kind", ["overflow", "spread", "offset"])
@pytest.mark.parametrize("n,m,k,sd", [(30_000, 4, 24, 8), (3000, 3, 64, 8),  # streamed sums with the next pass's tables; small fit
                                      (30_000, 3, 24, 16), (3000, 2, 64, 16), (5000, 3, 200, 10)])
def test_fit(ctx, n, m, k, sd, kind):
    x, _ = _case(kind, n, m, sd, k)
    init, reseed = data.index_streams(n, m, k, 4, seed=k)
    cb = ctx.empty((m, k, sd), F)
    ctx.lbg_fit(ctx.to_device(x), n, sd * m, m, sd, k, 4, init, reseed, cb)
    want = O.pq_fit(x, m, k, 4, init, reseed)["codebooks"]
    assert np.array_equal(cb.download().view(np.uint32), want.view(np.uint32))

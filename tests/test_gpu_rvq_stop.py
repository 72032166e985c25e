"""RVQ encode with the early stop, update, norm and test of a stage in one kernel: row and column remainders of
its tiles, whole groups of rows that have stopped, both code widths, against the CPU oracle."""
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


@pytest.mark.parametrize("n,dim,ld,stages,k", [(513, 4, 4, 3, 9), (577, 32, 32, 4, 16), (640, 36, 40, 3, 16),
                                               (1000, 100, 100, 3, 31), (703, 132, 136, 2, 300), (2049, 128, 129, 4, 16),
                                               # the tables of all stages in one launch: three parts and one product
                                               (900, 40, 40, 4, 100), (3000, 64, 64, 5, 32), (1200, 256, 256, 3, 256),
                                               # the codebooks of all stages in LDS for the reconstruction: whole groups
                                               # of columns, a last group of 8, all columns in one
                                               (16_400, 128, 128, 4, 256), (8000, 264, 264, 4, 256), (33_001, 64, 64, 8, 64),
                                               # 16 columns in a group, a last group of 8
                                               (16_391, 128, 128, 8, 256), (29_200, 72, 72, 8, 200),
                                               # groups of widths that are no multiple of 32, one of all columns
                                               (10_600, 200, 200, 6, 256), (8100, 264, 264, 8, 256), (29_200, 72, 72, 2, 256),
                                               (15_500, 136, 136, 2, 16),
                                               (16_400, 128, 128, 3, 300)])  # 16-bit codes
def test_rows_stop_one_by_one(ctx, n, dim, ld, stages, k):
    rng = np.random.default_rng(dim + n)
    cb = rng.standard_normal((stages, k, dim)).astype(F)
    cb *= (0.3 ** np.arange(stages)).astype(F)[:, None, None]
    stop = rng.integers(0, stages + 1, n)  # the stage after which a row is within eps
    stop[64:192] = 1                       # two whole groups of rows that stop first
    x = np.zeros((n, dim), F)
    for s in range(stages):
        x += np.where((stop > s)[:, None], cb[s, rng.integers(0, k, n)], F(0))
    x += np.where(stop == 0, 2.0, 1e-4).astype(F)[:, None] * rng.standard_normal((n, dim)).astype(F)
    eps = float(F(0.005 * np.sqrt(dim)))
    wide = np.full((n, ld), np.nan, F)
    wide[:, :dim] = x
    codes = ctx.empty((n, stages), np.uint16 if k > 256 else np.uint8)
    used, rec = ctx.empty((n,), np.uint8), ctx.empty((n, dim), np.uint16)
    (ctx.rvq_encode_u16 if k > 256 else ctx.rvq_encode)(O.EUCLIDEAN, ctx.to_device(wide), n, ld, dim, stages, k,
                                                        ctx.to_device(cb), eps, codes, used, rec)
    wcodes, wrec = O.rvq_quantize(O.EUCLIDEAN, x, cb, eps)
    wused = (wcodes != 0xFFFFFFFF).sum(1)
    assert len(np.unique(wused)) > 1
    assert np.array_equal(used.download(), wused)
    got = codes.download()
    for s in range(stages):
        assert np.array_equal(got[wused > s, s], wcodes[wused > s, s])
        assert not got[wused <= s, s].any()
    assert np.array_equal(rec.download(), wrec)

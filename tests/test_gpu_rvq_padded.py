"""Residual encodes of widths whose rows are copied once with zeros behind them: with and without the early stop, outputs that are
left out, spaced rows, values that are not finite, widths on both sides: against the oracle, bit for bit."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.mark.parametrize("metric", [O.SQEUCLIDEAN, O.EUCLIDEAN, O.COSINE, O.MANHATTAN])
@pytest.mark.parametrize("n,dim,extra,stages,k,eps", [(700, 100, 0, 5, 64, 0.01), (700, 100, 0, 5, 64, 0.0), (1000, 99, 3, 2, 70, 0.5), (600, 300, 0, 3, 256, 0.0),
                                                      (600, 50, 0, 1, 64, 0.0), (800, 20, 1, 4, 61, 1.0), (600, 10, 0, 3, 200, 0.0), (513, 101, 0, 8, 2, 0.01)])
def test_encode(metric, n, dim, extra, stages, k, eps):
    import vq_amd
    ctx = vq_amd.Context(0)
    rng = np.random.default_rng(n + dim)
    buf = rng.standard_normal((n, dim + extra)).astype(F)
    cb = (rng.standard_normal((stages, k, dim)) * 0.7 ** np.arange(stages)[:, None, None]).astype(F)
    buf[::50] *= F(1e-3)
    buf[3] = 0.0
    buf[9, 0] = np.inf
    for r in range(10, n, 7):  # rows that stop after one or two stages
        buf[r, :dim] = cb[:1 + r % 2, r % k].sum(0) + F(1e-5) * rng.standard_normal(dim).astype(F)
    x = np.ascontiguousarray(buf[:, :dim])
    dx, dcb = ctx.to_device(buf), ctx.to_device(cb)
    with np.errstate(all="ignore"):
        want, want_rec = O.rvq_quantize(metric, x, cb, eps)
    reached = want != 0xFFFFFFFF
    assert reached.all() == (eps == 0.0 or stages == 1)
    fine = np.arange(n) != 9  # (sums of infinities of both signs: no number, whatever its bits)
    for with_used, with_rec in ((True, True), (False, True), (False, False)):
        # (what each call has to write is something else before it)
        codes, used = ctx.to_device(~np.where(reached, want, 0).astype(np.uint8)), ctx.to_device(np.full(n, 99, np.uint8))
        rec = ctx.to_device(~np.asarray(want_rec).view(np.uint16))
        ctx.rvq_encode(metric, dx, n, dim + extra, dim, stages, k, dcb, eps, codes, used if with_used else None, rec if with_rec else None)
        assert np.array_equal(codes.download()[fine], np.where(reached, want, 0).astype(np.uint8)[fine])
        if with_used:
            assert np.array_equal(used.download()[fine], reached.sum(1)[fine])
        if with_rec:
            assert np.array_equal(rec.download()[fine], np.asarray(want_rec).view(np.uint16)[fine])
    assert np.array_equal(dx.download(), buf, equal_nan=True)
    ctx.close()

"""A few rows in one launch (k_assign_few, k_rvq_few, k_tsvq_few) and batches of host rows through the
host calls at every way they take (in place, one chunk, pipelined, with copying threads), against the CPU
oracle, bit for bit."""
import numpy as np
import pytest

from oracle import oracle as O
from tests import data
from tests.test_gpu_wide_bound import _case

pytestmark = pytest.mark.gpu
F = np.float32
METRICS = [O.SQEUCLIDEAN, O.EUCLIDEAN, O.COSINE, O.MANHATTAN]


@pytest.fixture(scope="module")
def ctx():
    import vq_amd
    c = vq_amd.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("metric", METRICS)
@pytest.mark.parametrize("n,m,sd,k", [(1, 1, 1, 1), (1, 16, 8, 256), (3, 5, 7, 255), (2, 2, 130, 257), (9, 3, 12, 1000), (512, 1, 8, 40)])
def test_assign_few(ctx, metric, n, m, sd, k):
    rng = np.random.default_rng(n + sd + k)
    x = np.round(rng.standard_normal((n, m * sd)) * 2).astype(F)  # ties
    cb = np.round(rng.standard_normal((m, k, sd)) * 2).astype(F)
    if k > 2:
        cb[:, 1] = 0.0
    if n > 2:
        x[1] = 0.0
        x[2, 0] = np.nan
        cb[-1, 0, 0] = np.inf
    want = O.pq_encode(metric, x, cb)
    codes = ctx.empty((n, m), np.uint16)
    ctx.assign_u16(metric, ctx.to_device(x), n, m * sd, m, sd, k, ctx.to_device(cb), codes)
    assert np.array_equal(codes.download(), want.astype(np.uint16))
    if k <= 256:
        codes8 = ctx.empty((n * m + 3,), np.uint8)
        ctx.assign(metric, ctx.to_device(x), n, m * sd, m, sd, k, ctx.to_device(cb), codes8)
        assert np.array_equal(codes8.download()[:n * m].reshape(n, m), want.astype(np.uint8))


def test_the_widest_block_is_the_same_for_few_rows_and_many(ctx):
    import vq_amd
    rng = np.random.default_rng(3)
    for sd in (1280, 1281):
        x, cb = rng.standard_normal((600, sd)).astype(F), rng.standard_normal((1, 5, sd)).astype(F)
        dx, dcb = ctx.to_device(x), ctx.to_device(cb)
        for n in (1, 512, 600):
            codes, wide, stages = ctx.empty((n,), np.uint8), ctx.empty((n,), np.uint16), ctx.empty((n, 1), np.uint8)
            calls = [lambda: ctx.assign(O.MANHATTAN, dx, n, sd, 1, sd, 5, dcb, codes),
                     lambda: ctx.assign_u16(O.MANHATTAN, dx, n, sd, 1, sd, 5, dcb, wide),
                     lambda: ctx.rvq_encode(O.MANHATTAN, dx, n, sd, sd, 1, 5, dcb, 0.0, stages)]
            for call, out in zip(calls, (codes, wide, stages)):
                if sd == 1280:
                    call()
                    assert np.array_equal(out.download().reshape(n, 1), O.pq_encode(O.MANHATTAN, x[:n], cb))
                else:
                    with pytest.raises(vq_amd.VqError) as e:
                        call()
                    assert e.value.code == vq_amd._ffi.ERR_UNSUPPORTED


@pytest.mark.parametrize("kind", ["collapsed", "near_ties", "grid", "spread", "overflow", "tiny", "offset", "edges"])
@pytest.mark.parametrize("n,m,sd,k", [(130, 1, 264, 31), (64, 2, 33, 60), (60, 8, 8, 256), (500, 1, 128, 100), (24, 2, 16, 500)])
def test_few_path_against_the_kernels_of_longer_calls(ctx, n, m, sd, k, kind):
    """Values at the ends of the range, near ties, non-finite rows and centroids: the one-launch kernels give the
    codes that the kernels of longer calls give, under the four metrics and in a residual encode."""
    x, cb = _case(kind, n, m, sd, k)
    dx, dcb = ctx.to_device(x), ctx.to_device(cb)
    for metric in METRICS:
        got = []
        for path in (0, 1):
            ctx.set_few_path(path)
            try:
                codes = ctx.empty((n, m), np.uint16)
                ctx.assign_u16(metric, dx, n, m * sd, m, sd, k, dcb, codes)
                got.append([codes.download()])
                if m > 1 and k <= 256:  # the column blocks' codebooks as the stages of one block
                    rows = ctx.to_device(np.ascontiguousarray(x[:, :sd]))
                    rcodes, used, rec = ctx.empty((n, m), np.uint8), ctx.empty(n, np.uint8), ctx.empty((n, sd), np.uint16)
                    ctx.rvq_encode(metric, rows, n, sd, sd, m, k, dcb, 0.5, rcodes, used, rec)
                    # (a NaN has many bit patterns)
                    f = rec.download()
                    got[-1] += [rcodes.download(), used.download(), np.where((f & 0x7FFF) > 0x7C00, 0x7E00, f)]
            finally:
                ctx.set_few_path(0)
        assert all(np.array_equal(a, b) for a, b in zip(*got)), (metric, kind)


@pytest.mark.parametrize("metric", METRICS)
@pytest.mark.parametrize("n,dim,stages,k,eps", [(1, 6, 3, 1, 0.0), (5, 33, 4, 20, 3.0), (512, 16, 2, 256, 0.0), (7, 300, 5, 60, 14.0)])
def test_rvq_few(ctx, metric, n, dim, stages, k, eps):
    rng = np.random.default_rng(dim)
    x, cb = rng.standard_normal((n, dim)).astype(F), (0.5 * rng.standard_normal((stages, k, dim))).astype(F)
    codes, rec = ctx.empty((n, stages), np.uint8), ctx.empty((n, dim), np.uint16)
    ctx.rvq_encode(metric, ctx.to_device(x), n, dim, dim, stages, k, ctx.to_device(cb), eps, codes, None, rec)
    want, want_rec = O.rvq_quantize(metric, x, cb, eps)
    assert np.array_equal(codes.download(), want.astype(np.uint8)) and np.array_equal(rec.download(), want_rec)


@pytest.mark.parametrize("metric", METRICS)
@pytest.mark.parametrize("n,dim,depth", [(1, 3, 2), (40, 70, 6), (512, 128, 9), (1, 257, 4), (100, 300, 7), (512, 1031, 5)])
def test_tsvq_few(ctx, metric, n, dim, depth):
    rng = np.random.default_rng(dim + depth)
    x = rng.standard_normal((max(n, 300), dim)).astype(F)
    tree = ctx.tsvq_build(ctx.to_device(x), len(x), dim, dim, depth)
    t = tree.download()
    q = x[:n].copy()
    q[0] = 0.0
    want = O.tsvq_descend(metric, q, t)
    try:
        for path in (0, 1):  # 1, and rows above 256 components: a wave per row
            ctx.set_tsvq_descend_path(path)
            leaf = ctx.to_device(np.full(n, -1, np.int32))
            ctx.tsvq_descend(metric, ctx.to_device(q), n, dim, tree, leaf)
            assert np.array_equal(leaf.download(), want), path
    finally:
        ctx.set_tsvq_descend_path(0)


@pytest.mark.parametrize("metric", METRICS)
@pytest.mark.parametrize("dim,depth", [(7, 3), (16, 4), (16, 6), (24, 8), (36, 3), (72, 3), (100, 9), (130, 1), (200, 1), (200, 4), (256, 3), (257, 2)])
def test_tsvq_few_levels_and_host_rows(ctx, metric, dim, depth):
    """On both sides of the line between a wave and four lanes per row, in GPU memory, and from host rows to f16 rows."""
    from vq_amd import api
    dist = {O.SQEUCLIDEAN: api.Distance.SquaredEuclidean, O.EUCLIDEAN: api.Distance.Euclidean, O.COSINE: api.Distance.CosineDistance,
            O.MANHATTAN: api.Distance.Manhattan}[metric]
    x = np.round(np.random.default_rng(dim).standard_normal((1000, dim)) * 4).astype(F)  # ties
    q = api.TSVQ.new(x, depth, dist)
    t = q.tree()
    want = O.tsvq_descend(metric, x[:512], t)
    rows = t["centroids"][want].astype(np.float16).view(np.uint16)
    tree = ctx.tsvq_build(ctx.to_device(x), len(x), dim, dim, depth)
    dx = ctx.to_device(x)
    for n in (1, 17, 32, 33, 129, 512):
        leaf = ctx.to_device(np.full(n, -1, np.int32))
        ctx.tsvq_descend(metric, dx, n, dim, tree, leaf)
        assert np.array_equal(leaf.download(), want[:n]), n
        assert np.array_equal(q.quantize_batch(x[:n]).view(np.uint16), rows[:n]), n


@pytest.mark.parametrize("metric", METRICS)
@pytest.mark.parametrize("dim,depth", [(32, 8), (128, 9)])
def test_tsvq_rows_on_both_sides_of_the_lines(ctx, metric, dim, depth):
    """Row widths that fit registers: which kernel takes a few rows depends on their number and the tree's size."""
    rng = np.random.default_rng(dim)
    x = np.round(rng.standard_normal((3000, dim)) * 2).astype(F)  # ties
    dx = ctx.to_device(x)
    tree = ctx.tsvq_build(dx, len(x), dim, dim, depth)
    assert (tree.n_nodes <= 511) == (depth == 8)
    want = O.tsvq_descend(metric, x[:513], tree.download())
    for n in (1, 64, 65, 256, 257, 384, 385, 512, 513):
        leaf = ctx.empty(n, np.int32)
        ctx.tsvq_descend(metric, dx, n, dim, tree, leaf)
        assert np.array_equal(leaf.download(), want[:n]), n


@pytest.mark.parametrize("n", [1, 5, 100, 2048, 2049, 8192, 33_001, 140_003])
def test_host_batches(n):
    from vq_amd import api
    rng = np.random.default_rng(n)
    x = rng.random((max(n, 600), 128), dtype=F)
    E = api.Distance.Euclidean
    st = data.index_streams(600, 16, 64, 2, seed=1)
    pq = api.ProductQuantizer.fit(x[:600], 16, 64, 2, E, 0, streams=st)
    cb = pq.codebooks()
    at = np.unique(np.concatenate([np.arange(min(n, 600)), rng.integers(0, n, 1500), np.arange(max(0, n - 600), n)]))
    want = O.pq_encode(O.EUCLIDEAN, x[at], cb).astype(np.uint8)
    assert np.array_equal(pq.encode(x[:n])[at], want)
    assert np.array_equal(pq.quantize_batch(x[:n])[at].view(np.uint16), O.pq_decode_f16(want, cb))
    rv = api.ResidualQuantizer.fit(x[:600], 2, 64, 2, 0.0, E, 0, streams=data.index_streams(600, 2, 64, 2, seed=2))
    codes, rec = O.rvq_quantize(O.EUCLIDEAN, x[at], rv.codebooks(), 0.0)
    assert np.array_equal(rv.encode(x[:n])[at], codes.astype(np.uint8))
    assert np.array_equal(rv.quantize_batch(x[:n])[at].view(np.uint16), rec)
    ts = api.TSVQ.new(x[:600], 5, E)
    t = ts.tree()
    leaves = ts.leaves(x[:n])
    assert np.array_equal(leaves[at], O.tsvq_descend(O.EUCLIDEAN, x[at], dict(t, n_nodes=len(t["left"]))))
    assert np.array_equal(ts.quantize_batch(x[:n])[at].view(np.uint16), O.f32_to_f16_bits(t["centroids"][leaves[at]]).reshape(len(at), 128))

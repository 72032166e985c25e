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
    c.set_few_path(1)  # short calls, too, by the kernels named here (test_gpu_few_rows.py has the others)
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


@pytest.mark.parametrize("n,m,sd,k,kind", [(131_075, 1, 256, 256, "collapsed"), (140_001, 1, 304, 256, "grid"),
                                           (65_540, 2, 104, 200, "near_ties"), (14_600, 9, 72, 256, "edges"),
                                           (140_000, 1, 264, 33, "spread"), (45_000, 3, 64, 256, "overflow")])
def test_resident_codes(ctx, n, m, sd, k, kind):
    """Large calls: the operands resident in LDS, several tiles per wave; also a fit's pass (codes in planes,
    compared through the centroids)."""
    x, cb = _case(kind, n, m, sd, k)
    codes = ctx.empty((n, m), np.uint8)
    dx, dcb = ctx.to_device(x), ctx.to_device(cb)
    with np.errstate(all="ignore"):
        ctx.assign(O.EUCLIDEAN, dx, n, m * sd, m, sd, k, dcb, codes)
        got = codes.download()
        pick = np.unique(np.concatenate([np.arange(300), np.random.default_rng(1).integers(0, n, 3000), np.arange(n - 300, n)]))
        assert np.array_equal(got[pick], O.pq_encode(O.EUCLIDEAN, x[pick], cb).astype(np.uint8))
        # every row against the all-vector kernels
        ctx.set_assign_path(1)
        try:
            ctx.assign(O.EUCLIDEAN, dx, n, m * sd, m, sd, k, dcb, codes)
        finally:
            ctx.set_assign_path(0)
        assert np.array_equal(got, codes.download())


def test_resident_fit(ctx):
    n, m, sd, k, iters = 70_003, 2, 64, 256, 3
    rng = np.random.default_rng(5)
    x = rng.standard_normal((n, m * sd)).astype(F)
    init = np.stack([rng.permutation(n)[:k] for _ in range(m)]).astype(np.uint32)
    reseed = rng.integers(0, n, (m, k * iters), dtype=np.uint32)
    dx, out = ctx.to_device(x), []
    for path in (0, 1):
        cb = ctx.empty((m, k, sd), np.float32)
        ctx.set_assign_path(path)
        try:
            ctx.lbg_fit(dx, n, m * sd, m, sd, k, iters, init, reseed, cb)
        finally:
            ctx.set_assign_path(0)
        out.append(cb.download())
    assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))


@pytest.mark.parametrize("kind", ["crowded", "clumps", "nan0", "nan7"])
@pytest.mark.parametrize("metric", [O.SQEUCLIDEAN, O.EUCLIDEAN])
@pytest.mark.parametrize("n,m,sd,k", [(131_075, 1, 128, 256), (44_000, 3, 72, 250), (140_000, 1, 256, 70)])
def test_rows_with_many_candidates(ctx, n, m, sd, k, metric, kind):
    """What the resident pass leaves open to three and more centroids: clumps of 2 to 90 neighbours (more than one batch
    of candidates, ties among them), a codebook that leaves every row open (more entries than have masks), NaN."""
    rng = np.random.default_rng(sd + k)
    x, cb = rng.standard_normal((n, m, sd)).astype(F), rng.standard_normal((m, k, sd)).astype(F)
    if kind == "crowded":
        cb = (cb[:, :1] + F(1e-6) * cb).astype(F)
    else:
        at = 0
        for size in (2, 3, 5, 20, 90):
            end = min(k, at + size)
            cb[:, at:end] = cb[:, at:at + 1] + F(1e-6) * cb[:, at:end]
            cb[:, end - 1] = cb[:, at]  # the last of a clump equal to its first
            at = end
        cb = cb[:, rng.permutation(k)].copy()
        x[::2] = cb[np.arange(m)[None, :], rng.integers(0, k, (x[::2].shape[0], 1))] + F(0.3) * x[::2]
        if kind == "nan0":
            cb[:, 0, 3] = np.nan
        elif kind == "nan7":
            cb[:, 7, 3] = np.nan
    x = np.ascontiguousarray(x.reshape(n, m * sd))
    dx, dcb, codes = ctx.to_device(x), ctx.to_device(cb), ctx.empty((n, m), np.uint8)
    ctx.assign(metric, dx, n, m * sd, m, sd, k, dcb, codes)
    got = codes.download()
    assert ctx.last_recheck_split()[0] > 0
    pick = np.concatenate([np.arange(1500), np.arange(n - 1500, n)])
    with np.errstate(all="ignore"):
        assert np.array_equal(got[pick], O.pq_encode(metric, x[pick], cb).astype(np.uint8))
    ctx.set_assign_path(1)
    try:
        ctx.assign(metric, dx, n, m * sd, m, sd, k, dcb, codes)
    finally:
        ctx.set_assign_path(0)
    assert np.array_equal(got, codes.download())


@pytest.mark.parametrize("n,m,sd,k", [(600, 26, 32, 2), (4000, 26, 104, 2), (4000, 26, 100, 2), (5100, 26, 64, 256)])
def test_blocks_whose_only_change_is_an_undecided_pair(ctx, n, m, sd, k):
    """The same rows in every column block: in the second pass one row changes its cluster, by a margin of 2e-5 that only the
    check of two candidates decides, in all blocks at once.  No block has converged before the third pass."""
    far = k - 2
    h, nb = (n - far) // 2, n - far - (n - far) // 2
    v = np.zeros(n)
    v[1:h], v[h:n - far - 1] = 0.02, 1.0
    # the row is nearer to the second cluster's first centre, and 2.5e-6 below the middle of the two means
    v[n - far - 1] = ((v[:h].mean() + (nb - 1) / nb) / 2 - 2.5e-6) / (1 - 0.5 / nb)
    x = np.zeros((n, m, sd), F)
    x[:, :, 0] = v.astype(F)[:, None]
    for j in range(far):  # clusters of one row each
        x[n - far + j, :, 1 + j % (sd - 1)] = (4.0 + j // (2 * (sd - 1))) * (-1) ** (j // (sd - 1))
    x = x.reshape(n, m * sd)
    init = np.tile(np.concatenate([[0, h], np.arange(n - far, n)]).astype(np.uint32), (m, 1))
    reseed = np.zeros((m, 6 * k), np.uint32)
    dcb = ctx.empty((m, k, sd), F)
    iters, used = ctx.lbg_fit(ctx.to_device(x), n, m * sd, m, sd, k, 6, init, reseed, dcb)
    want = O.pq_fit(x, m, k, 6, init, reseed)
    assert np.all(want["iters"] == 3)
    assert np.array_equal(iters, want["iters"]) and np.array_equal(used, want["reseeds"])
    assert np.array_equal(dcb.download().view(np.uint32), want["codebooks"].view(np.uint32))


# rounds of 16,384 rows (64 compute units per column block): tiles of the last one dealt to all workgroups below half a round, and a
# workgroup's eight side by side beyond; one tile more than whole rounds, one row more than a tile
@pytest.mark.parametrize("n", [32_768, 32_769, 33_000, 40_928, 40_960, 40_961, 49_151])
def test_last_round_of_tiles(n):
    import vq_amd
    ctx = vq_amd.Context(0)
    rng = np.random.default_rng(n)
    x, cb = rng.random((n, 256), dtype=np.float32), rng.random((4, 256, 64), dtype=np.float32)
    codes = ctx.empty((n, 4), np.uint8)
    ctx.assign(O.EUCLIDEAN, ctx.to_device(x), n, 256, 4, 64, 256, ctx.to_device(cb), codes)
    assert np.array_equal(codes.download(), O.pq_encode(O.EUCLIDEAN, x, cb).astype(np.uint8))
    ctx.close()

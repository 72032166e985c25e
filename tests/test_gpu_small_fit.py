"""The one-launch update of small LBG fits (two launches per iteration) against the CPU oracle, bit for
bit: centroids, iterations run, re-seed rows used."""
import numpy as np
import pytest

from oracle import oracle as O
from tests import data

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module")
def ctx():
    import vq_amd
    c = vq_amd.Context(0)
    yield c
    c.close()


# n, m, sub_dim, k, iterations, kind
CASES = [(16, 4, 8, 16, 3, "normal"),          # one row per cluster
         (8191, 4, 8, 256, 3, "normal"), (8193, 4, 8, 250, 3, "normal"),  # a step of codes, and one row more
         (70_001, 4, 8, 256, 2, "skewed"),     # clusters above 1024 members in several parts, the list worked off twice
         (30_000, 1, 8, 100, 3, "skewed"), (20_000, 3, 4, 64, 3, "skewed"),
         (9000, 2, 12, 40, 4, "same"),         # one cluster, every other one re-seeded
         (2000, 5, 8, 7, 30, "blobs"),         # early stop
         (3000, 2, 32, 20, 3, "normal"), (5000, 1, 36, 64, 3, "normal"), (4097, 1, 100, 33, 3, "normal"),
         (12_000, 1, 256, 256, 2, "skewed"), (20_001, 2, 40, 64, 3, "skewed"), (10_000, 1, 48, 16, 3, "same"), (6000, 2, 64, 32, 3, "skewed"), (300, 1, 1000, 5, 2, "normal"),
         # blocks of their own width up to 39 centroids, padded from 40 on
         (431, 15, 4, 32, 4, "normal"), (900, 3, 4, 39, 3, "normal"), (900, 3, 4, 40, 3, "normal"), (2000, 3, 12, 39, 3, "blobs"), (2000, 3, 12, 40, 3, "blobs"),
         (2000, 5, 20, 39, 3, "normal"), (2000, 5, 20, 40, 3, "normal"), (3000, 2, 28, 39, 3, "skewed"), (3000, 2, 28, 40, 3, "skewed")]


@pytest.mark.parametrize("n,m,sd,k,iters,kind", CASES)
def test_small_fit(ctx, n, m, sd, k, iters, kind):
    rng = np.random.default_rng(n + sd)
    dim = m * sd
    x = rng.standard_normal((n, dim)).astype(F)
    if kind == "skewed":
        x[rng.random(n) < 0.7] = x[0]  # most rows in one cluster
    elif kind == "same":
        x[:] = x[0]
    elif kind == "blobs":
        x = (10.0 * rng.integers(0, k, (n, 1)) + 0.01 * x).astype(F)
    init, reseed = data.index_streams(n, m, k, iters, seed=n)
    dcb = ctx.empty((m, k, sd), F)
    it, used = ctx.lbg_fit(ctx.to_device(x), n, dim, m, sd, k, iters, init, reseed, dcb)
    ref = O.pq_fit(x, m, k, iters, init, reseed)
    assert np.array_equal(dcb.download().view(np.uint32), ref["codebooks"].view(np.uint32))
    assert np.array_equal(it, ref["iters"]) and np.array_equal(used, ref["reseeds"])


@pytest.mark.parametrize("sd,m,largest", [(8, 32, 3000), (8, 32, 9000), (16, 16, 5000), (16, 16, 9000), (4, 64, 3000),
                                          (12, 16, 5000), (32, 12, 1025), (1028, 2, 1030)])
def test_small_fit_cluster_sizes(ctx, sd, m, largest):
    """Clusters of every size around the batches of eight members, of 1024 and 1025 (the order of summation
    changes) and above 8192 rows in one workgroup's list (its sizes are not known when the sums begin), several
    in a workgroup (m * k > 256) and at different places of it (a block's clusters are one further on)."""
    rng = np.random.default_rng(sd + largest)
    k = 64 if sd < 1024 else 140
    sizes = [1, 2, 7, 8, 9, 15, 16, 17, 23, 24, 25, 31, 32, 33, 39, 40, 41, 1023, 1024, 1025, largest]
    sizes += [200 if sd < 1024 else 90] * (k - len(sizes))
    label = rng.permutation(np.repeat(np.arange(k), sizes))
    n = len(label)
    x = (50.0 * label[:, None] + rng.random((n, m * sd))).astype(F)
    first = np.array([int(np.flatnonzero(label == j)[0]) for j in range(k)])
    init = np.stack([first[(np.arange(k) + s) % k] for s in range(m)]).astype(np.uint32)
    reseed = np.zeros((m, k), np.uint32)
    want = O.pq_fit(x, m, k, 2, init, reseed)
    dcb = ctx.empty((m, k, sd), F)
    it, used = ctx.lbg_fit(ctx.to_device(x), n, m * sd, m, sd, k, 2, init, reseed, dcb)
    assert want["rc"] == 0 and np.array_equal(it, want["iters"]) and np.array_equal(used, want["reseeds"])
    assert np.array_equal(dcb.download().view(np.uint32), want["codebooks"].view(np.uint32))


@pytest.mark.parametrize("n,m,sd,k", [(12_000, 1, 36, 64), (12_289, 2, 36, 200), (12_000, 1, 100, 64), (12_288, 1, 300, 256), (10_000, 1, 512, 256),
                                      (8192, 1, 48, 30), (8193, 2, 52, 60), (12_000, 20, 48, 100), (32_768, 1, 40, 200), (32_769, 1, 40, 200),
                                      # several blocks: the line rises with the number of clusters
                                      (36_000, 3, 36, 100), (36_001, 3, 36, 100), (39_872, 4, 64, 256), (39_873, 4, 64, 256), (50_041, 2, 48, 256), (32_769, 2, 100, 200)])
def test_small_fit_tiles(ctx, n, m, sd, k):
    """Blocks above 32 floats by tiles whose last one overlaps (or whole, where there are many): clusters on both sides
    of the size from which each part's members are added by tiles too, and one that is re-seeded."""
    rng = np.random.default_rng(n + sd)
    line = 1024 * -(-n // 4096)
    sizes = [line + 1, line, 1025] if 2 * line + 1100 + k < n else [line + 1, 1024]
    rest = n - sum(sizes)
    sizes += [rest // (k - len(sizes))] * (k - len(sizes) - 1)
    sizes.append(n - sum(sizes))
    label = rng.permutation(np.repeat(np.arange(k), sizes))
    x = (50.0 * label[:, None] + rng.random((n, m * sd))).astype(F)
    first = np.array([int(np.flatnonzero(label == j)[0]) for j in range(k)])
    first[k // 2] = first[k // 2 + 1]
    init = np.stack([first[(np.arange(k) + s) % k] for s in range(m)]).astype(np.uint32)
    reseed = rng.integers(0, n, (m, 2 * k), dtype=np.uint32)
    want = O.pq_fit(x, m, k, 2, init, reseed)
    dcb = ctx.empty((m, k, sd), F)
    it, used = ctx.lbg_fit(ctx.to_device(x), n, m * sd, m, sd, k, 2, init, reseed, dcb)
    assert want["rc"] == 0 and np.array_equal(it, want["iters"]) and np.array_equal(used, want["reseeds"]) and used.min() > 0
    assert np.array_equal(dcb.download().view(np.uint32), want["codebooks"].view(np.uint32))


@pytest.mark.parametrize("n,m,sd,k", [(12_288, 1, 36, 64), (12_288, 2, 52, 60), (16_000, 3, 100, 40), (9000, 1, 512, 30)])
def test_small_fit_three_large_clusters(ctx, n, m, sd, k):
    """Three clusters of every block that are taken by tiles, side by side, and of several blocks more than there are turns."""
    rng = np.random.default_rng(n + m)
    line = 1024 * -(-n // 4096)
    sizes = [line + 1, line + 2, line + 1] if 3 * line + 4 + k < n else [line + 1, line + 2]
    rest = n - sum(sizes)
    sizes += [rest // (k - len(sizes))] * (k - len(sizes) - 1)
    sizes.append(n - sum(sizes))
    label = rng.permutation(np.repeat(np.arange(k), sizes))
    x = (50.0 * label[:, None] + rng.random((n, m * sd))).astype(F)
    first = np.array([int(np.flatnonzero(label == j)[0]) for j in range(k)])
    init = np.stack([first[(np.arange(k) + 7 * s) % k] for s in range(m)]).astype(np.uint32)
    reseed = rng.integers(0, n, (m, 2 * k), dtype=np.uint32)
    want = O.pq_fit(x, m, k, 2, init, reseed)
    dcb = ctx.empty((m, k, sd), F)
    it, used = ctx.lbg_fit(ctx.to_device(x), n, m * sd, m, sd, k, 2, init, reseed, dcb)
    assert want["rc"] == 0 and np.array_equal(it, want["iters"]) and np.array_equal(used, want["reseeds"])
    assert np.array_equal(dcb.download().view(np.uint32), want["codebooks"].view(np.uint32))


# both sides of the lines of one block that is the whole row, of a first fit and of a residual stage
@pytest.mark.parametrize("residual,n,sd,k", [
    (False, 54_000, 40, 200), (False, 54_001, 40, 200), (False, 58_000, 24, 100), (False, 58_001, 24, 100), (False, 20_480, 128, 64), (False, 20_481, 128, 64),
    (True, 40_480, 32, 64), (True, 40_481, 32, 64), (True, 33_760, 64, 64), (True, 33_761, 64, 64), (True, 30_000, 128, 100), (True, 30_001, 128, 100),
    (True, 16_071, 224, 128), (True, 16_072, 224, 128), (True, 104_001, 16, 170), (True, 30_001, 100, 100)])
def test_fit_of_one_block_at_its_lines(ctx, residual, n, sd, k):
    rng = np.random.default_rng(n + sd)
    x = (rng.random((n, sd)) + 3 * rng.integers(0, 4, (n, 1))).astype(F)
    init = rng.choice(n, k, replace=False).astype(np.uint32)[None]
    reseed = rng.integers(0, n, (1, 2 * k), dtype=np.uint32)
    dx, dcb = ctx.to_device(x), ctx.empty((1, k, sd), F)
    if residual:
        pcb, pcodes = rng.random((9, sd)).astype(F), rng.integers(0, 9, n, dtype=np.uint8)
        it, used = ctx.lbg_fit_residual(dx, n, sd, sd, k, 2, init[0], reseed[0], dcb, ctx.to_device(pcb), 9, ctx.to_device(pcodes))
        x = x - pcb[pcodes]
    else:
        it, used = ctx.lbg_fit(dx, n, sd, 1, sd, k, 2, init, reseed, dcb)
    want = O.pq_fit(x, 1, k, 2, init, reseed)
    assert want["rc"] == 0 and np.all(it == want["iters"]) and np.all(used == want["reseeds"])
    assert np.array_equal(dcb.download().view(np.uint32), want["codebooks"].view(np.uint32))

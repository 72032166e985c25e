"""Reconstruction from codes: the table in LDS whole or by groups of column blocks, and the gather through the
vector cache, at sizes that end inside a run of rows, a workgroup's pieces or a group; exact against numpy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module")
def ctx():
    import vq_amd
    c = vq_amd.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("n,m,sd,k", [
    (1, 1, 8, 2), (1025, 3, 8, 40), (70_001, 1, 8, 256), (5463, 12, 16, 256), (70_000, 1, 512, 20),  # whole table / gather
    (110_001, 10, 8, 1024), (66_000, 17, 8, 2048), (33_001, 33, 24, 300), (263_000, 4, 16, 3000),   # groups, the last short
    (130_000, 9, 16, 5000), (4097, 2, 64, 700), (999, 5, 12, 300),                                  # a block too large: gather
    (87_401, 12, 8, 1024), (53_003, 20, 8, 2048), (262_145, 4, 8, 256), (52_429, 10, 8, 300),  # table in LDS: binary16
    (21_001, 25, 8, 200), (10_699, 49, 8, 11),
    (87_401, 12, 4, 1024), (53_003, 20, 4, 2048), (33_000, 17, 4, 256), (175_001, 3, 4, 2000),  # table in LDS: f32
    # 60 million components and more: also centroids of several pieces, f16 and f32
    (470_001, 8, 16, 256), (157_003, 12, 32, 256), (500_009, 5, 24, 40)])
def test_decode(ctx, n, m, sd, k):
    rng = np.random.default_rng(n + k)
    cb = (rng.standard_normal((m, k, sd)) * 100).astype(F)
    codes = rng.integers(0, k, (n, m), dtype=np.uint16)
    want = cb[np.arange(m)[None, :], codes].reshape(n, m * sd)
    wide = k > 256
    dcodes, dcb = ctx.to_device(codes.astype(np.uint16 if wide else np.uint8)), ctx.to_device(cb)
    out = ctx.to_device(np.full((n + 1, m * sd), 0x5555, np.uint16))
    (ctx.decode_f16_u16 if wide else ctx.decode_f16)(dcodes, n, m, sd, k, dcb, out)
    got = out.download()
    assert np.array_equal(got[:n], want.astype(np.float16).view(np.uint16)) and (got[n] == 0x5555).all()
    out32 = ctx.to_device(np.full((n + 1, m * sd), 7.0, F))
    (ctx.decode_f32_u16 if wide else ctx.decode_f32)(dcodes, n, m, sd, k, dcb, out32)
    got = out32.download()
    assert np.array_equal(got[:n], want) and (got[n] == 7.0).all()


@pytest.mark.parametrize("off", [2, 16, 32, 64])
def test_output_off_alignment(ctx, off):
    """An output that starts anywhere in a line: the table in LDS only where lines are filled."""
    rng = np.random.default_rng(off)
    n, m, k = 35_537, 16, 200
    cb, codes = rng.standard_normal((m, k, 8)).astype(F), rng.integers(0, k, (n, m))
    out = ctx.to_device(np.full(n * m * 8 + 64, 0x5555, np.uint16))

    class Part:
        ptr = out.ptr + off
    ctx.decode_f16(ctx.to_device(codes.astype(np.uint8)), n, m, 8, k, ctx.to_device(cb), Part())
    got = out.download()
    want = cb[np.arange(m)[None, :], codes].reshape(-1).astype(np.float16).view(np.uint16)
    assert np.array_equal(got[off // 2:off // 2 + len(want)], want)
    assert (got[:off // 2] == 0x5555).all() and (got[off // 2 + len(want):] == 0x5555).all()


@pytest.mark.parametrize("dim", [8, 24, 128, 12, 7])
def test_tree_decode(ctx, dim):
    rng = np.random.default_rng(dim)
    x = rng.standard_normal((3000, dim)).astype(F)
    tree = ctx.tsvq_build(ctx.to_device(x), 3000, dim, dim, 5)
    cen = tree.download()["centroids"]
    leaf = rng.integers(0, len(cen), 2047).astype(np.int32)
    out = ctx.to_device(np.full((2048, dim), 0x5555, np.uint16))
    ctx.tsvq_decode_f16(tree, ctx.to_device(leaf), 2047, out)
    got = out.download()
    assert np.array_equal(got[:2047], cen[leaf].astype(np.float16).view(np.uint16)) and (got[2047] == 0x5555).all()


@pytest.mark.parametrize("off", [0, 2, 8])
@pytest.mark.parametrize("n,m,sd,k", [
    # read from memory: units of one, two and four components, ends inside a thread's and a workgroup's share
    (1, 1, 1, 1), (1023, 3, 7, 40), (1500, 2, 6, 300), (2049, 5, 12, 300), (90_001, 3, 5, 2000), (300_001, 3, 2, 30_000),
    # the table in LDS: two codes per eight components or more, narrow blocks, whole and short last pieces, 160 KB
    (2_600_003, 1, 1, 256), (650_001, 2, 2, 256), (280_001, 3, 3, 200), (200_003, 7, 4, 256), (180_001, 3, 5, 300), (160_001, 3, 6, 256),
    (120_007, 3, 7, 256), (46_003, 11, 5, 1024), (70_001, 4, 9, 2000), (60_001, 7, 12, 256), (9_001, 7, 45, 30), (66_001, 8, 10, 1024)])
def test_decode_any_width(ctx, n, m, sd, k, off):
    rng = np.random.default_rng(n + sd)
    cb = (rng.standard_normal((m, k, sd)) * 100).astype(F)
    codes = rng.integers(0, k, (n, m), dtype=np.uint16)
    want = cb[np.arange(m)[None, :], codes].reshape(-1).astype(np.float16).view(np.uint16)
    out = ctx.to_device(np.full(n * m * sd + 16, 0x5555, np.uint16))

    class Part:
        ptr = out.ptr + off
    if k > 256:
        ctx.decode_f16_u16(ctx.to_device(codes), n, m, sd, k, ctx.to_device(cb), Part())
    else:
        ctx.decode_f16(ctx.to_device(codes.astype(np.uint8)), n, m, sd, k, ctx.to_device(cb), Part())
    got = out.download()
    assert np.array_equal(got[off // 2:off // 2 + len(want)], want)
    assert (got[:off // 2] == 0x5555).all() and (got[off // 2 + len(want):] == 0x5555).all()


def test_tree_decode_from_a_table(ctx):
    """More leaves than a tree's table in LDS needs to pay, widths of every unit."""
    rng = np.random.default_rng(5)
    x = rng.standard_normal((4000, 50)).astype(F)
    for dim, n in ((50, 60_001), (44, 120_001), (25, 110_003)):
        tree = ctx.tsvq_build(ctx.to_device(np.ascontiguousarray(x[:, :dim])), 4000, dim, dim, 4)
        cen = tree.download()["centroids"]
        leaf = rng.integers(0, len(cen), n).astype(np.int32)
        out = ctx.to_device(np.full((n + 1, dim), 0x5555, np.uint16))
        ctx.tsvq_decode_f16(tree, ctx.to_device(leaf), n, out)
        got = out.download()
        assert np.array_equal(got[:n], cen[leaf].astype(np.float16).view(np.uint16)) and (got[n] == 0x5555).all()

"""TSVQ levels whose nodes each fit one workgroup: sums, variances, median and partition of a node in LDS.  Node
sizes around the tiles (128 rows of a leaf sum, the workgroups' 256 and 1024 rows, the longest node that is taken
that way), widths around 32 components and 64 lanes, ties, signed zeros and infinities, against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.test_gpu_tsvq import assert_same_tree, bfs_order

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module")
def ctx():
    import vq_amd
    c = vq_amd.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("n,dim,depth,kind", [
    (2, 4, 1, "normal"), (3, 65, 2, "normal"), (127, 33, 3, "grid"), (129, 31, 7, "normal"), (257, 64, 4, "zeros"),
    (1023, 128, 5, "normal"), (1025, 12, 9, "grid"), (2049, 200, 3, "normal"), (4096, 32, 2, "normal"),
    (4097, 36, 2, "ties"), (8193, 16, 2, "normal"), (16384, 8, 2, "ties"), (16385, 8, 3, "normal"), (33000, 5, 4, "grid"),
    (1500, 1100, 3, "normal"), (3000, 24, 6, "inf"),
])
def test_small_nodes(ctx, n, dim, depth, kind):
    rng = np.random.default_rng(n + dim)
    x = rng.standard_normal((n, dim)).astype(F)
    if kind == "grid":
        x = np.round(x * 2).astype(F)
    elif kind == "ties":  # two values in the widest column: the median is one of them
        x[:, dim - 1] = np.where(rng.random(n) < 0.6, F(-40), F(40))
    elif kind == "zeros":
        x = np.where(rng.random((n, dim)) < 0.7, np.where(rng.random((n, dim)) < 0.5, F(0.0), F(-0.0)), x).astype(F)
    elif kind == "inf":
        x[::501, 3] = F(1e30)
        x[1::503, 7] = F(-1e30)
    got = ctx.tsvq_build(ctx.to_device(x), n, dim, dim, depth).download()
    want, _ = bfs_order(O.tsvq_fit(x, depth))
    assert_same_tree(got, want)

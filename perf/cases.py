"""Performance cases of the library: what its users call, over the sizes they call it with.

Two kinds of program use the library.  One holds its vectors in host arrays and calls the classes of
`vq_amd.api` (ops "fit" and "quantize": the call takes host arrays and returns host arrays, and the
whole of it counts).  The other keeps its rows in GPU memory and drives the C ABI through
`vq_amd.Context` (the other ops: torch tensors hold the rows and receive the results).

  fit            train a quantizer of vq_amd.api on host rows, read its codebooks (and rotation) or its tree
  quantize       one vector, or a batch of host rows, to its f16 reconstruction
  pq_train       LBG on every column block of resident rows, then the encode of the rows
  pq_encode      resident rows to codes and codes to f16 rows, any metric, k also above 256
  rvq_train      residual training, stage by stage, on resident rows
  rvq_encode     resident rows through every stage: codes and f16 sums
  tsvq_build     the tree from resident rows
  tsvq_quantize  resident rows down a tree: leaf numbers and f16 rows

Every result follows the operation order that the library documents and its tests compare bit for
bit, so the tolerance is "exact" except where a matrix product of free order is in the path (the
rotation of the optimized product quantizer).
"""
import math

import numpy as np
import torch

import vq_amd
from vq_amd import api

METRICS = {"sqeuclidean": (vq_amd.SQEUCLIDEAN, api.Distance.SquaredEuclidean),
           "euclidean": (vq_amd.EUCLIDEAN, api.Distance.Euclidean),
           "cosine": (vq_amd.COSINE, api.Distance.CosineDistance),
           "manhattan": (vq_amd.MANHATTAN, api.Distance.Manhattan)}


def listed():
    return [
        # a service that compresses one vector as it arrives: latency only
        dict(name="quantize_one", op="quantize", quantizer="pq", n=1, dim=128, m=16, k=256, metric="euclidean"),
        # the evaluation protocol's timed quantize-all, host rows in and host f16 rows out
        dict(name="quantize_batch_50k", op="quantize", quantizer="pq", n=50_000, dim=128, m=16, k=256, metric="euclidean"),
        # the evaluation protocol's training at its ordinary size
        dict(name="fit_pq_10k", op="fit", quantizer="pq", n=10_000, dim=128, m=16, k=256, iters=10, metric="euclidean"),
        # the same protocol for the optimized product quantizer: five rotations with a training each
        dict(name="fit_opq_50k", op="fit", quantizer="opq", n=50_000, dim=128, m=16, k=256, iters=10, outer=5,
             metric="euclidean"),
        # the headline configuration: a million rows kept on the GPU, trained on and encoded
        dict(name="pq_train_1m", op="pq_train", n=1_000_000, dim=128, m=16, k=256, iters=10, metric="euclidean"),
        # word vectors of 100 components: column blocks of 10, an odd number of rows, fewer centroids than a byte holds
        dict(name="pq_train_ragged", op="pq_train", n=60_007, dim=100, m=10, k=200, iters=10, metric="euclidean"),
        # normalised embeddings encoded under the cosine distance
        dict(name="pq_encode_cosine", op="pq_encode", n=200_000, dim=96, m=12, k=256, metric="cosine"),
        # finer codebooks than a byte addresses: 16-bit codes
        dict(name="pq_encode_k1024", op="pq_encode", n=300_000, dim=128, m=16, k=1024, metric="euclidean"),
        # the residual quantizer's training at its full size: the largest case
        dict(name="rvq_train_1m", op="rvq_train", n=1_000_000, dim=256, stages=8, k=256, iters=10, metric="euclidean"),
        # encode with the evaluation protocol's early stop
        dict(name="rvq_encode_eps", op="rvq_encode", n=200_000, dim=128, stages=4, k=256, epsilon=0.01, metric="euclidean"),
        # the evaluation protocol's tree: ten levels, so most nodes are small
        dict(name="tsvq_build_100k", op="tsvq_build", n=100_000, dim=128, depth=10),
        # a large set of unit vectors down a tree of eight levels
        dict(name="tsvq_quantize_1m", op="tsvq_quantize", n=1_000_000, dim=128, depth=8, metric="cosine"),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over the logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _blocks(rng, most):
    """(m, sub_dim) as they occur: four to ten components per code mostly, two to 48 at the ends."""
    while True:
        sd = rng.choice([2, 3, 4, 5, 6, 7, 8, 8, 8, 9, 10, 12, 15, 16, 16, 20, 24, 25, 32, 48])
        m = rng.randint(1, 64)
        if 16 <= m * sd <= most:
            return m, sd


def draw(rng):
    op = rng.choice(["quantize", "quantize", "fit", "fit", "pq_train", "pq_train", "pq_encode", "pq_encode",
                     "rvq_train", "rvq_encode", "tsvq_build", "tsvq_quantize"])
    metric = rng.choice(["euclidean", "euclidean", "sqeuclidean", "cosine", "manhattan"])
    if op in ("quantize", "fit"):
        kind = rng.choice(["pq", "pq", "opq", "rvq", "tsvq"])
        m, sd = _blocks(rng, 256)
        c = dict(op=op, quantizer=kind, n=_log(rng, 1 if op == "quantize" else 1000, 100_000), dim=m * sd, metric=metric)
        if kind == "tsvq":
            return dict(c, depth=rng.randint(3, 10))
        c["k"] = _log(rng, 16, 256)
        if kind == "rvq":
            c.update(stages=rng.randint(2, 6), epsilon=rng.choice([0.0, 0.01]))
        else:
            c["m"] = m
        if op == "fit":
            c["iters"] = rng.randint(5, 15)
            if kind == "opq":
                c["outer"] = rng.randint(1, 5)
        return c
    if op in ("pq_train", "pq_encode"):
        m, sd = _blocks(rng, 512)
        c = dict(op=op, dim=m * sd, m=m, metric=metric)
        c["k"] = _log(rng, 16, 256) if rng.random() < 0.75 else _log(rng, 257, 2048)
        c["n"] = _log(rng, 4000, min(1_000_000, 128_000_000 // c["dim"], 128_000_000 * 256 // (c["dim"] * c["k"])))
        if op == "pq_train":
            c["iters"] = rng.randint(3, 12)
        return c
    if op in ("rvq_train", "rvq_encode"):
        dim = rng.choice([32, 64, 96, 100, 128, 200, 256, 300])
        c = dict(op=op, n=_log(rng, 4000, min(1_000_000, 128_000_000 // dim)), dim=dim, stages=rng.randint(2, 8), k=_log(rng, 16, 256),
                 metric=rng.choice(["euclidean", "sqeuclidean"]))
        c.update(dict(iters=rng.randint(4, 10)) if op == "rvq_train" else dict(epsilon=rng.choice([0.0, 0.01])))
        return c
    dim = rng.choice([16, 24, 50, 64, 96, 100, 128, 128, 200, 256])
    c = dict(op=op, n=_log(rng, 2000, min(1_000_000, 128_000_000 // dim)), dim=dim, depth=rng.randint(3, 10))
    if op == "tsvq_quantize":
        c["metric"] = metric
    return c


# ---- inputs ----------------------------------------------------------------------------------------
_kept = {}


def _context():
    """The one context that a program keeps."""
    if "ctx" not in _kept:
        _kept["ctx"] = vq_amd.Context(0)
    return _kept["ctx"]


class _Dev:
    """A torch tensor where the binding takes a device array."""

    def __init__(self, shape, dtype):
        self.t = torch.empty(shape, dtype=dtype, device="cuda")
        self.ptr = self.t.data_ptr()


def _rows(n, dim, seed, unit=False, centers=1024, sigma=0.05):
    """A mixture of Gaussians (unit: scaled to length one), on the GPU."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    c = torch.randn((centers, dim), generator=g, device="cuda") if unit else torch.rand((centers, dim), generator=g, device="cuda")
    x = _Dev((n, dim), torch.float32)
    torch.randn((n, dim), generator=g, device="cuda", out=x.t)
    x.t.mul_(0.5 if unit else sigma)
    x.t.add_(c[torch.randint(0, centers, (n,), generator=g, device="cuda")])
    if unit:
        x.t.div_(x.t.norm(dim=1, keepdim=True))
    return x


def _streams(n, problems, k, iters, seed):
    """k distinct first rows and k * iters re-seed rows for each problem."""
    rng = np.random.default_rng([seed, 77])
    init = np.empty((problems, k), np.uint32)
    for p in range(problems):
        got = rng.permutation(n)[:k] if n < 8 * k else np.empty(0, np.int64)
        while got.size < k:
            got = rng.permutation(np.unique(np.concatenate([got, rng.integers(0, n, 2 * k)])))[:k]
        init[p] = got
    return init, rng.integers(0, n, (problems, max(1, k * iters)), dtype=np.uint32)


def _train(ctx, x, n, dim, m, k, seed, iters=4):
    """Codebooks of the rows' own clusters, for the encode cases."""
    rows = min(n, max(20_000, 4 * k))
    if rows < k:
        raise ValueError("fewer rows than centroids")
    cb = _Dev((m, k, dim // m), torch.float32)
    init, reseed = _streams(rows, m, k, iters, seed)
    ctx.lbg_fit(x.ptr, rows, dim, m, dim // m, k, iters, init, reseed, cb.ptr)
    return cb


def _host_fit(c, x, iters, seed):
    dist = METRICS[c["metric"]][1]
    if c["quantizer"] == "pq":
        return api.ProductQuantizer.fit(x, c["m"], c["k"], iters, dist, seed)
    if c["quantizer"] == "opq":
        return api.OptimizedProductQuantizer.fit(x, c["m"], c["k"], iters, c.get("outer", 1), dist, seed)
    if c["quantizer"] == "rvq":
        return api.ResidualQuantizer.fit(x, c["stages"], c["k"], iters, c["epsilon"], dist, seed)
    return api.TSVQ.new(x, c["depth"], dist)


def prepare(case, seed):
    c, op, n, dim = dict(case), case["op"], case["n"], case["dim"]
    s = dict(case=c, op=op)
    if op in ("fit", "quantize"):  # host programs: numpy arrays, uniform rows as in the evaluation protocol
        rng = np.random.default_rng(seed)
        s["x"] = rng.random((n, dim), dtype=np.float32)
        if op == "quantize":
            s["q"] = _host_fit(c, rng.random((4000, dim), dtype=np.float32), 3, seed)
        else:
            s["seed"] = seed
        return s
    ctx = s["ctx"] = _context()
    s["metric"] = METRICS[c["metric"]][0] if "metric" in c else None
    unit = op in ("tsvq_build", "tsvq_quantize") or c.get("metric") == "cosine"
    x = s["x"] = _rows(n, dim, seed, unit)
    if op in ("pq_train", "pq_encode"):
        s["codes"] = _Dev((n, c["m"]), torch.uint8 if c["k"] <= 256 else torch.int16)
        if op == "pq_train":
            s["streams"] = _streams(n, c["m"], c["k"], c["iters"], seed)
            s["cb"] = _Dev((c["m"], c["k"], dim // c["m"]), torch.float32)
        else:
            s["cb"] = _train(ctx, x, n, dim, c["m"], c["k"], seed)
            s["out"] = _Dev((n, dim), torch.float16)
    elif op == "rvq_train":
        s["streams"] = _streams(n, c["stages"], c["k"], c["iters"], seed)
        s["res"], s["codes"] = _Dev((n, dim), torch.float32), _Dev((n,), torch.uint8)
        s["cb"] = _Dev((c["stages"], c["k"], dim), torch.float32)
    elif op == "rvq_encode":
        s["cb"] = _Dev((c["stages"], c["k"], dim), torch.float32)
        rows = min(n, 20_000)
        res, codes = _Dev((rows, dim), torch.float32), _Dev((rows,), torch.uint8)
        _rvq_train(ctx, vq_amd.EUCLIDEAN, x, res, codes, s["cb"], rows, dim, c["stages"], c["k"], 3,
                   _streams(rows, c["stages"], c["k"], 3, seed))
        ctx.sync()
        s["codes"], s["used"] = _Dev((n, c["stages"]), torch.uint8), _Dev((n,), torch.uint8)
        s["out"] = _Dev((n, dim), torch.float16)
    elif op == "tsvq_quantize":
        s["tree"] = ctx.tsvq_build(x, min(n, 50_000), dim, dim, c["depth"])
        s["leaf"], s["out"] = _Dev((n,), torch.int32), _Dev((n, dim), torch.float16)
    return s


# ---- passes ----------------------------------------------------------------------------------------
def _rvq_train(ctx, metric, x, res, codes, cb, n, dim, stages, k, iters, streams):
    """The stage loop of a residual quantizer without an early stop: the residual update of a stage
    goes along with the training of the next, and nothing looks at the last stage's residual."""
    init, reseed = streams
    ctx.copy_f32(res, x, n * dim)
    for st in range(stages):
        p = cb.ptr + st * k * dim * 4
        if st == 0:
            ctx.lbg_fit(res.ptr, n, dim, 1, dim, k, iters, init[st], reseed[st], p)
        else:
            ctx.lbg_fit_residual(res.ptr, n, dim, dim, k, iters, init[st], reseed[st], p, p - k * dim * 4, k, codes.ptr)
        if st + 1 < stages:
            ctx.assign(metric, res.ptr, n, dim, 1, dim, k, p, codes.ptr)


def run(state):
    s, c = state, state["case"]
    op, n, dim = c["op"], c["n"], c["dim"]
    if op == "quantize":
        return s["q"].quantize(s["x"][0]) if n == 1 else s["q"].quantize_batch(s["x"])
    if op == "fit":
        q = _host_fit(c, s["x"], c.get("iters", 0), s["seed"])
        if c["quantizer"] == "tsvq":
            return q.tree()
        return (q.codebooks(), q.rotation()) if c["quantizer"] == "opq" else q.codebooks()
    ctx, x = s["ctx"], s["x"]
    if op == "pq_train":
        m, k, sd = c["m"], c["k"], dim // c["m"]
        done = ctx.lbg_fit(x.ptr, n, dim, m, sd, k, c["iters"], *s["streams"], s["cb"].ptr)
        (ctx.assign if k <= 256 else ctx.assign_u16)(s["metric"], x.ptr, n, dim, m, sd, k, s["cb"].ptr, s["codes"].ptr)
        return s["cb"].t, s["codes"].t, done
    if op == "pq_encode":
        m, k, sd = c["m"], c["k"], dim // c["m"]
        (ctx.assign if k <= 256 else ctx.assign_u16)(s["metric"], x.ptr, n, dim, m, sd, k, s["cb"].ptr, s["codes"].ptr)
        (ctx.decode_f16 if k <= 256 else ctx.decode_f16_u16)(s["codes"], n, m, sd, k, s["cb"], s["out"])
        return s["codes"].t, s["out"].t
    if op == "rvq_train":
        _rvq_train(ctx, s["metric"], x, s["res"], s["codes"], s["cb"], n, dim, c["stages"], c["k"], c["iters"], s["streams"])
        return s["cb"].t, s["res"].t, s["codes"].t
    if op == "rvq_encode":
        ctx.rvq_encode(s["metric"], x, n, dim, dim, c["stages"], c["k"], s["cb"], c["epsilon"], s["codes"], s["used"], s["out"])
        return s["codes"].t, s["used"].t, s["out"].t
    if op == "tsvq_build":
        t = ctx.tsvq_build(x, n, dim, dim, c["depth"])
        return t.download()
    ctx.tsvq_descend(s["metric"], x, n, dim, s["tree"], s["leaf"])
    ctx.tsvq_decode_f16(s["tree"], s["leaf"], n, s["out"])
    return s["leaf"].t, s["out"].t


# ---- what a pass cannot do without -----------------------------------------------------------------
def work(case):
    c = case
    op, n, dim = c["op"], c["n"], c["dim"]
    k, m, stages, depth = c.get("k", 0), c.get("m", 1), c.get("stages", 1), c.get("depth", 0)
    kind = c.get("quantizer") or op.split("_")[0]
    width = 2 if k > 256 else 1
    rows = 4.0 * n * dim
    score = 2.0 * n * dim * k  # one distance per row and centroid, a multiply and an add per component
    books = 4.0 * k * dim * (stages if kind == "rvq" else 1)
    tree = 4.0 * min(2 ** (depth + 1), 2 * n) * dim
    if op == "quantize":
        flops = {"pq": score, "opq": score + 2.0 * n * dim * dim, "rvq": stages * score, "tsvq": 2.0 * n * dim * depth}[kind]
        return {"bytes": rows + rows / 2 + (tree if kind == "tsvq" else books), "flops": flops}
    if op == "fit":
        it = c.get("iters", 0)
        flops = {"pq": it * score, "opq": c.get("outer", 1) * ((it + 1) * score + 4.0 * n * dim * dim),
                 "rvq": stages * (it + 1) * score, "tsvq": 4.0 * n * dim * depth}[kind]
        return {"bytes": rows + (tree if kind == "tsvq" else books), "flops": flops}
    if op == "pq_train":
        return {"bytes": rows + books + n * m * width, "flops": (c["iters"] + 1) * score}
    if op == "pq_encode":
        return {"bytes": rows + books + n * m * width + rows / 2, "flops": score}
    if op == "rvq_train":
        return {"bytes": 2 * rows + books + n, "flops": stages * (c["iters"] + 1) * score}
    if op == "rvq_encode":
        return {"bytes": rows + books + n * (stages + 1) + rows / 2, "flops": stages * score}
    if op == "tsvq_build":
        return {"bytes": rows + tree, "flops": 4.0 * n * dim * depth}
    return {"bytes": rows + tree + 4.0 * n + rows / 2, "flops": 2.0 * n * dim * depth}


def tolerance(case):
    if case.get("quantizer") == "opq":
        return {"rel": 1e-5, "max": 1e-3}  # the rotated rows are a matrix product in f32
    return "exact"

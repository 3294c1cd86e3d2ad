"""The measured workloads of the tropical GEMM: what its users run, over the range they run it.

``listed()`` names fixed cases, ``draw(rng)`` gives one more of the same ranges.  Sizes come from
workloads.py, __graft_entry__.smoke() and the tests, or are generic.  Inputs live on the GPU and are
made from the seed alone.
"""
from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "tropical-gemm_amd"))

from tropical_gemm import einsum as tg_einsum  # noqa: E402
from tropical_gemm import ops, pytorch as tg_torch  # noqa: E402

_TORCH = {"f32": torch.float32, "f64": torch.float64, "i32": torch.int32, "i64": torch.int64}
_SIZE = {"f32": 4, "f64": 8, "i32": 4, "i64": 8}
_DEV = "cuda"
_EINSUM = "jik,lkj,lm->im"


def _gemm(name, semiring, dtype, m, n, k, argmax=True, data="normal"):
    return dict(name=name, op="gemm", semiring=semiring, dtype=dtype, batch=0, m=m, n=n, k=k,
                argmax=argmax, data=data)


def _train(name, semiring, dtype, batch, m, n, k):
    return dict(name=name, op="train", semiring=semiring, dtype=dtype, batch=batch, m=m, n=n, k=k,
                argmax=True, data="unit" if semiring == "maxmul" else "normal")


def _einsum_case(name, i, j, k, l, m):  # noqa: E741
    return dict(name=name, op="einsum", semiring="maxplus", dtype="f32", i=i, j=j, k=k, l=l, m=m,
                data="normal")


def listed():
    return [
        # One small product with its argmax, no size a multiple of anything: the latency of a call
        # (the size smoke() checks).
        _gemm("small_67x45x131", "maxplus", "f32", 67, 45, 131),
        # One decoding step of a few sequences against a dense 4096-state transition matrix.
        _gemm("decode_4x4096x4096", "maxplus", "f32", 4, 4096, 4096),
        # An ordinary product with argmax that fills the GPU for a few tens of microseconds (C1).
        _gemm("square_1024", "maxplus", "f32", 1024, 1024, 1024),
        # All-pairs shortest paths: one distance product with predecessors on a graph whose vertex
        # count is no round number; a tenth of the edges missing (C2's data).
        _gemm("apsp_2001", "minplus", "f32", 2001, 2001, 2001, data="distance"),
        # A large value-only product (C3).
        _gemm("maxmul_8192x4096x2048", "maxmul", "f32", 8192, 4096, 2048, argmax=False, data="unit"),
        # Viterbi over many sequences: integer scores, 128 states (C4).
        _gemm("viterbi_262144x128x128", "maxplus", "i32", 262144, 128, 128, data="scores"),
        # A short inner dimension, bound by its outputs (M1).
        _gemm("shortk_65536x2048x8", "maxplus", "f32", 65536, 2048, 8),
        # Double precision with argmax at an ordinary size.
        _gemm("f64_1024", "maxplus", "f64", 1024, 1024, 1024),
        # 64-bit integer scores with argmax (I1's data).
        _gemm("i64_2048", "maxplus", "i64", 2048, 2048, 2048, data="wide"),
        # A training step of a batched tropical layer (heads of an attention-like block), through
        # autograd: forward, grad_A and grad_B.
        _train("train_batched_64x128", "maxplus", "f32", 64, 128, 128, 128),
        # A training step of one large tropical layer (P's forward and C5's backward).
        _train("train_4096", "maxplus", "f32", 0, 4096, 4096, 4096),
        # A tensor network contracted by the einsum: two products after two permutations (E1).
        _einsum_case("einsum_2048", 2048, 32, 64, 2048, 2048),
    ]


# Cost of a product of each type next to an f32 one, for the bound on drawn cases.
_WEIGHT = {"f32": 1.0, "i32": 1.3, "f64": 2.5, "i64": 4.5}
_MAX_COST = 4096.0 ** 3
_MAX_BYTES = 1.2e9


def _log(rng, lo, hi):
    """A size spread over its logarithm: half of them any whole number, the rest multiples of 4,
    16 or 64 (where that stays in range)."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    q = rng.choice([1, 1, 1, 4, 16, 64])
    v = max(lo, min(hi, v))
    return v if v < 2 * q else max(lo, v // q * q)


def draw(rng):
    while True:
        c = _draw(rng)
        w = work(c)
        if w["flops"] / 2 * _WEIGHT[c["dtype"]] <= _MAX_COST and w["bytes"] <= _MAX_BYTES:
            c.pop("name", None)
            return c


def _draw(rng):
    kind = rng.choice(["gemm", "gemm", "gemm", "decode", "apsp", "viterbi", "shortk", "batched",
                       "train", "train_batched", "einsum"])
    sr = rng.choice(["maxplus", "minplus", "maxmul"])
    if kind == "einsum":
        return _einsum_case("", _log(rng, 64, 2048), _log(rng, 4, 32), _log(rng, 4, 64),
                            _log(rng, 64, 2048), _log(rng, 64, 2048))
    if kind == "apsp":
        v = _log(rng, 100, 4096)
        return _gemm("", "minplus", "f32", v, v, v, data="distance")
    if kind == "viterbi":
        s = _log(rng, 16, 256)
        return _gemm("", "maxplus", "i32", _log(rng, 1024, 262144), s, s, data="scores")
    if kind == "decode":
        s = _log(rng, 128, 4096)
        return _gemm("", rng.choice(["maxplus", "minplus"]), rng.choice(["f32", "f32", "i32"]),
                     _log(rng, 1, 16), s, s, data="any")
    if kind == "shortk":
        return _gemm("", sr, rng.choice(["f32", "f32", "f64", "i32"]), _log(rng, 1024, 65536),
                     _log(rng, 64, 2048), _log(rng, 1, 32), argmax=rng.random() < 0.5, data="any")
    if kind in ("train", "train_batched"):
        hi = 4096 if kind == "train" else 256
        batch = 0 if kind == "train" else _log(rng, 2, 256)
        return _train("", sr, rng.choice(["f32", "f32", "f64"]), batch, _log(rng, 16, hi),
                      _log(rng, 16, hi), _log(rng, 16, hi))
    dt = rng.choice(["f32", "f32", "f32", "f64", "i32", "i64"])
    if kind == "batched":
        c = _gemm("", sr, dt, _log(rng, 16, 256), _log(rng, 16, 256), _log(rng, 16, 256),
                  argmax=rng.random() < 0.5, data="any")
        c["batch"] = _log(rng, 2, 256)
        return c
    return _gemm("", sr, dt, _log(rng, 16, 8192), _log(rng, 16, 8192), _log(rng, 16, 4096),
                 argmax=rng.random() < 0.5, data="any")


def _shapes(c):
    if c["op"] == "einsum":
        return [(c["j"], c["i"], c["k"]), (c["l"], c["k"], c["j"]), (c["l"], c["m"])]
    lead = (c["batch"],) if c["batch"] else ()
    return [lead + (c["m"], c["k"]), lead + (c["k"], c["n"])]


def _values(shape, dtype, data, side, semiring, g):
    t = _TORCH[dtype]
    if data == "any":
        data = ("scores" if dtype in ("i32", "i64") else "unit" if semiring == "maxmul" else "normal")
    if data == "normal":
        return torch.randn(shape, generator=g, device=_DEV, dtype=t)
    if data == "unit":  # (0, 1]
        return 1 - torch.rand(shape, generator=g, device=_DEV, dtype=t)
    if data == "distance":  # [0, 100), a tenth +inf, a zero diagonal
        d = torch.rand(shape, generator=g, device=_DEV, dtype=t) * 99.0
        d[torch.rand(shape, generator=g, device=_DEV) < 0.1] = float("inf")
        d.fill_diagonal_(0.0)
        return d
    lim = {"scores": 1000 if side == 0 else 50, "wide": 10 ** 9}[data]
    hi = 1 if data == "scores" and side == 1 else lim + 1
    return torch.randint(-lim, hi, shape, generator=g, device=_DEV, dtype=t)


def _inputs(c, seed):
    g = torch.Generator(device=_DEV)
    g.manual_seed(seed)
    xs = [_values(s, c["dtype"], c["data"], min(q, 1), c["semiring"], g).contiguous()
          for q, s in enumerate(_shapes(c))]
    if c["op"] == "train":
        shape = xs[0].shape[:-1] + (c["n"],)
        xs.append(torch.randn(shape, generator=g, device=_DEV, dtype=_TORCH[c["dtype"]]))
    return xs


def prepare(case, seed):
    xs = _inputs(case, seed)
    if case["op"] == "train":
        xs[0].requires_grad_(True)
        xs[1].requires_grad_(True)
    return dict(case=case, x=xs)


_LAYER = {
    ("maxplus", False): tg_torch.tropical_maxplus_matmul_gpu,
    ("minplus", False): tg_torch.tropical_minplus_matmul_gpu,
    ("maxmul", False): tg_torch.tropical_maxmul_matmul_gpu,
    ("maxplus", True): tg_torch.tropical_maxplus_matmul_batched,
    ("minplus", True): tg_torch.tropical_minplus_matmul_batched,
    ("maxmul", True): tg_torch.tropical_maxmul_matmul_batched,
}


def run(state):
    c, x = state["case"], state["x"]
    if c["op"] == "einsum":
        return tg_einsum.einsum(_EINSUM, *x, semiring=c["semiring"])
    if c["op"] == "train":
        y = _LAYER[c["semiring"], c["batch"] > 0](x[0], x[1])
        ga, gb = torch.autograd.grad(y, (x[0], x[1]), x[2])
        return y.detach(), ga, gb
    f = ops.gemm_batched if c["batch"] else ops.gemm
    y, idx = f(c["semiring"], x[0], x[1], c["argmax"])
    return (y, idx) if c["argmax"] else y


def work(case):
    c = case
    if c["op"] == "einsum":
        jk = c["j"] * c["k"]
        # jik,lkj -> il, then il,lm -> im; or lkj,lm -> jkm first: the smaller of the two orders.
        flops = 2 * min(c["i"] * jk * c["l"] + c["i"] * c["l"] * c["m"],
                        jk * c["l"] * c["m"] + c["i"] * jk * c["m"])
        return dict(bytes=4 * (c["i"] * jk + c["l"] * jk + c["l"] * c["m"] + c["i"] * c["m"]),
                    flops=flops)
    b, s = max(c["batch"], 1), _SIZE[c["dtype"]]
    m, n, k = c["m"], c["n"], c["k"]
    if c["op"] == "train":
        # A, B and the output's gradient in; the output and both gradients out.
        return dict(bytes=b * s * 2 * (m * k + k * n + m * n), flops=b * (2 * m * n * k + 2 * m * n))
    return dict(bytes=b * (s * (m * k + k * n + m * n) + (4 * m * n if c["argmax"] else 0)),
                flops=2 * b * m * n * k)


def tolerance(case):
    """Every value is one product that the inputs hold and every argmax the first that attains it;
    gradients are sums in a documented order: all of them the same bits on every implementation."""
    return "exact"


def _product(semiring, x, y):
    return x * y if semiring == "maxmul" else x + y


def _select(semiring, a, b, dtype):
    """The optimum over k of a (x) b in `dtype` and the first k attaining it, one k at a time."""
    better = torch.lt if semiring == "minplus" else torch.gt
    a, b = a.to(dtype), b.to(dtype)
    shape = a.shape[:-1] + b.shape[-1:]
    best = _product(semiring, a[..., :, :1], b[..., :1, :]).expand(shape).clone()
    idx = torch.zeros(shape, dtype=torch.int32, device=a.device)
    for k in range(1, a.shape[-1]):
        p = _product(semiring, a[..., :, k:k + 1], b[..., k:k + 1, :])
        take = better(p, best)
        idx.masked_fill_(take, k)
        best = torch.where(take, p, best)
    return best, idx


def _optimum(semiring, a, b):
    join = torch.minimum if semiring == "minplus" else torch.maximum
    dtype = torch.float64 if a.is_floating_point() else torch.int64
    a, b = a.to(dtype), b.to(dtype)
    best = _product(semiring, a[..., :, :1], b[..., :1, :]).expand(a.shape[:-1] + b.shape[-1:]).clone()
    for k in range(1, a.shape[-1]):
        best = join(best, _product(semiring, a[..., :, k:k + 1], b[..., k:k + 1, :]))
    return best


def exact(case, seed):
    c = case
    x = _inputs(c, seed)
    sr = c["semiring"]
    if c["op"] == "einsum":
        j, i, k = x[0].shape
        left = x[0].permute(1, 0, 2).reshape(i, j * k)
        right = x[1].permute(2, 1, 0).reshape(j * k, c["l"])
        return _optimum(sr, _optimum(sr, left, right), x[2].double())
    if c["op"] == "gemm":
        y = _optimum(sr, x[0], x[1])
        return (y, None) if c["argmax"] else y
    # Gradients follow the winners of the inputs' own precision.
    _, idx = _select(sr, x[0], x[1], x[0].dtype)
    idx = idx.long()
    a, b, g = (t.double() for t in x)
    win_a, win_b = a.gather(-1, idx), b.gather(-2, idx)  # A[i, k*], B[k*, j]
    ga = torch.zeros_like(a).scatter_add_(-1, idx, g * win_b if sr == "maxmul" else g)
    gb = torch.zeros_like(b).scatter_add_(-2, idx, g * win_a if sr == "maxmul" else g)
    return _product(sr, win_a, win_b), ga, gb

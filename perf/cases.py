"""What this framework is timed on: krn tile programs as a user writes and launches them, on one MI355X.

A program that serves a model prepares its launches once (`launcher.bind` on the tensors it keeps) and replays them, so
`prepare` makes inputs, outputs and the bound launch, and `run` is one replay; `lib.matmul` is called directly, as its
users call it. Tensors are torch memory handed to the runtime without a copy.

Families (`"op"`):
  gemm       C = A @ B^T, the weight layout of a linear layer: bf16, f16, fp8 (per-tensor scales), int8 (W8A8, per-row and
             per-column scales), 16-bit output. Few rows are decoding, thousands are prefill or a batch.
  matmul     `lib.matmul` on krn's own kernel: A @ B with B stored K x N and a fused epilogue, any sizes.
  attention  the flash-attention tile program: prefill (causal or not, ragged lengths) and decode (one or a few queries
             against a long cache), head dimension 64 and 128.
  softmax    the long-row softmax program: attention scores, router logits, a vocabulary.
  matmul_f32 the f32 tile matmul, whose products run in float32.
  attention_d32  flash attention with a head dimension that has no kernel of its own: what any other tile program with
             products, masks and reductions gets.
"""

import math
import os
from typing import TypeVar

import torch

# a process has one HIP runtime: torch brings its own, so the framework is pointed at that one before it loads any
os.environ["ROCM_PATH"] = os.path.dirname(torch.__file__)

from krn_amd import Blocks, Const, Matrix, T, Tensor, arange, block, kernel, maximum, pipelined, struct, where, zeros
from krn_amd.dtypes import BF16, F8E4M3, F16, F32, I8
from krn_amd.lib import lib
from krn_amd.runtime.api import device_of
from krn_amd.runtime.hip import HIPTensor

F = TypeVar("F")


@struct
class Tiling:
    bm: Const[int] = 256
    bn: Const[int] = 256
    bk: Const[int] = 64


@kernel
def linear(t: Tiling, a: Matrix[F], b: Matrix[F], c: Matrix[F]) -> None:
    rows, cols = block.tile(t.bm, t.bn)
    acc = zeros(T.f32, t.bm, t.bn)
    for ks in pipelined(a.shape[1], t.bk):
        acc += a[rows, ks] @ b[cols, ks].transpose()
    c[rows, cols] = acc.to(c.dtype)


@kernel
def linear_fp8(
    t: Tiling, a: Matrix[T.f8e4m3fn], b: Matrix[T.f8e4m3fn], c: Matrix[T.bf16], scale_a: T.f32, scale_b: T.f32
) -> None:
    rows, cols = block.tile(t.bm, t.bn)
    acc = zeros(T.f32, t.bm, t.bn)
    for ks in pipelined(a.shape[1], t.bk):
        acc += a[rows, ks] @ b[cols, ks].transpose()
    c[rows, cols] = (acc * (scale_a * scale_b)).to(T.bf16)


@kernel
def linear_w8a8(
    t: Tiling, a: Matrix[T.i8], w: Matrix[T.i8], scale_a: Matrix[T.f32], scale_w: Matrix[T.f32], c: Matrix[T.bf16]
) -> None:
    rows, cols = block.tile(t.bm, t.bn)
    acc = zeros(T.i32, t.bm, t.bn)
    for ks in pipelined(a.shape[1], t.bk):
        acc += a[rows, ks] @ w[cols, ks].transpose()
    c[rows, cols] = (acc.to(T.f32) * scale_a[rows, 0:1] * scale_w[0:1, cols]).to(T.bf16)


@kernel
def matmul_f32(t: Tiling, a: Matrix[T.f32], b: Matrix[T.f32], c: Matrix[T.f32]) -> None:
    rows, cols = block.tile(t.bm, t.bn)
    acc = zeros(T.f32, t.bm, t.bn)
    for ks in pipelined(a.shape[1], t.bk):
        acc += a[rows, ks] @ b[ks, cols]
    c[rows, cols] = acc


@struct
class Attention:
    bq: Const[int] = 128
    bk: Const[int] = 64
    d: Const[int] = 128
    causal: Const[bool] = False


@kernel
def attention(
    t: Attention,
    q: Tensor[F, int, int, int],
    k: Tensor[F, int, int, int],
    v: Tensor[F, int, int, int],
    o: Tensor[F, int, int, int],
    scale: T.f32,
) -> None:
    rows, head = block.tile(t.bq), block.index().y
    q_pos = arange(t.bq, 0, rank=2, start=block.index().x * t.bq)
    m, total, acc = zeros(T.f32, t.bq, 1).sub(1.0e30), zeros(T.f32, t.bq, 1), zeros(T.f32, t.bq, t.d)
    qt = q[head, rows, slice(0, t.d)]
    for c in range(0, k.shape[1], t.bk):
        s = (qt @ k[head, c : c + t.bk, slice(0, t.d)].transpose()).mul(scale)
        if t.causal:
            s = where(arange(t.bk, 1, rank=2, start=c) <= q_pos, s, -1.0e30)
        m_new = m.maximum(s.max(keepdims=True))
        p, corr = (s - m_new).exp2(), (m - m_new).exp2()
        total *= corr
        total += p.sum(keepdims=True)
        acc *= corr
        acc += p.to(q.dtype) @ v[head, c : c + t.bk, slice(0, t.d)]
        m = m_new
    o[head, rows, slice(0, t.d)] = (acc / total).to(o.dtype)


@struct
class Rows:
    rows: Const[int] = 4
    cols: Const[int] = 1024


@kernel
def softmax(t: Rows, x: Matrix[F], y: Matrix[F]) -> None:
    rows = block.tile(t.rows)
    m = zeros(T.f32, t.rows, 1).sub(3.0e38)
    s = zeros(T.f32, t.rows, 1)
    for cs in pipelined(x.shape[1], t.cols):
        v = x[rows, cs].to(T.f32)
        m_new = maximum(m, v.max(keepdims=True))
        s = s * (m - m_new).exp() + (v - m_new).exp().sum(keepdims=True)
        m = m_new
    for cs in pipelined(x.shape[1], t.cols):
        y[rows, cs] = (x[rows, cs].to(T.f32) - m).exp().div(s).to(y.dtype)


TORCH = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32, "fp8": torch.float8_e4m3fn, "i8": torch.int8}
KRN = {"bf16": BF16, "f16": F16, "f32": F32, "fp8": F8E4M3, "i8": I8}
SIZE = {"bf16": 2, "f16": 2, "f32": 4, "fp8": 1, "i8": 1}
FLOP_LIMIT = 2.0 * 8192**3


def listed():
    return [
        # the linear layer of a large prefill or training batch: whole tiles, the matrix cores' rate
        {"name": "gemm_bf16_8192", "op": "gemm", "dtype": "bf16", "m": 8192, "n": 8192, "k": 8192},
        # one token through an fp8 weight: the weight is read once, nothing else matters
        {"name": "gemm_fp8_decode", "op": "gemm", "dtype": "fp8", "m": 1, "n": 8192, "k": 8192},
        # an int8 up-projection over a prefill of 4096 tokens
        {"name": "gemm_w8a8_prefill", "op": "gemm", "dtype": "i8", "m": 4096, "n": 14336, "k": 4096},
        # the down-projection of a decoding batch of 256 sequences: few output tiles, a long K
        {"name": "gemm_bf16_batch", "op": "gemm", "dtype": "bf16", "m": 256, "n": 4096, "k": 14336},
        # a feed-forward layer of sizes that fit no tile, with its bias and activation
        {"name": "matmul_f16_ragged", "op": "matmul", "dtype": "f16", "m": 1000, "n": 3001, "k": 777,
         "epilogue": "bias_gelu"},
        # self-attention over a batch of four prompts
        {"name": "attn_prefill", "op": "attention", "dtype": "bf16", "heads": 128, "sq": 4096, "sk": 4096, "d": 128,
         "causal": True},
        # the next token of the same four sequences: one query per head against the cache
        {"name": "attn_decode", "op": "attention", "dtype": "bf16", "heads": 128, "sq": 1, "sk": 4096, "d": 128,
         "causal": False},
        # an encoder layer over one short ragged sequence
        {"name": "attn_short", "op": "attention", "dtype": "f16", "heads": 16, "sq": 1000, "sk": 1000, "d": 64,
         "causal": False},
        # a large softmax over whole lines
        {"name": "softmax_f16", "op": "softmax", "dtype": "f16", "rows": 32768, "cols": 4096},
        # a softmax over an odd number of classes, rows at every alignment
        {"name": "softmax_bf16_odd", "op": "softmax", "dtype": "bf16", "rows": 1024, "cols": 50001},
        # the smallest call: a float32 product of 256 x 256 matrices
        {"name": "matmul_f32_256", "op": "matmul_f32", "m": 256, "n": 256, "k": 256, "tile": 32},
        # attention heads of 32 elements
        {"name": "attn_d32", "op": "attention_d32", "dtype": "bf16", "heads": 16, "sq": 512, "sk": 512, "tile": 64,
         "causal": True},
    ]


def _size(rng, low, high):
    """A size between low and high, spread over its logarithm."""
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def _inner(rng, low, high):
    """A size as layers have them: mostly a multiple of 128, sometimes of 16, sometimes anything."""
    step = rng.choice([128, 128, 128, 16, 1])
    return max(step, _size(rng, low, high) // step * step)


def draw(rng):
    op = rng.choice(["gemm", "gemm", "gemm", "matmul", "attention", "attention", "attention", "softmax", "matmul_f32",
                     "attention_d32"])
    if op == "gemm":
        dtype = rng.choice(["bf16", "f16", "fp8", "i8"])
        n, k = _inner(rng, 512, 16384), _inner(rng, 512, 16384)
        m = _size(rng, 1, 8192)
        m = max(1, min(m, int(FLOP_LIMIT / (2 * n * k))))
        return {"op": op, "dtype": dtype, "m": m, "n": n, "k": k}
    if op == "matmul":
        return {"op": op, "dtype": rng.choice(["bf16", "f16"]), "m": _size(rng, 16, 4096), "n": _inner(rng, 64, 8192),
                "k": _inner(rng, 64, 8192), "epilogue": rng.choice(["none", "bias", "relu", "bias_gelu", "silu"])}
    if op == "attention":
        dtype, d, heads = rng.choice(["bf16", "f16"]), rng.choice([64, 128]), _size(rng, 4, 128)
        if rng.random() < 0.5:  # decode: one query, or the few of a speculative step
            return {"op": op, "dtype": dtype, "heads": heads, "sq": rng.choice([1, 1, 1, 4, 8]),
                    "sk": _size(rng, 256, 16384), "d": d, "causal": False}
        seq = _size(rng, 64, 4096)
        return {"op": op, "dtype": dtype, "heads": heads, "sq": seq, "sk": seq, "d": d, "causal": rng.random() < 0.6}
    if op == "softmax":
        cols = _inner(rng, 64, 65536)
        return {"op": op, "dtype": rng.choice(["bf16", "f16", "f32"]), "rows": _size(rng, 16, max(16, 2**27 // cols)),
                "cols": cols}
    if op == "matmul_f32":
        return {"op": op, "m": _size(rng, 32, 2048), "n": _size(rng, 32, 2048), "k": _size(rng, 32, 2048),
                "tile": rng.choice([32, 64])}
    seq = _size(rng, 64, 1024)
    return {"op": op, "dtype": rng.choice(["bf16", "f16"]), "heads": _size(rng, 2, 32), "sq": seq, "sk": seq,
            "tile": rng.choice([32, 64]), "causal": rng.random() < 0.5}


def _random(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, *shape, scale=1.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32) * scale


def _inputs(case, seed):
    """The input tensors of a case, from its seed alone."""
    g, op, dtype = _random(seed), case["op"], TORCH[case.get("dtype", "f32")]
    if op in ("gemm", "matmul", "matmul_f32"):
        m, n, k = case["m"], case["n"], case["k"]
        a, b = _normal(g, m, k), _normal(g, *((n, k) if op == "gemm" else (k, n)), scale=k**-0.5)
        if dtype == torch.int8:  # symmetric per-row quantisation of activations and weights
            sa, sw = a.abs().amax(1, keepdim=True) / 127, b.abs().amax(1, keepdim=True) / 127
            return {"a": (a / sa).round().to(dtype), "b": (b / sw).round().to(dtype), "sa": sa,
                    "sb": sw.reshape(1, n).contiguous()}
        if dtype == torch.float8_e4m3fn:
            sa, sb = float(a.abs().amax()) / 448, float(b.abs().amax()) / 448
            return {"a": (a / sa).to(dtype), "b": (b / sb).to(dtype), "sa": sa, "sb": sb}
        return {"a": a.to(dtype), "b": b.to(dtype), "bias": _normal(g, n).to(dtype)}
    if op == "softmax":
        return {"x": (_normal(g, case["rows"], case["cols"]) * 4).to(dtype)}
    d = case.get("d", 32)
    return {"q": _normal(g, case["heads"], case["sq"], d).to(dtype),
            "k": _normal(g, case["heads"], case["sk"], d).to(dtype),
            "v": _normal(g, case["heads"], case["sk"], d).to(dtype)}


def _krn(device, t):
    """torch memory as a krn tensor, without a copy."""
    kinds = {torch.bfloat16: BF16, torch.float16: F16, torch.float32: F32, torch.float8_e4m3fn: F8E4M3, torch.int8: I8}
    return HIPTensor(device, t.data_ptr(), kinds[t.dtype], tuple(t.shape), owner=t)


def prepare(case, seed):
    device, op = device_of("gfx950"), case["op"]
    given = _inputs(case, seed)
    x = {name: _krn(device, t) if isinstance(t, torch.Tensor) else t for name, t in given.items()}
    out_type = TORCH[case.get("dtype", "f32")] if case.get("dtype") not in ("fp8", "i8") else torch.bfloat16
    shape = {"softmax": lambda: (case["rows"], case["cols"]),
             "attention": lambda: (case["heads"], case["sq"], case["d"]),
             "attention_d32": lambda: (case["heads"], case["sq"], 32)}.get(op, lambda: (case["m"], case["n"]))()
    out = torch.empty(shape, device="cuda", dtype=out_type)
    y = _krn(device, out)
    if op == "gemm":
        tiling = Tiling(256, 256, 128 if case["dtype"] in ("fp8", "i8") else 64)
        if case["dtype"] == "fp8":
            call = linear_fp8[tiling].bind(x["a"], x["b"], y, x["sa"], x["sb"])
        elif case["dtype"] == "i8":
            call = linear_w8a8[tiling].bind(x["a"], x["b"], x["sa"], x["sb"], y)
        else:
            call = linear[tiling].bind(x["a"], x["b"], y)
    elif op == "matmul":
        bias = x["bias"] if "bias" in case["epilogue"] else None

        def call():
            lib.matmul(x["a"], x["b"], epilogue=case["epilogue"], bias=bias, out=y, library="ours")
    elif op == "matmul_f32":
        call = matmul_f32[Tiling(case["tile"], case["tile"], case["tile"] // 2)].bind(x["a"], x["b"], y)
    elif op == "softmax":
        launch = Blocks(-(-case["rows"] // 4))
        call = device.launcher(softmax, launch).bind(Rows(), x["x"], y)
    else:
        d = case.get("d", 32)
        tiling = Attention(128, 64, d, case["causal"]) if op == "attention" else Attention(case["tile"], case["tile"], d,
                                                                                           case["causal"])
        launch = Blocks(-(-case["sq"] // tiling.bq), case["heads"])
        call = device.launcher(attention, launch).bind(tiling, x["q"], x["k"], x["v"], y, math.log2(math.e) / math.sqrt(d))
    torch.cuda.synchronize()  # the runtime has streams of its own
    return {"call": call, "out": out, "inputs": given}


def run(state):
    state["call"]()
    return state["out"]


def work(case):
    op, size = case["op"], SIZE[case.get("dtype", "f32")]
    if op in ("gemm", "matmul", "matmul_f32"):
        m, n, k = case["m"], case["n"], case["k"]
        out = 4 if op == "matmul_f32" else 2
        vectors = 4 * (m + n) if size == 1 and case["dtype"] == "i8" else 2 * n if "bias" in case.get("epilogue", "") else 0
        return {"bytes": size * (m * k + n * k) + out * m * n + vectors, "flops": 2 * m * n * k}
    if op == "softmax":
        return {"bytes": 2 * size * case["rows"] * case["cols"], "flops": 0}
    d, h, sq, sk = case.get("d", 32), case["heads"], case["sq"], case["sk"]
    pairs = sq * (sq + 1) / 2 if case["causal"] else sq * sk
    return {"bytes": size * h * d * (2 * sq + 2 * sk), "flops": 4 * h * d * pairs}


def tolerance(case):
    """About four times the distance of the path from 64 bits, which the rounding of the result to its type gives most
    of; attention rounds its probabilities to 16 bits as well. int8 products are exact, and so is their scaling."""
    if case.get("dtype") == "i8":
        return "exact"
    if case["op"] == "matmul_f32":
        return {"rel": 2e-6}
    if case["op"] == "softmax":
        return {"rel": {"bf16": 7e-3, "f16": 9e-4, "f32": 2e-6}[case["dtype"]]}
    if case["op"] in ("attention", "attention_d32"):
        return {"rel": {"bf16": 9e-3, "f16": 1.2e-3}[case["dtype"]]}
    return {"rel": {"bf16": 7e-3, "fp8": 7e-3, "f16": 9e-4}[case["dtype"]]}


def exact(case, seed):
    x, op = _inputs(case, seed), case["op"]
    wide = {name: t.to(torch.float64) if isinstance(t, torch.Tensor) else t for name, t in x.items()}
    if op in ("gemm", "matmul", "matmul_f32"):
        c = wide["a"] @ (wide["b"].T if op == "gemm" else wide["b"])
        if "sa" in x:
            return c * (wide["sa"] * wide["sb"])
        epilogue = case.get("epilogue", "")
        if "bias" in epilogue:
            c += wide["bias"]
        if "relu" in epilogue:
            c = c.relu()
        if "gelu" in epilogue:
            c = 0.5 * c * (1 + torch.erf(c / math.sqrt(2)))
        if "silu" in epilogue:
            c = c * torch.sigmoid(c)
        return c
    if op == "softmax":
        return torch.softmax(wide["x"], dim=1)
    out = torch.empty(wide["q"].shape, device="cuda", dtype=torch.float64)
    hidden = torch.ones(case["sq"], case["sk"], device="cuda", dtype=torch.bool).triu(1) if case["causal"] else None
    for h in range(case["heads"]):
        s = (wide["q"][h] @ wide["k"][h].T) / math.sqrt(case.get("d", 32))
        if hidden is not None:
            s.masked_fill_(hidden, -math.inf)
        out[h] = torch.softmax(s, dim=1) @ wide["v"][h]
    return out

"""The calls a program makes of this library, from the smallest to the largest, as measurable cases.

Each case is one call through a public entry point: ``tensorvia_amd.gemm`` on torch tensors, or the
C-ABI (``tv_hip_gemm``, ``tv_hip_gemm_ex``, ``tv_hip_repack``) with a descriptor that the program
packed when it loaded its weights, as a serving loop does.  Three kinds of calls:

* ``mul``: A @ B, with B row-major (``kn``) or the transposed view of a row-major [N, K] tensor
  (``nk``), optionally batched, B shared by the batch or one per batch entry;
* ``linear``: act(x @ W + bias) through the fused epilogue;
* ``permute``: a permuted view copied to a contiguous tensor.

``draw`` gives further cases of the same families: other sizes (odd ones among them), data types,
weight layouts and activations.
"""
from __future__ import annotations

import ctypes
import math

import torch

import tensorvia_amd as tv

_DT = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16,
       "i8": torch.int8, "i16": torch.int16, "i32": torch.int32}
_ES = {"f64": 8, "f32": 4, "bf16": 2, "f16": 2, "i8": 1, "i16": 2, "i32": 4}
_ACT = {"none": tv.ACT_NONE, "relu": tv.ACT_RELU, "silu": tv.ACT_SILU, "sigmoid": tv.ACT_SIGMOID, "tanh": tv.ACT_TANH}


def _mul(family, a, b, c, batch, m, k, n, layout="kn", shared=True, values="uniform", entry="gemm"):
    return {"kind": "mul", "family": family, "a": a, "b": b, "c": c, "batch": batch, "m": m, "k": k, "n": n,
            "layout": layout, "shared": shared, "values": values, "entry": entry}


def _linear(dt, m, k, n, layout, act, bias):
    return {"kind": "linear", "family": "linear", "a": dt, "b": dt, "c": dt, "batch": 0, "m": m, "k": k, "n": n,
            "layout": layout, "shared": True, "values": "weights", "act": act, "bias": bias}


def _permute(dt, shape, axes):
    return {"kind": "permute", "family": "permute", "dt": dt, "shape": "x".join(map(str, shape)),
            "axes": "".join(map(str, axes))}


def listed():
    def named(name, case):
        return {"name": name, **case}
    return [
        # A tiny product of an application with many of them: launch and host cost.
        named("small_f32", _mul("small", "f32", "f32", "f32", 0, 32, 64, 48)),
        # One token through an MLP up-projection: the weights stream from memory.
        named("decode_bf16", _mul("decode", "bf16", "bf16", "bf16", 0, 1, 4096, 11008, values="weights", entry="abi")),
        # The same layer for 48 sequences decoded together, weights stored [out, in] and used as W.t().
        named("decode48_f16", _mul("decode_batch", "f16", "f16", "f16", 0, 48, 4096, 11008, layout="nk", values="weights",
                                   entry="abi")),
        # Attention scores Q @ K^T, K a transposed view: the output is most of the traffic.
        named("scores_f16", _mul("scores", "f16", "f16", "f16", 32, 2048, 128, 2048, layout="nk", shared=False,
                                 values="heads")),
        # Attention output P @ V, P the softmax of the scores.
        named("values_bf16", _mul("values", "bf16", "bf16", "bf16", 32, 2048, 2048, 128, shared=False, values="probs")),
        # A prompt of 333 tokens through a linear layer with bias and SiLU (fused epilogue).
        named("prefill_silu_bf16", _linear("bf16", 333, 4096, 11008, "kn", "silu", True)),
        # The README benchmark's product.
        named("gemm_f32", _mul("gemm", "f32", "f32", "f32", 0, 2592, 2048, 4096)),
        # Odd sizes in fp32: no row is a whole number of 16-byte chunks.
        named("gemm_f32_odd", _mul("gemm", "f32", "f32", "f32", 0, 1001, 777, 1003)),
        # Quantised product, 8-bit in and out with wrap-around, exact.
        named("gemm_i8", _mul("gemm", "i8", "i8", "i8", 0, 4096, 4096, 4096)),
        # A batch of long prompts through one weight matrix: the largest call.
        named("gemm_bf16_batched", _mul("gemm_batched", "bf16", "bf16", "bf16", 16, 2048, 4096, 4096)),
        # A product in double precision.
        named("gemm_f64", _mul("general", "f64", "f64", "f64", 0, 1000, 1000, 1000)),
        # The materialised transpose of K [heads, tokens, head size].
        named("transpose_f16", _permute("f16", (32, 2048, 128), (0, 2, 1))),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _size(rng, lo, hi):
    """A size of [lo, hi]: as drawn (odd or even), or rounded to a multiple of 64."""
    x = _log(rng, lo, hi)
    return max(64, x // 64 * 64) if rng.random() < 0.6 and x >= 64 else x


def draw(rng):
    f = rng.choice(["small", "decode", "decode_batch", "scores", "values", "linear", "gemm_f32", "gemm_i8", "gemm_half",
                    "gemm_batched", "general", "permute"])
    if f == "small":
        dt = rng.choice(["f32", "f32", "bf16", "f16", "i8"])
        batch = rng.choice([0, 0, _log(rng, 2, 8)])
        return _mul("small", dt, dt, dt, batch, _log(rng, 1, 96), _log(rng, 1, 96), _log(rng, 1, 96), shared=False)
    if f == "decode":
        dt = rng.choice(["bf16", "bf16", "f16", "i8", "f32"])
        return _mul("decode", dt, dt, "i32" if dt == "i8" else dt, 0, _log(rng, 1, 8), _size(rng, 1024, 4096),
                    _size(rng, 1024, 11008), layout=rng.choice(["kn", "nk"]), values="weights", entry="abi")
    if f == "decode_batch":
        dt = rng.choice(["bf16", "f16", "f16", "i8"])
        return _mul("decode_batch", dt, dt, "i32" if dt == "i8" else dt, 0, _log(rng, 9, 128), _size(rng, 1024, 4096),
                    _size(rng, 1024, 11008), layout=rng.choice(["kn", "nk"]), values="weights", entry="abi")
    if f in ("scores", "values"):
        dt = rng.choice(["bf16", "f16"])
        heads, s, d = rng.choice([8, 12, 16, 32]), _size(rng, 64, 2048), rng.choice([64, 80, 96, 128])
        if f == "scores":
            return _mul("scores", dt, dt, dt, heads, s, d, s, layout="nk", shared=False, values="heads")
        return _mul("values", dt, dt, dt, heads, s, s, d, shared=False, values="probs")
    if f == "linear":
        return _linear(rng.choice(["bf16", "f16"]), _log(rng, 129, 1024), _size(rng, 1024, 4096), _size(rng, 1024, 11008),
                       rng.choice(["kn", "nk"]), rng.choice(["none", "relu", "silu", "sigmoid", "tanh"]), rng.random() < 0.7)
    if f == "gemm_f32":
        return _mul("gemm", "f32", "f32", "f32", 0, _size(rng, 128, 2592), _size(rng, 128, 2048), _size(rng, 128, 4096),
                    layout=rng.choice(["kn", "nk"]))
    if f == "gemm_i8":
        return _mul("gemm", "i8", "i8", rng.choice(["i8", "i32"]), 0, _size(rng, 256, 4096), _size(rng, 256, 4096),
                    _size(rng, 256, 4096), layout=rng.choice(["kn", "nk"]))
    if f == "gemm_half":
        dt = rng.choice(["bf16", "f16"])
        return _mul("gemm", dt, dt, dt, 0, _size(rng, 256, 4096), _size(rng, 256, 4096), _size(rng, 256, 4096),
                    layout=rng.choice(["kn", "nk"]))
    if f == "gemm_batched":
        dt = rng.choice(["bf16", "f16"])
        return _mul("gemm_batched", dt, dt, dt, _log(rng, 2, 16), _size(rng, 128, 2048), _size(rng, 256, 4096),
                    _size(rng, 256, 4096), shared=rng.random() < 0.6)
    if f == "general":
        # Pairs the matrix cores have no type for: doubles, fp32 activations on 16-bit weights,
        # integers wider than 8 bits.
        a, b, c = rng.choice([("f64", "f64", "f64"), ("f64", "f64", "f64"), ("f32", "bf16", "f32"), ("f32", "f16", "f32"),
                              ("i32", "i32", "i32"), ("i16", "i16", "i16")])
        return _mul("general", a, b, c, 0, _size(rng, 32, 1280), _size(rng, 32, 600), _size(rng, 32, 1280),
                    layout=rng.choice(["kn", "nk"]))
    dt = rng.choice(["f16", "bf16", "f32", "i8", "f64"])
    heads, s, d = rng.choice([4, 8, 16, 32]), _size(rng, 64, 2048), rng.choice([48, 64, 80, 128])
    if dt == "f64":
        heads = min(heads, 8)
    if rng.random() < 0.5:  # [heads, tokens, size] -> [heads, size, tokens]
        return _permute(dt, (heads, s, d), (0, 2, 1))
    return _permute(dt, (1, s, heads, d), (0, 2, 1, 3))  # [1, tokens, heads, size] -> [1, heads, tokens, size]


# ---- inputs ------------------------------------------------------------------------------------

def _uniform(shape, lo, hi, dt, g):
    if dt.startswith("i"):
        return torch.randint(int(lo), int(hi) + 1, shape, generator=g, device="cuda", dtype=torch.int32).to(_DT[dt])
    t = torch.rand(shape, generator=g, device="cuda", dtype=torch.float64 if dt == "f64" else torch.float32)
    return t.mul_(hi - lo).add_(lo).to(_DT[dt])


def _normal(shape, scale, dt, g):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(scale).to(_DT[dt])


def _inputs(case, seed):
    """The operands as a program holds them; B of layout nk is the transposed view of [.., N, K]."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    batch, m, k, n = case["batch"], case["m"], case["k"], case["n"]
    lead = (batch,) if batch else ()
    sa = lead + (m, k)
    sb = (() if case["shared"] else lead) + ((k, n) if case["layout"] == "kn" else (n, k))
    da, db, v = case["a"], case["b"], case["values"]
    if v == "uniform":  # seeded Tensor::Random ranges of the benchmark configurations
        lim = 10 if da.startswith("i") else 1
        a, b = _uniform(sa, -lim, lim, da, g), _uniform(sb, -lim, lim, db, g)
    elif v == "weights":  # activations normal(0, 1), weights uniform[-0.05, 0.05]; int8 quantised
        if da == "i8":
            a, b = _uniform(sa, -127, 127, da, g), _uniform(sb, -127, 127, db, g)
        else:
            a, b = _normal(sa, 1.0, da, g), _uniform(sb, -0.05, 0.05, db, g)
    elif v == "heads":  # queries and keys normal(0, 1) / sqrt(head size)
        a, b = _normal(sa, 1 / math.sqrt(k), da, g), _normal(sb, 1 / math.sqrt(k), db, g)
    else:  # attention probabilities and values
        a = torch.softmax(torch.randn(sa, generator=g, device="cuda", dtype=torch.float32), -1).to(_DT[da])
        b = _normal(sb, 1.0, db, g)
    if case["layout"] == "nk":
        b = b.transpose(-1, -2)
    bias = _uniform((n,), -1, 1, case["c"], g) if case.get("bias") else None
    return a, b, bias


def _permute_input(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    shape = tuple(map(int, case["shape"].split("x")))
    dt = case["dt"]
    src = _uniform(shape, -100, 100, dt, g) if dt == "i8" else _normal(shape, 1.0, dt, g)
    return src, src.permute(tuple(map(int, case["axes"])))


def prepare(case, seed):
    if case["kind"] == "permute":
        src, view = _permute_input(case, seed)
        out = torch.empty(view.shape, dtype=view.dtype, device="cuda")
        args = tv.TvRepackArgs()
        args.ndim, args.elem_size = view.dim(), view.element_size()
        for d in range(view.dim()):
            args.shape[d], args.strides[d] = view.shape[d], view.stride(d)
        args.src, args.dst = src.data_ptr(), out.data_ptr()
        return {"call": "repack", "args": args, "out": out, "keep": src}
    a, b, bias = _inputs(case, seed)
    if case["kind"] == "mul" and case["entry"] == "gemm":
        return {"call": "gemm", "a": a, "b": b, "out_dtype": tv.torch_to_tv(_DT[case["c"]])}
    out = torch.empty((a.shape[0], b.shape[1]), dtype=_DT[case["c"]], device="cuda")
    state = {"call": "abi", "args": tv.make_args(a, b, out), "out": out, "keep": (a, b, bias)}
    if case["kind"] == "linear":
        ep = tv.TvEpilogue()
        ep.act = _ACT[case["act"]]
        if bias is not None:
            ep.bias, ep.sbias_n = bias.data_ptr(), 1
        state["call"], state["epilogue"] = "abi_ex", ep
    return state


def run(state):
    call = state["call"]
    if call == "gemm":
        return tv.gemm(state["a"], state["b"], out_dtype=state["out_dtype"])
    stream = torch.cuda.current_stream().cuda_stream
    if call == "abi":
        tv.check(tv.lib().tv_hip_gemm(ctypes.byref(state["args"]), stream))
    elif call == "abi_ex":
        tv.check(tv.lib().tv_hip_gemm_ex(ctypes.byref(state["args"]), ctypes.byref(state["epilogue"]), stream))
    else:
        tv.check(tv.lib().tv_hip_repack(ctypes.byref(state["args"]), stream))
    return state["out"]


# ---- what a pass cannot do without, and what it must return --------------------------------------

def work(case):
    if case["kind"] == "permute":
        return {"bytes": 2 * math.prod(map(int, case["shape"].split("x"))) * _ES[case["dt"]], "flops": 0}
    bt = case["batch"] or 1
    m, k, n = case["m"], case["k"], case["n"]
    nbytes = bt * m * k * _ES[case["a"]] + (1 if case["shared"] else bt) * k * n * _ES[case["b"]] + bt * m * n * _ES[case["c"]]
    if case.get("bias"):
        nbytes += n * _ES[case["c"]]
    return {"bytes": nbytes, "flops": 2 * bt * m * n * k}


def tolerance(case):
    if case["kind"] == "permute" or case["c"].startswith("i"):
        return "exact"
    # About four times the distance from the 64-bit result that this path and torch's own product
    # show over the ranges: at 16 bits that is the rounding of the result (1.66e-3, 2.1e-4; two
    # orders of summation differ by less, 4e-5), else the summation (f32 2e-8 to 8e-7 with K).
    return {"rel": {"bf16": 6.6e-3, "f16": 8.4e-4, "f32": 3.2e-6, "f64": 5e-15}[case["c"]]}


def exact(case, seed):
    if case["kind"] == "permute":
        return _permute_input(case, seed)[1].contiguous()
    a, b, bias = _inputs(case, seed)
    c = torch.matmul(a.double(), b.double().contiguous())
    if case["c"].startswith("i"):  # sums below 2^53: exact; the result type keeps its low bits
        return c.to(torch.int64).to(_DT[case["c"]])
    if bias is not None:
        c += bias.double()
    act = case.get("act", "none")
    if act != "none":
        c = {"relu": torch.relu, "silu": torch.nn.functional.silu, "sigmoid": torch.sigmoid, "tanh": torch.tanh}[act](c)
    return c

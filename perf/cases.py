"""Workloads of the tensor library: what a program that runs transformer models
on it has it do, one call (or one short chain of calls) per case.

A case is a dict of plain values whose "kind" selects the work:

  decoder  the non-GEMM chain of a decoder layer on f16 activations:
           residual add + RMSNorm, RoPE on q and k, SwiGLU
  vision   the non-GEMM chain of a vision-encoder layer: layer norm, bias +
           tanh-GELU over the MLP width, residual add
  attn     scaled dot-product attention on device buffers
  quant    linear layer with Q8_0 / Q4_0 weights, f16 activations
  linear   linear layer with f16 or f32 weights
  rows     one row operation over the last dimension
  view     strided / permuted view with optional broadcast operands
  reduce   whole-tensor sum and max, or argmax
  embed    embedding lookup

prepare() builds the operands on the GPU from the seed alone and wraps the
library's device buffers as torch tensors (no copy), which is what run()
returns; exact() computes the same outputs in float64 with plain torch.
"""
import math

import torch

from inference_c_amd import Sdk
from inference_c_amd.sdk import TensorView

EPS = 1e-6
THETA = 10000.0
POSITION = 7          # RoPE offset: positions POSITION ..
TORCH = {"f16": torch.float16, "f32": torch.float32, "f64": torch.float64,
         "u8": torch.uint8, "u32": torch.int32}
TYPESTR = {"f16": "<f2", "f32": "<f4", "f64": "<f8", "u8": "|u1", "u32": "<i4"}
SIZE = {"f16": 2, "f32": 4}
BLOCK = {"q8_0": 34, "q4_0": 18}

_sdk = None


def sdk():
    global _sdk
    if _sdk is None:
        _sdk = Sdk()
        _sdk.require_device()
    return _sdk


# ---- the cases ------------------------------------------------------------------

def listed():
    return [
        # one decode step of a small decoder layer: three launches, nothing to stream
        {"name": "decoder_decode", "kind": "decoder", "tokens": 1, "hidden": 2048, "heads": 32,
         "kv_heads": 32, "dim": 64, "inter": 8192},
        # the same layer over a 4096-token prompt: memory bandwidth
        {"name": "decoder_prefill", "kind": "decoder", "tokens": 4096, "hidden": 2048, "heads": 32,
         "kv_heads": 32, "dim": 64, "inter": 8192},
        # prompt attention of a grouped-query decoder
        {"name": "attn_prefill", "kind": "attn", "dtype": "f16", "batch": 1, "heads": 32,
         "kv_heads": 8, "q_len": 2048, "kv_len": 2048, "dim": 128, "causal": True, "mask": False},
        # vision encoder with a class token (ragged length) and 80-wide heads
        {"name": "attn_vision", "kind": "attn", "dtype": "f16", "batch": 1, "heads": 16,
         "kv_heads": 16, "q_len": 1025, "kv_len": 1025, "dim": 80, "causal": False, "mask": False},
        # vision encoder kept in f32
        {"name": "attn_vision_f32", "kind": "attn", "dtype": "f32", "batch": 1, "heads": 12,
         "kv_heads": 12, "q_len": 1024, "kv_len": 1024, "dim": 64, "causal": False, "mask": False},
        # one decode step of eight sequences over their KV caches
        {"name": "attn_decode", "kind": "attn", "dtype": "f16", "batch": 8, "heads": 32,
         "kv_heads": 8, "q_len": 1, "kv_len": 4096, "dim": 128, "causal": True, "mask": False},
        # MLP up-projection of a 512-token prompt with 8-bit weights
        {"name": "quant_prefill", "kind": "quant", "format": "q8_0", "rows": 512, "in": 4096,
         "out": 14336},
        # one decode step of four sequences through a large 4-bit MLP projection
        {"name": "quant_decode", "kind": "quant", "format": "q4_0", "rows": 4, "in": 8192,
         "out": 28672},
        # f16 projection with bias for a batch of 16 decode steps
        {"name": "linear_batch", "kind": "linear", "dtype": "f16", "rows": 16, "in": 4096,
         "out": 4096, "bias": True},
        # sampling: softmax over the vocabulary for a batch of logits
        {"name": "softmax_vocab", "kind": "rows", "op": "softmax", "dtype": "f32", "rows": 32,
         "width": 128256},
        # image preprocessing: NHWC pixels to normalised NCHW, (x - mean) / std
        {"name": "image_nchw", "kind": "view", "form": "nhwc_nchw", "dtype": "f32", "a": 8, "b": 512,
         "c": 512, "d": 3, "operands": True},
        # activation statistics: sum and max of one tensor of odd size
        {"name": "sum_max", "kind": "reduce", "op": "sum_max", "dtype": "f32", "n": (1 << 22) + 3},
    ]


def _log(rng, low, high):
    """An integer of [low, high], uniform in its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["decoder", "vision", "attn", "attn", "attn", "quant", "quant", "linear",
                       "linear", "rows", "rows", "view", "reduce", "embed"])
    if kind == "decoder":
        dim = rng.choice([64, 128])
        heads = rng.choice([9, 14, 15, 16, 32])
        kv = rng.choice([h for h in range(1, heads + 1) if heads % h == 0])
        return {"kind": kind, "tokens": _log(rng, 1, 3000), "hidden": rng.choice([576, 960, 2048, 3072]),
                "heads": heads, "kv_heads": kv, "dim": dim,
                "inter": rng.choice([1536, 2560, 4864, 8192])}
    if kind == "vision":
        width = rng.choice([768, 1000, 1152, 1280])
        return {"kind": kind, "dtype": rng.choice(["f16", "f16", "f32"]), "tokens": _log(rng, 40, 6000),
                "width": width, "inter": rng.choice([width * 4, 4304])}
    if kind == "attn":
        dtype = rng.choice(["f16", "f16", "f16", "f32"])
        dim = rng.choice([64, 64, 128, 128, 32, 72, 80, 96, 256])
        kv = rng.choice([1, 2, 3, 4, 8, 12])
        heads = kv * rng.choice([1, 1, 2, 3, 4])
        form = rng.choice(["prefill", "prefill", "decode", "chunk"])
        if form == "decode":      # one new token against the cache
            c = {"batch": _log(rng, 1, 24), "q_len": 1, "kv_len": _log(rng, 64, 8192)}
        elif form == "chunk":     # a few new tokens (speculation, chunked prompts)
            c = {"batch": _log(rng, 1, 4), "q_len": _log(rng, 2, 64), "kv_len": _log(rng, 128, 4096)}
        else:
            n = _log(rng, 64, 2048)
            c = {"batch": 1 if n > 512 else _log(rng, 1, 8), "q_len": n, "kv_len": n}
        while c["batch"] * heads * c["q_len"] * c["kv_len"] * dim > 8 << 30:
            c["batch"] = max(1, c["batch"] // 2)
            c["q_len"], c["kv_len"] = max(1, c["q_len"] * 3 // 4), c["kv_len"] * 3 // 4
        return {"kind": kind, "dtype": dtype, "heads": heads, "kv_heads": kv, "dim": dim, **c,
                "causal": rng.random() < 0.6, "mask": rng.random() < 0.2}
    if kind == "quant":
        rows = _log(rng, 1, 2048)
        inn, out = 32 * _log(rng, 16, 256), _log(rng, 256, 8192)
        while rows * inn * out > 512 * 4096 * 14336:
            rows = rows // 2
        return {"kind": kind, "format": rng.choice(["q8_0", "q4_0"]), "rows": rows, "in": inn,
                "out": out}
    if kind == "linear":
        dtype = rng.choice(["f16", "f16", "f16", "f32"])
        rows, out = _log(rng, 1, 1024), _log(rng, 128, 8192)
        inn = rng.choice([1, 8, 8, 8]) * _log(rng, 32, 1000)
        return {"kind": kind, "dtype": dtype, "rows": rows, "in": inn, "out": out,
                "bias": rng.random() < 0.5}
    if kind == "rows":
        op = rng.choice(["softmax", "rms_norm", "layer_norm", "row_sum", "row_max"])
        width = _log(rng, 64, 150000)
        return {"kind": kind, "op": op, "dtype": rng.choice(["f16", "f32"]),
                "rows": _log(rng, 1, max(1, min(65536, (1 << 24) // width))), "width": width}
    if kind == "view":
        form = rng.choice(["nhwc_nchw", "nchw_nhwc", "transpose", "heads"])
        if form in ("nhwc_nchw", "nchw_nhwc"):
            d = {"a": rng.randint(1, 8), "b": _log(rng, 96, 512), "c": _log(rng, 96, 512), "d": 3}
        elif form == "transpose":
            d = {"a": rng.choice([1, 1, 8]), "b": _log(rng, 64, 2048), "c": _log(rng, 64, 2048), "d": 1}
        else:
            d = {"a": rng.randint(1, 4), "b": _log(rng, 64, 2048), "c": rng.choice([8, 12, 16, 32]),
                 "d": rng.choice([64, 72, 128])}
        return {"kind": kind, "form": form, "dtype": rng.choice(["f16", "f32"]), **d,
                "operands": rng.random() < 0.5}
    if kind == "reduce":
        op = rng.choice(["sum_max", "argmax"])
        return {"kind": kind, "op": op,
                "dtype": "f32" if op == "sum_max" else rng.choice(["f16", "f32"]),
                "n": _log(rng, 1000, 1 << 25)}
    return {"kind": "embed", "dtype": rng.choice(["f16", "f32"]), "count": _log(rng, 1, 16384),
            "vocab": rng.choice([32000, 49152]), "width": rng.choice([576, 960, 2048])}


# ---- inputs ---------------------------------------------------------------------

def _inputs(c, seed):
    """Name -> torch tensor on the GPU, from the seed alone."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 17)

    def normal(shape, dtype, mean=0.0, std=1.0):
        x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
        return (x * std + mean).to(TORCH[dtype])

    kind = c["kind"]
    if kind == "decoder":
        t, h = c["tokens"], c["hidden"]
        return {"x": normal((t, h), "f16"), "r": normal((t, h), "f16"),
                "w": normal((h,), "f16", 1.0, 0.1), "q": normal((t, c["heads"], c["dim"]), "f16"),
                "k": normal((t, c["kv_heads"], c["dim"]), "f16"),
                "gate": normal((t, c["inter"]), "f16"), "up": normal((t, c["inter"]), "f16")}
    if kind == "vision":
        t, w, d = c["tokens"], c["width"], c["dtype"]
        out = {"x": normal((t, w), d), "w": normal((w,), d, 1.0, 0.1), "b": normal((w,), d, 0.0, 0.1),
               "h": normal((t, c["inter"]), d), "hb": normal((c["inter"],), d, 0.0, 0.1)}
        out["y"] = normal((t, w), d)
        return out
    if kind == "attn":
        b, d = c["batch"], c["dtype"]
        out = {"q": normal((b, c["heads"], c["q_len"], c["dim"]), d),
               "k": normal((b, c["kv_heads"], c["kv_len"], c["dim"]), d),
               "v": normal((b, c["kv_heads"], c["kv_len"], c["dim"]), d)}
        if c["mask"]:   # a relative-position style bias
            out["mask"] = normal((c["q_len"], c["kv_len"]), d, 0.0, 0.5)
        return out
    if kind == "quant":
        blocks = c["in"] // 32
        w = normal((c["out"], blocks, 32), "f32", 0.0, 0.05)
        big = w.abs().amax(-1, keepdim=True)
        levels = 127.0 if c["format"] == "q8_0" else 7.0
        scale = (big / levels).to(torch.float16)
        q = torch.round(w / scale.float()).clamp_(-levels, levels)
        if c["format"] == "q8_0":
            body = q.to(torch.int8).view(torch.uint8)
        else:
            n = (q + 8).to(torch.uint8)
            body = n[..., :16] | (n[..., 16:] << 4)
        packed = torch.cat([scale.view(torch.uint8), body], dim=-1).contiguous()
        return {"x": normal((c["rows"], c["in"]), "f16"), "packed": packed}
    if kind == "linear":
        d = c["dtype"]
        out = {"x": normal((c["rows"], c["in"]), d), "w": normal((c["out"], c["in"]), d, 0.0, 0.05)}
        if c["bias"]:
            out["bias"] = normal((c["out"],), d)
        return out
    if kind == "rows":
        d, w = c["dtype"], c["width"]
        # logits of a few units for the softmax; activations for the rest
        out = {"x": normal((c["rows"], w), d, 0.25, 2.0 if c["op"] == "softmax" else 1.0)}
        if c["op"] in ("rms_norm", "layer_norm"):
            out["w"] = normal((w,), d, 1.0, 0.1)
        if c["op"] == "layer_norm":
            out["b"] = normal((w,), d, 0.0, 0.1)
        return out
    if kind == "view":
        shape, order = _view_shape(c)
        d = c["dtype"]
        out = {"x": normal(shape, d)}
        if c["operands"]:
            small = _broadcast_shape(c, [shape[i] for i in order])
            out["add"] = normal(small, d)
            out["mul"] = normal(small, d, 2.0, 0.5)
        return out
    if kind == "reduce":
        return {"x": normal((c["n"],), c["dtype"], 0.25, 1.0)}
    ids = torch.randint(0, c["vocab"], (c["count"],), generator=g, device="cuda", dtype=torch.int32)
    return {"table": normal((c["vocab"], c["width"]), c["dtype"]), "ids": ids}


def _view_shape(c):
    """Shape of the stored tensor and the order of its axes in the output."""
    if c["form"] == "nhwc_nchw":
        return (c["a"], c["b"], c["c"], c["d"]), (0, 3, 1, 2)
    if c["form"] == "nchw_nhwc":
        return (c["a"], c["d"], c["b"], c["c"]), (0, 2, 3, 1)
    if c["form"] == "transpose":
        return (c["a"], c["b"], c["c"]), (0, 2, 1)
    return (c["a"], c["b"], c["c"], c["d"]), (0, 2, 1, 3)


def _broadcast_shape(c, out):
    """Per-channel operands: channel axis of images, last axis elsewhere."""
    axis = 1 if c["form"] == "nhwc_nchw" else len(out) - 1
    return tuple(n if i == axis else 1 for i, n in enumerate(out))


# ---- state ------------------------------------------------------------------------

class _Memory:
    """A library tensor's device memory for torch.as_tensor (no copy)."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.__cuda_array_interface__ = {
            "shape": tensor.shape, "typestr": TYPESTR[tensor.dtype],
            "data": (tensor.device_ptr(), False), "version": 2}


def _as_torch(tensor):
    return torch.as_tensor(_Memory(tensor), device="cuda")


def _output_spec(c):
    """Output name -> (dtype, shape) of the buffers the caller preallocates."""
    kind = c["kind"]
    if kind == "decoder":
        h, i = (c["tokens"], c["hidden"]), (c["tokens"], c["inter"])
        return {"sum": ("f16", h), "normed": ("f16", h), "act": ("f16", i)}
    if kind == "vision":
        h, i = (c["tokens"], c["width"]), (c["tokens"], c["inter"])
        out = {"normed": (c["dtype"], h), "act": (c["dtype"], i), "sum": (c["dtype"], h)}
        return out
    if kind == "attn":
        return {"out": (c["dtype"], (c["batch"], c["heads"], c["q_len"], c["dim"]))}
    if kind == "quant":
        return {"out": ("f16", (c["rows"], c["out"]))}
    if kind == "linear":
        return {"out": (c["dtype"], (c["rows"], c["out"]))}
    if kind == "rows":
        if c["op"] in ("row_sum", "row_max"):
            return {"out": ("f32", (c["rows"],))}
        return {"out": (c["dtype"], (c["rows"], c["width"]))}
    if kind == "view":
        shape, order = _view_shape(c)
        return {"out": (c["dtype"], tuple(shape[i] for i in order))}
    if kind == "reduce":
        if c["op"] == "argmax":
            return {"index": ("u32", (1,))}
        return {"sum": ("f64", (1,)), "max": ("f32", (1,))}
    return {"out": (c["dtype"], (c["count"], c["width"]))}


def prepare(case, seed):
    lib = sdk()
    tensors, views = {}, {}
    dtypes = {v: k for k, v in TORCH.items()}
    for name, value in _inputs(case, seed).items():
        tensors[name] = lib.tensor(dtypes[value.dtype], tuple(value.shape))
        views[name] = _as_torch(tensors[name])
        views[name].copy_(value)
    outputs = {}
    for name, (dtype, shape) in _output_spec(case).items():
        tensors["out_" + name] = lib.tensor(dtype, shape)
        outputs[name] = _as_torch(tensors["out_" + name])
        outputs[name].zero_()
    if case["kind"] == "decoder":      # rotated in place
        outputs["q"], outputs["k"] = views["q"], views["k"]
    state = {"case": case, "t": tensors, "out": outputs}
    if case["kind"] == "view":
        shape, order = _view_shape(case)
        strides = [math.prod(shape[i + 1:]) for i in range(len(shape))]
        state["view"] = TensorView.make([shape[i] for i in order], [strides[i] for i in order])
    # torch fills on its own stream, the library reads on another
    torch.cuda.synchronize()
    return state


def run(state):
    c, t, call = state["case"], state["t"], sdk().call
    kind = c["kind"]
    if kind == "decoder":
        call("tensor_residual_rms_norm_f16", t["x"], t["r"], t["w"], EPS, t["out_sum"], t["out_normed"])
        call("tensor_rope_f16", t["q"], t["k"], c["heads"], c["kv_heads"], c["dim"], THETA, POSITION)
        call("tensor_silu_multiply_f16", t["gate"], t["up"], t["out_act"])
    elif kind == "vision":
        d = c["dtype"]
        call(f"tensor_layer_norm_{d}", t["x"], t["w"], t["b"], EPS, t["out_normed"])
        call(f"tensor_bias_gelu_{d}", t["h"], t["hb"], t["out_act"])
        call("tensor_residual_add_f16" if d == "f16" else "tensor_add_f32", t["x"], t["y"], t["out_sum"])
    elif kind == "attn":
        call(f"tensor_sdpa_device_{c['dtype']}", t["q"], t["k"], t["v"], t.get("mask"),
             c["dim"] ** -0.5, int(c["causal"]), t["out_out"])
    elif kind == "quant":
        call(f"tensor_linear_{c['format']}_f16", t["x"], t["packed"], t["out_out"])
    elif kind == "linear":
        call(f"tensor_linear_{c['dtype']}", t["x"], t["w"], t.get("bias"), t["out_out"])
    elif kind == "rows":
        name = f"tensor_{c['op']}_{c['dtype']}"
        if c["op"] == "softmax":
            call(name, t["x"], 0, t["out_out"])
        elif c["op"] == "rms_norm":
            call(name, t["x"], t["w"], EPS, t["out_out"])
        elif c["op"] == "layer_norm":
            call(name, t["x"], t["w"], t["b"], EPS, t["out_out"])
        else:
            call(name, t["x"], t["out_out"])
    elif kind == "view":
        call(f"tensor_view_add_mul_{c['dtype']}", t["x"], state["view"], t.get("add"), t.get("mul"),
             t["out_out"])
    elif kind == "reduce":
        if c["op"] == "argmax":
            call(f"tensor_argmax_{c['dtype']}", t["x"], t["out_index"])
        else:
            call("tensor_sum_max_f32", t["x"], t["out_sum"], t["out_max"])
    else:
        call(f"tensor_embedding_lookup_{c['dtype']}", t["table"], t["ids"], t["out_out"])
    return state["out"]


# ---- what a pass cannot do without ---------------------------------------------------

def work(case):
    c, kind = case, case["kind"]
    if kind == "decoder":
        t = c["tokens"]
        return {"bytes": 2 * (4 * t * c["hidden"] + c["hidden"] + 2 * t * (c["heads"] + c["kv_heads"]) * c["dim"]
                              + 3 * t * c["inter"]), "flops": 0}
    if kind == "vision":
        t, w, e = c["tokens"], c["width"], SIZE[c["dtype"]]
        return {"bytes": e * (4 * t * w + 2 * w + 2 * t * c["inter"] + c["inter"]), "flops": 0}
    if kind == "attn":
        e, b, ql, kl, d = SIZE[c["dtype"]], c["batch"], c["q_len"], c["kv_len"], c["dim"]
        pairs = ql * kl
        if c["causal"]:      # query i sees keys 0 .. i + max(kl - ql, 0)
            offset = max(kl - ql, 0)
            pairs = sum(min(kl, i + offset + 1) for i in range(ql))
        return {"bytes": e * (2 * b * c["heads"] * ql * d + 2 * b * c["kv_heads"] * kl * d
                              + (ql * kl if c["mask"] else 0)),
                "flops": 4 * b * c["heads"] * pairs * d}
    if kind == "quant":
        return {"bytes": 2 * c["rows"] * (c["in"] + c["out"]) + c["out"] * (c["in"] // 32) * BLOCK[c["format"]],
                "flops": 2 * c["rows"] * c["in"] * c["out"]}
    if kind == "linear":
        e = SIZE[c["dtype"]]
        return {"bytes": e * (c["rows"] * (c["in"] + c["out"]) + c["out"] * c["in"] + (c["out"] if c["bias"] else 0)),
                "flops": 2 * c["rows"] * c["in"] * c["out"]}
    if kind == "rows":
        n, e = c["rows"] * c["width"], SIZE[c["dtype"]]
        reduced = c["op"] in ("row_sum", "row_max")
        return {"bytes": n * e + (4 * c["rows"] if reduced else n * e), "flops": 0}
    if kind == "view":
        return {"bytes": 2 * SIZE[c["dtype"]] * c["a"] * c["b"] * c["c"] * c["d"], "flops": 0}
    if kind == "reduce":
        return {"bytes": SIZE[c["dtype"]] * c["n"], "flops": 0}
    return {"bytes": 2 * SIZE[c["dtype"]] * min(c["count"], c["vocab"]) * c["width"] + 4 * c["count"], "flops": 0}


def tolerance(case):
    kind = case["kind"]
    half = case.get("dtype", "f16") == "f16"
    if kind == "embed" or (kind == "reduce" and case["op"] == "argmax"):
        return "exact"
    if kind == "rows" and case["op"] == "row_max":
        return "exact"
    if kind == "view" and not case["operands"]:
        return "exact"
    # about four times the error against float64 that the library shows
    if kind in ("rows", "vision", "view", "decoder"):
        # f16: one rounding of the result, 2.1e-4; f32: sums and exponentials, 1.2e-7
        return {"rel": 1e-3} if half else {"rel": 1e-6}
    if kind == "reduce":
        return {"rel": 1e-6}    # f32 sums of a lane's values, f64 across lanes
    if kind == "attn":
        # f16: probabilities and outputs rounded to f16, 2.9e-4; f32: the
        # rounding of the scores reaches the probabilities through exp, 3e-7
        return {"rel": 1.2e-3} if half else {"rel": 2e-6}
    # linear, quant: one rounding of the output in f16, 2.1e-4; f32 sums of
    # up to 8000 products, 2.6e-7
    return {"rel": 1e-3} if half else {"rel": 2e-6}


# ---- the same in 64 bits ---------------------------------------------------------------

def _gelu(x):
    y = 0.5 * x * (1 + torch.tanh(0.7978845608028654 * (x + 0.044715 * x ** 3)))
    return torch.where(x >= 5, x, torch.where(x <= -5, torch.zeros_like(x), y))


def _rotate(x):
    """Split-half RoPE of x [tokens, heads, dim] at positions POSITION .."""
    dim = x.shape[-1]
    d = torch.arange(dim // 2, device=x.device, dtype=torch.float64)
    p = torch.arange(x.shape[0], device=x.device, dtype=torch.float64) + POSITION
    angle = p[:, None] / THETA ** (2 * d / dim)[None, :]
    cos, sin = torch.cos(angle)[:, None, :], torch.sin(angle)[:, None, :]
    a, b = x[..., :dim // 2], x[..., dim // 2:]
    return torch.cat([a * cos - b * sin, a * sin + b * cos], dim=-1)


def _attention(c, a):
    q, k, v = a["q"], a["k"], a["v"]
    group = c["heads"] // c["kv_heads"]
    ql, kl = c["q_len"], c["kv_len"]
    bias = a.get("mask", torch.zeros((), device=q.device, dtype=torch.float64))
    if c["causal"]:
        i = torch.arange(ql, device=q.device)[:, None] + max(kl - ql, 0)
        hidden = torch.arange(kl, device=q.device)[None, :] > i
        bias = torch.zeros((ql, kl), device=q.device, dtype=torch.float64) + bias
        bias = bias.masked_fill(hidden, -math.inf)
    out = torch.empty_like(q)
    for b in range(c["batch"]):
        for h in range(c["heads"]):
            s = q[b, h] @ k[b, h // group].t().contiguous() * c["dim"] ** -0.5 + bias
            out[b, h] = torch.softmax(s, dim=-1) @ v[b, h // group]
    return out


def exact(case, seed):
    c, kind = case, case["kind"]
    a = {n: x.double() if x.is_floating_point() else x for n, x in _inputs(case, seed).items()}
    if kind == "decoder":
        # the second step reads the sum as it is stored, in f16
        s = a["x"] + a["r"]
        stored = s.half().double()
        normed = stored * torch.rsqrt(stored.square().mean(-1, keepdim=True) + EPS) * a["w"]
        act = a["gate"] * torch.sigmoid(a["gate"]) * a["up"]
        return {"sum": s, "normed": normed, "act": act, "q": _rotate(a["q"]), "k": _rotate(a["k"])}
    if kind == "vision":
        x = a["x"]
        centred = x - x.mean(-1, keepdim=True)
        normed = centred * torch.rsqrt(centred.square().mean(-1, keepdim=True) + EPS) * a["w"] + a["b"]
        return {"normed": normed, "act": _gelu(a["h"] + a["hb"]), "sum": x + a["y"]}
    if kind == "attn":
        return {"out": _attention(c, a)}
    if kind == "quant":
        packed = a["packed"]
        scale = packed[..., :2].contiguous().view(torch.float16).double()
        if c["format"] == "q8_0":
            q = packed[..., 2:].contiguous().view(torch.int8).double()
        else:
            body = packed[..., 2:]
            q = torch.cat([body & 15, body >> 4], dim=-1).double() - 8
        w = (q * scale).reshape(c["out"], c["in"])
        return {"out": a["x"] @ w.t().contiguous()}
    if kind == "linear":
        y = a["x"] @ a["w"].t().contiguous()
        return {"out": y + a["bias"] if c["bias"] else y}
    if kind == "rows":
        x, op = a["x"], c["op"]
        if op == "softmax":
            return {"out": torch.softmax(x, dim=-1)}
        if op == "row_sum":
            return {"out": x.sum(-1)}
        if op == "row_max":
            return {"out": x.amax(-1)}
        centred = x - x.mean(-1, keepdim=True) if op == "layer_norm" else x
        y = centred * torch.rsqrt(centred.square().mean(-1, keepdim=True) + EPS) * a["w"]
        return {"out": y + a["b"] if op == "layer_norm" else y}
    if kind == "view":
        _, order = _view_shape(c)
        x = a["x"].permute(order)
        return {"out": ((x + a["add"]) * a["mul"] if c["operands"] else x).contiguous()}
    if kind == "reduce":
        if c["op"] == "argmax":
            return {"index": None}
        return {"sum": a["x"].sum().reshape(1), "max": a["x"].max().reshape(1)}
    return {"out": a["table"][a["ids"].long()]}

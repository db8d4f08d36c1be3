"""What a program built on this package has it do, as cases that can be timed.

A case is a dict of plain values.  ``listed()`` gives the ones that are looked
at first, ``draw(rng)`` one more of the same ranges, ``prepare`` what a program
holds before the call (weights quantized at load, activations of the moment),
``run`` one pass through the package's public entry points, ``work`` the bytes
and operations a pass cannot do without and ``tolerance`` how far another
correct implementation of the same precision may be off.

The kinds of case:

* ``token``: one step of text generation -- the projections of some transformer
  layers (q, k, v, o as ``nn.QuantizedLinear``, the gated MLP as ``nn.SwiGLU``)
  for a few sequences.  Attention and norms between them are other code.
* ``product``: ``quantized_matmul`` with one or more weights in turn, from one
  row of x (decode) to thousands (prefill), every width and mode.
* ``qqmm``: ``qqmm``, which quantizes x as well.
* ``experts``: the expert-routed MLP ``nn.SwitchGLU`` on router output.
* ``tune``: forward and backward through a frozen quantized layer.
* ``store``: ``quantize`` a weight and ``dequantize`` it, as loading and
  exporting a model do.

Several weights in a pass stand for the layers of a model: a decode step reads
each of them once, from memory and not from a cache.
"""
from __future__ import annotations

import math
import random

import torch

import mlx_amd
from mlx_amd import nn

DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
SIZE = {"float32": 4, "float16": 2, "bfloat16": 2}
FP_MODES = {"mxfp4": (32, 4), "mxfp8": (32, 8), "nvfp4": (16, 4)}

# (hidden, ffn, kv): widths of dense layers that the benchmark and the tests use
LAYERS = ((4096, 14336, 1024), (4096, 11008, 4096), (3584, 18944, 512), (2048, 8192, 512),
          (5120, 13824, 5120), (8192, 28672, 1024))
# (N, K) of single products, from an attention projection to a vocabulary
PRODUCTS = ((1024, 1024), (1024, 4096), (2048, 2048), (4096, 4096), (14336, 4096), (4096, 14336),
            (11008, 4096), (4096, 11008), (5120, 13824), (18944, 3584), (8192, 8192),
            (32000, 4096), (128256, 4096))
# (hidden, ffn, experts, top)
EXPERTS = ((4096, 14336, 8, 2), (2048, 1408, 64, 6), (1024, 1024, 32, 4))


def listed():
    return [
        # chat with one user: each token reads every weight once
        {"name": "token, 1 sequence", "kind": "token", "rows": 1, "hidden": 4096, "ffn": 14336,
         "kv": 1024, "layers": 4, "group": 64, "bits": 4, "dtype": "bfloat16"},
        # a small server (or speculative decoding) with weights kept at 8 bits
        {"name": "token, 8 sequences, 8-bit", "kind": "token", "rows": 8, "hidden": 3584,
         "ffn": 18944, "kv": 512, "layers": 2, "group": 128, "bits": 8, "dtype": "float16"},
        # the smallest call in use: one row against a small projection, in the default type
        {"name": "small product", "kind": "product", "rows": 1, "n": 1024, "k": 1024,
         "weights": 1, "mode": "affine", "group": 64, "bits": 4, "dtype": "float32"},
        # decode with an odd code width, as mixed-width recipes give some layers
        {"name": "decode, 6-bit", "kind": "product", "rows": 1, "n": 11008, "k": 4096,
         "weights": 8, "mode": "affine", "group": 32, "bits": 6, "dtype": "bfloat16"},
        # continuous batching: some tens of sequences in a decode step
        {"name": "batch of 48", "kind": "product", "rows": 48, "n": 14336, "k": 4096,
         "weights": 8, "mode": "affine", "group": 64, "bits": 4, "dtype": "bfloat16"},
        # a prompt of 2048 tokens
        {"name": "prefill", "kind": "product", "rows": 2048, "n": 14336, "k": 4096,
         "weights": 1, "mode": "affine", "group": 64, "bits": 4, "dtype": "bfloat16"},
        # a shorter, ragged prompt on weights in a floating-point format, down projection
        {"name": "prefill 509, mxfp4", "kind": "product", "rows": 509, "n": 4096, "k": 14336,
         "weights": 1, "mode": "mxfp4", "group": 32, "bits": 4, "dtype": "bfloat16"},
        # both operands in 8 bits
        {"name": "qqmm, mxfp8", "kind": "qqmm", "rows": 2048, "n": 14336, "k": 4096,
         "mode": "mxfp8", "dtype": "bfloat16"},
        # one step of a few sequences through a mixture of experts
        {"name": "experts, 8 tokens", "kind": "experts", "tokens": 8, "hidden": 4096,
         "ffn": 14336, "experts": 8, "top": 2, "group": 64, "bits": 4, "dtype": "bfloat16"},
        # a prompt through the same block
        {"name": "experts, 2048 tokens", "kind": "experts", "tokens": 2048, "hidden": 4096,
         "ffn": 14336, "experts": 8, "top": 2, "group": 64, "bits": 4, "dtype": "bfloat16"},
        # fine-tuning adapters around frozen 4-bit layers
        {"name": "tune", "kind": "tune", "batch": 2, "rows": 512, "n": 14336, "k": 4096,
         "group": 64, "bits": 4, "dtype": "bfloat16"},
        # converting a checkpoint
        {"name": "store", "kind": "store", "n": 14336, "k": 4096, "mode": "affine", "group": 64,
         "bits": 4, "dtype": "bfloat16"},
    ]


def _log_int(rng: random.Random, low: int, high: int) -> int:
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def _ragged(rng: random.Random, n: int) -> int:
    """Outer sizes as they come: mostly whole tiles, sometimes any number."""
    return n if rng.random() < 0.6 else max(64, n - rng.randrange(1, n // 3))


def _inner(rng: random.Random, k: int, step: int) -> int:
    """Inner sizes are whole groups (and multiples of 64, as model widths are)."""
    step = max(step, 64)
    return k if rng.random() < 0.6 else max(step, (k - rng.randrange(1, k // 3)) // step * step)


def _width(rng: random.Random):
    bits = rng.choice((4, 4, 4, 8, 8, 2, 3, 5, 6))
    return bits, rng.choice((32, 64, 64, 128))


def draw(rng):
    kind = rng.choice(("token", "token", "product", "product", "product", "qqmm", "experts",
                       "tune", "store"))
    dtype = rng.choice(("bfloat16", "bfloat16", "float16"))
    most = max(_seconds(c) for c in listed())
    while True:
        if kind == "token":
            hidden, ffn, kv = rng.choice(LAYERS)
            bits, group = _width(rng)
            hidden, ffn = _inner(rng, hidden, 128), _inner(rng, ffn, 128)
            case = {"kind": kind, "rows": _log_int(rng, 1, 16), "hidden": hidden, "ffn": ffn,
                    "kv": min(kv, hidden), "layers": 1, "group": group, "bits": bits,
                    "dtype": dtype}
            case["layers"] = max(1, min(8, round(4e8 / work(case)["bytes"])))
        elif kind == "product":
            n, k = rng.choice(PRODUCTS)
            mode = rng.choice(("affine", "affine", "affine", "mxfp4", "mxfp8", "nvfp4"))
            bits, group = _width(rng)
            group, bits = FP_MODES.get(mode, (group, bits))
            rows = _log_int(rng, 1, 8192)
            if mode == "affine" and rng.random() < 0.2:
                dtype = "float32"
            case = {"kind": kind, "rows": rows, "n": _ragged(rng, n), "k": _inner(rng, k, group),
                    "weights": 1, "mode": mode, "group": group, "bits": bits, "dtype": dtype}
            if rows <= 64:
                case["weights"] = max(1, min(8, round(2e8 / work(case)["bytes"])))
        elif kind == "qqmm":
            n, k = rng.choice(PRODUCTS)
            mode = rng.choice(("mxfp4", "mxfp8", "nvfp4"))
            case = {"kind": kind, "rows": _log_int(rng, 1, 8192), "n": _ragged(rng, n),
                    "k": _inner(rng, k, 128), "mode": mode, "dtype": dtype}
        elif kind == "experts":
            hidden, ffn, experts, top = rng.choice(EXPERTS)
            case = {"kind": kind, "tokens": _log_int(rng, 1, 2048), "hidden": hidden, "ffn": ffn,
                    "experts": experts, "top": top, "group": rng.choice((32, 64, 64, 128)),
                    "bits": rng.choice((4, 4, 8)), "dtype": dtype}
        elif kind == "tune":
            n, k = rng.choice(PRODUCTS[:-2])
            case = {"kind": kind, "batch": rng.randrange(1, 5), "rows": _log_int(rng, 16, 1024),
                    "n": _inner(rng, n, 128), "k": _inner(rng, k, 128),
                    "group": rng.choice((32, 64, 64, 128)), "bits": rng.choice((4, 4, 8)),
                    "dtype": dtype}
        else:
            n, k = rng.choice(PRODUCTS)
            mode = rng.choice(("affine", "affine", "affine", "mxfp4", "mxfp8", "nvfp4"))
            bits, group = _width(rng)
            group, bits = FP_MODES.get(mode, (group, bits))
            case = {"kind": kind, "n": _ragged(rng, n), "k": _inner(rng, k, group), "mode": mode,
                    "group": group, "bits": bits,
                    "dtype": rng.choice(("float32", "float16", "bfloat16"))}
        if _seconds(case) <= most:
            return case


def _seconds(case) -> float:
    """A case's cost, roughly, so that none is drawn that is beyond the listed ones."""
    w = work(case)
    slow = 5.0 if case["dtype"] == "float32" else 1.0  # float32 products are three 16-bit ones
    return w["bytes"] / 5e12 + slow * w["flops"] / 1e15


# ---------------------------------------------------------------- preparation
class _Source:
    """Seeded values on the GPU."""

    def __init__(self, seed: int):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def activations(self, *shape, dtype):
        # unit variance, with the few large channels that hidden states have
        x = torch.randn(shape, generator=self.g, device="cuda")
        wide = torch.rand(shape[-1], generator=self.g, device="cuda") < 0.01
        return (x * torch.where(wide, 6.0, 1.0)).to(dtype)

    def weight(self, *shape, dtype):
        std = 1.0 / math.sqrt(shape[-1])
        return (torch.randn(shape, generator=self.g, device="cuda") * std).to(dtype)

    def experts_of(self, tokens, experts, top):
        # router logits with some experts more popular than others
        logits = torch.randn((tokens, experts), generator=self.g, device="cuda")
        logits += 0.5 * torch.randn((experts,), generator=self.g, device="cuda")
        return torch.topk(logits, top, dim=-1).indices


def _linear(src, n, k, group, bits, dtype):
    layer = nn.QuantizedLinear(k, n, False, group, bits, dtype=dtype)
    layer.weight, layer.scales, layer.biases = mlx_amd.quantize(
        src.weight(n, k, dtype=dtype), group, bits)
    return layer


def prepare(case, seed):
    src = _Source(seed)
    dtype = DTYPES[case["dtype"]]
    kind = case["kind"]
    if kind == "token":
        g, b, h, f = case["group"], case["bits"], case["hidden"], case["ffn"]
        layers = []
        for _ in range(case["layers"]):
            mlp = nn.SwiGLU(h, f, group_size=g, bits=b, dtype=dtype)
            mlp.gate_proj = _linear(src, f, h, g, b, dtype)
            mlp.up_proj = _linear(src, f, h, g, b, dtype)
            mlp.down_proj = _linear(src, h, f, g, b, dtype)
            layers.append({
                "q": _linear(src, h, h, g, b, dtype), "k": _linear(src, case["kv"], h, g, b, dtype),
                "v": _linear(src, case["kv"], h, g, b, dtype), "o": _linear(src, h, h, g, b, dtype),
                "mlp": mlp,
                # what the norms and the attention of the layer give it
                "x": src.activations(case["rows"], 1, h, dtype=dtype),
                "attended": src.activations(case["rows"], 1, h, dtype=dtype),
                "normed": src.activations(case["rows"], 1, h, dtype=dtype),
            })
        return {"kind": kind, "layers": layers}
    if kind == "product":
        q = [mlx_amd.quantize(src.weight(case["n"], case["k"], dtype=dtype), case["group"],
                              case["bits"], case["mode"]) for _ in range(case["weights"])]
        x = [src.activations(case["rows"], case["k"], dtype=dtype) for _ in q]
        return {"kind": kind, "x": x, "q": q, "group": case["group"], "bits": case["bits"],
                "mode": case["mode"]}
    if kind == "qqmm":
        q = mlx_amd.quantize(src.weight(case["n"], case["k"], dtype=dtype), mode=case["mode"])
        return {"kind": kind, "x": src.activations(case["rows"], case["k"], dtype=dtype), "q": q,
                "mode": case["mode"]}
    if kind == "experts":
        g, b, h, f, e = (case[k] for k in ("group", "bits", "hidden", "ffn", "experts"))
        block = nn.SwitchGLU(h, f, e, group_size=g, bits=b, dtype=dtype)
        for layer, n, k in ((block.gate_proj, f, h), (block.up_proj, f, h), (block.down_proj, h, f)):
            layer.weight, layer.scales, layer.biases = mlx_amd.quantize(
                src.weight(e, n, k, dtype=dtype), g, b)
        return {"kind": kind, "block": block,
                "x": src.activations(case["tokens"], h, dtype=dtype),
                "indices": src.experts_of(case["tokens"], e, case["top"])}
    if kind == "tune":
        q = mlx_amd.quantize(src.weight(case["n"], case["k"], dtype=dtype), case["group"],
                             case["bits"])
        x = src.activations(case["batch"], case["rows"], case["k"], dtype=dtype)
        dy = torch.randn((case["batch"], case["rows"], case["n"]), generator=src.g, device="cuda")
        return {"kind": kind, "x": x.requires_grad_(), "q": q, "dy": dy.to(dtype),
                "group": case["group"], "bits": case["bits"]}
    return {"kind": kind, "w": src.weight(case["n"], case["k"], dtype=dtype),
            "group": case["group"], "bits": case["bits"], "mode": case["mode"], "dtype": dtype}


# ---------------------------------------------------------------- one pass
def run(s):
    kind = s["kind"]
    if kind == "token":
        out = []
        with torch.no_grad():
            for layer in s["layers"]:
                x = layer["x"]
                out.append((layer["q"](x), layer["k"](x), layer["v"](x),
                            layer["o"](layer["attended"]), layer["mlp"](layer["normed"])))
        return out
    if kind == "product":
        return [mlx_amd.quantized_matmul(x, *q, group_size=s["group"], bits=s["bits"],
                                         mode=s["mode"]) for x, q in zip(s["x"], s["q"])]
    if kind == "qqmm":
        return mlx_amd.qqmm(s["x"], *s["q"], mode=s["mode"])
    if kind == "experts":
        with torch.no_grad():
            return s["block"](s["x"], s["indices"])
    if kind == "tune":
        y = mlx_amd.quantized_matmul(s["x"], *s["q"], group_size=s["group"], bits=s["bits"])
        (dx,) = torch.autograd.grad(y, s["x"], s["dy"])
        return y.detach(), dx
    q = mlx_amd.quantize(s["w"], s["group"], s["bits"], s["mode"])
    w = mlx_amd.dequantize(*q, group_size=s["group"], bits=s["bits"], mode=s["mode"],
                           dtype=s["dtype"])
    # (torch cannot index uint32 tensors: the packed words are handed on as int32)
    return (q[0].view(torch.int32), *q[1:], w)


# ---------------------------------------------------------------- accounts
def _packed(n, k, group, bits, mode, size):
    """Bytes of a quantized [n, k] matrix."""
    per_group = 1 if mode in FP_MODES else 2 * size
    return n * k * bits // 8 + n * (k // group) * per_group


def work(case):
    size, kind = SIZE[case["dtype"]], case["kind"]
    if kind == "token":
        h, f, kv, m = case["hidden"], case["ffn"], case["kv"], case["rows"]
        total = {"bytes": 0, "flops": 0}
        for n, k in ((h, h), (kv, h), (kv, h), (h, h), (f, h), (f, h), (h, f)):
            total["bytes"] += _packed(n, k, case["group"], case["bits"], "affine", size)
            total["flops"] += 2 * m * n * k
        total["bytes"] += m * size * (3 * h + 3 * h + 2 * kv)  # three inputs; q, k, v, o, mlp
        return {k: v * case["layers"] for k, v in total.items()}
    if kind == "product":
        m, n, k = case["rows"], case["n"], case["k"]
        one = _packed(n, k, case["group"], case["bits"], case["mode"], size) + m * (n + k) * size
        return {"bytes": case["weights"] * one, "flops": case["weights"] * 2 * m * n * k}
    if kind == "qqmm":
        m, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": _packed(n, k, *FP_MODES[case["mode"]], case["mode"], size)
                + m * (n + k) * size, "flops": 2 * m * n * k}
    if kind == "experts":
        t, h, f, e, top = (case[k] for k in ("tokens", "hidden", "ffn", "experts", "top"))
        used = e * (1 - (1 - top / e) ** t)  # experts that some token is sent to, on average
        one = 2 * _packed(f, h, case["group"], case["bits"], "affine", size) \
            + _packed(h, f, case["group"], case["bits"], "affine", size)
        return {"bytes": used * one + t * h * size + t * top * (h * size + 8),
                "flops": t * top * 2 * 3 * h * f}
    if kind == "tune":
        m, n, k = case["batch"] * case["rows"], case["n"], case["k"]
        return {"bytes": _packed(n, k, case["group"], case["bits"], "affine", size)
                + 2 * m * (n + k) * size, "flops": 2 * 2 * m * n * k}
    n, k = case["n"], case["k"]
    packed = _packed(n, k, case["group"], case["bits"], case["mode"], size)
    return {"bytes": n * k * size + packed + n * k * size, "flops": 0}


def tolerance(case):
    if case["kind"] == "store":
        return "exact"  # packing and unpacking are defined to the bit
    # dequantized weights and results are rounded to the type, sums are kept in 32 bits;
    # float32 products may be formed from three of 16-bit halves (2**-17 each)
    return {"float32": {"rel": 2e-5, "max": 5e-4}, "float16": {"rel": 2e-3, "max": 3e-2},
            "bfloat16": {"rel": 1e-2, "max": 2e-1}}[case["dtype"]]

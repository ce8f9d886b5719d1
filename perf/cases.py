"""The calls whose speed is measured: quantized linear layers from one decoded
token to long prompts, the block Programs built from them, packing and
unpacking of weights, and the other ops of a decode step.

Weights are N(0, 0.02) and activations N(0, 1) (the distributions of the
benchmark), made on the GPU from the seed; weights are packed here with plain
torch arithmetic in the documented format, so that ``exact`` needs nothing
of the package. Matrix products write into an output that the caller keeps
(``quantized_matmul_into``), as a serving loop does; Programs and the other
ops return new tensors.
"""
from __future__ import annotations

import math
import random

import torch

import affon_amd as A
from affon_amd import _native

_DTYPE = {"f32": torch.float32, "bf16": torch.bfloat16, "u32": torch.int32, "i64": torch.int64}
_BYTES = {"f32": 4, "bf16": 2}
_SESSION = None


def _session():
    """One Session for the process, as a program that serves one GPU keeps."""
    global _SESSION
    if _SESSION is None:
        _SESSION = A.Session("rocm")
    return _SESSION


def listed():
    return [
        # One generated token through the widest layer of a Llama-8B-shaped
        # block: the benchmark's headline decode.
        {"name": "decode_m1_4bit", "kind": "matmul", "M": 1, "N": 14336, "K": 4096, "bits": 4, "group": 64,
         "x": "bf16", "param": "bf16", "policy": "backend_equivalent"},
        # The reference's own published workload (8-bit, 2048 x 1024, f32
        # activations) at its smallest: one row, where launches count.
        {"name": "decode_m1_8bit_f32", "kind": "matmul", "M": 1, "N": 2048, "K": 1024, "bits": 8, "group": 64,
         "x": "f32", "param": "f32", "policy": "backend_equivalent"},
        # The same workload at its largest batch.
        {"name": "batch_m128_8bit_f32", "kind": "matmul", "M": 128, "N": 2048, "K": 1024, "bits": 8, "group": 64,
         "x": "f32", "param": "f32", "policy": "backend_equivalent"},
        # A prompt of 512 tokens through the down projection.
        {"name": "prefill_m512_4bit", "kind": "matmul", "M": 512, "N": 4096, "K": 14336, "bits": 4, "group": 64,
         "x": "bf16", "param": "bf16", "policy": "backend_equivalent"},
        # The largest: 2048 rows of a 70B-shaped layer at groups of 32, with
        # the policy that admits rounded weights.
        {"name": "prefill_m2048_4bit_g32", "kind": "matmul", "M": 2048, "N": 28672, "K": 8192, "bits": 4, "group": 32,
         "x": "bf16", "param": "bf16", "policy": "approximate"},
        # A short prompt through a down projection of inner width 11008 cut
        # over eight GPUs: K = 1376, a whole number of groups of 32 and of
        # nothing larger.
        {"name": "ragged_m100_4bit_g32", "kind": "matmul", "M": 100, "N": 4096, "K": 1376, "bits": 4, "group": 32,
         "x": "bf16", "param": "bf16", "policy": "backend_equivalent"},
        # Query, key and value projections with output biases of one token.
        {"name": "attention_m1_4bit", "kind": "attention", "M": 1, "width": 4096, "kv": 1024, "bits": 4, "group": 64,
         "x": "bf16", "param": "bf16"},
        # The feed-forward part of a block for a decode batch of 16 (8-bit
        # weights) and for a prompt of 512: gate and up read the bf16
        # activations, down reads their f32 product.
        {"name": "feed_forward_m16_8bit", "kind": "feed_forward", "M": 16, "width": 4096, "inner": 14336, "bits": 8,
         "group": 64, "x": "bf16", "param": "bf16"},
        {"name": "feed_forward_m512_4bit", "kind": "feed_forward", "M": 512, "width": 4096, "inner": 14336, "bits": 4,
         "group": 64, "x": "bf16", "param": "bf16"},
        # Packing a checkpoint's f32 matrix, and expanding a packed one.
        {"name": "quantize_f32_4bit", "kind": "quantize", "N": 14336, "K": 4096, "bits": 4, "group": 64, "w": "f32",
         "param": "bf16"},
        {"name": "dequantize_bf16_4bit", "kind": "dequantize", "N": 14336, "K": 4096, "bits": 4, "group": 64,
         "w": "bf16", "param": "bf16"},
        # The other ops of a decode step of 32 sequences: token embeddings
        # (index_select), rms_norm, and softmax over the vocabulary.
        {"name": "row_ops_m32", "kind": "row_ops", "M": 32, "width": 4096, "vocab": 128256, "x": "f32"},
    ]


def _log(rng, low, high, step=1):
    """A multiple of step from low to high, spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    return max(low, min(high, int(round(v / step)) * step))


def draw(rng: random.Random):
    kind = rng.choice(["matmul"] * 8 + ["attention", "feed_forward", "feed_forward", "quantize", "dequantize",
                                        "row_ops"])
    if kind == "row_ops":
        vocab = _log(rng, 1000, 128256)
        return {"kind": kind, "M": _log(rng, 1, 512), "width": _log(rng, 512, 4096), "vocab": vocab,
                "x": rng.choice(["f32", "bf16"])}
    bits, group = rng.choice([2, 4, 4, 4, 8, 8]), rng.choice([32, 64, 64, 128])
    if kind in ("quantize", "dequantize"):
        return {"kind": kind, "N": _log(rng, 256, 14336), "K": _log(rng, 1024, 8192, 128), "bits": bits,
                "group": group, "w": rng.choice(["f32", "bf16"]), "param": rng.choice(["f32", "bf16"])}
    if kind == "attention":
        heads, share = rng.choice([8, 16, 32, 64]), rng.choice([1, 4, 8])
        return {"kind": kind, "M": _log(rng, 1, 512), "width": 128 * heads, "kv": 128 * heads // share, "bits": bits,
                "group": group, "x": "bf16", "param": rng.choice(["bf16", "bf16", "f32"])}
    if kind == "feed_forward":
        width = 256 * rng.randint(4, 16)
        return {"kind": kind, "M": _log(rng, 1, 512), "width": width, "inner": 128 * int(width * 3.5 / 128),
                "bits": bits, "group": group, "x": "bf16", "param": rng.choice(["bf16", "bf16", "f32"])}
    x = rng.choice(["bf16", "bf16", "bf16", "f32"])
    # Layer widths are mostly whole multiples of 256; shards and odd models
    # leave whole groups only.
    step = rng.choice([256, 256, group])
    case = {"kind": kind, "M": _log(rng, 1, 2048), "N": _log(rng, 256, 28672), "K": _log(rng, 1024, 14336, step),
            "bits": bits, "group": group, "x": x,
            "param": rng.choice([x, "bf16"]) if x == "f32" else rng.choice(["bf16", "bf16", "f32"]),
            "policy": rng.choice(["backend_equivalent", "backend_equivalent", "backend_equivalent", "approximate"])}
    most = 512 * 4096 * 14336  # multiply-adds
    while case["M"] * case["N"] * case["K"] > most:
        case["M"] = max(1, case["M"] * 3 // 4)
    return case


# ---- inputs ----

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(g, shape, std=1.0, dtype="f32"):
    return (torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std).to(_DTYPE[dtype])


def _packed(g, N, K, bits, group, param):
    """Packed words [N, K*bits/32] (int32 bits), scales and biases of an
    N(0, 0.02) matrix: per group scale = (max - min) / (2^bits - 1), bias = min."""
    words = torch.empty((N, K * bits // 32), device="cuda", dtype=torch.int32)
    scales = torch.empty((N, K // group), device="cuda", dtype=_DTYPE[param])
    biases = torch.empty_like(scales)
    top, per = (1 << bits) - 1, 32 // bits
    shift = (torch.arange(per, device="cuda") * bits).to(torch.int32)
    rows = max(1, (1 << 26) // K)
    for n in range(0, N, rows):
        w = _normal(g, (min(rows, N - n), K // group, group), 0.02)
        low = w.amin(-1)
        s, b = ((w.amax(-1) - low) / top).to(_DTYPE[param]), low.to(_DTYPE[param])
        q = ((w - b.float()[..., None]) / s.float()[..., None]).round_().clamp_(0, top)
        q = q.to(torch.int32).reshape(w.shape[0], K // per, per)
        words[n:n + rows] = (q << shift).sum(-1, dtype=torch.int32)
        scales[n:n + rows], biases[n:n + rows] = s, b
    return words, scales, biases


def _dense64(words, scales, biases, bits, group):
    """The matrix that packed weights stand for, in 64 bits."""
    N = words.shape[0]
    shift = (torch.arange(32 // bits, device="cuda") * bits).to(torch.int32)
    q = ((words[..., None] >> shift) & ((1 << bits) - 1)).reshape(N, -1, group).to(torch.float64)
    return (q * scales.double()[..., None] + biases.double()[..., None]).reshape(N, -1)


def _upload(t):
    """A Session tensor with a torch tensor's values."""
    name = {v: k for k, v in _DTYPE.items()}[t.dtype]
    out = _session().empty(name, tuple(t.shape))
    t = t.contiguous()
    torch.cuda.synchronize()
    _native.check(_native.load().affon_rocm_memcpy_d2d(_session()._handle, out.data_ptr, t.data_ptr(),
                                                       t.numel() * t.element_size()), "copy")
    return out


class _Interface:
    """A Session tensor as torch can look at it, without a copy."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.__cuda_array_interface__ = {
            "shape": tensor.shape, "typestr": {"f32": "<f4", "bf16": "<i2", "u32": "<i4", "i64": "<i8"}[tensor.dtype],
            "data": (tensor.data_ptr, False), "version": 2, "strides": None}


def _look(tensor):
    t = torch.as_tensor(_Interface(tensor), device="cuda")
    return t.view(torch.bfloat16) if tensor.dtype == "bf16" else t


_FEED = (("gate", "inner", "width"), ("up", "inner", "width"), ("down", "width", "inner"))


def _inputs(case, seed):
    """The case's inputs as torch tensors."""
    g, kind = _generator(seed), case["kind"]
    if kind == "matmul":
        x = _normal(g, (case["M"], case["K"]), 1.0, case["x"])
        return x, _packed(g, case["N"], case["K"], case["bits"], case["group"], case["param"])
    if kind == "attention":
        x = _normal(g, (case["M"], case["width"]), 1.0, case["x"])
        outs = (("query", case["width"]), ("key", case["kv"]), ("value", case["kv"]))
        return x, {n: (_packed(g, N, case["width"], case["bits"], case["group"], case["param"]),
                       _normal(g, (N,), 0.1, case["param"])) for n, N in outs}
    if kind == "feed_forward":
        x = _normal(g, (case["M"], case["width"]), 1.0, case["x"])
        return x, {n: _packed(g, case[o], case[i], case["bits"], case["group"], case["param"]) for n, o, i in _FEED}
    if kind == "quantize":
        return _normal(g, (case["N"], case["K"]), 0.02, case["w"])
    if kind == "dequantize":
        return _packed(g, case["N"], case["K"], case["bits"], case["group"], case["param"])
    table = _normal(g, (case["vocab"], case["width"]), 0.02, case["x"])
    index = torch.randint(0, case["vocab"], (case["M"],), generator=g, device="cuda")
    index[case["M"] // 2 + 1:case["M"] // 2 + 2] = -1  # a padding token among them: selects zeros
    return (table, index, _normal(g, (case["M"], case["width"]), 1.0, case["x"]),
            _normal(g, (case["M"], case["vocab"]), 4.0, case["x"]))


def _block(case, layers, biases):
    """A decoder block with these projections (the other ones share them)."""
    from affon_amd.checkpoint import QuantizedLinear
    from affon_amd.decoder import PROJECTIONS, DecoderShape, QuantizedDecoderBlock

    if case["kind"] == "attention":
        shape = DecoderShape(case["width"], case["width"], case["width"] // 128, case["kv"] // 128)
    else:
        shape = DecoderShape(case["width"], case["inner"], case["width"] // 128, case["width"] // 128)
    linear = {}
    for name, _, _, _ in PROJECTIONS:
        out_features, in_features = shape.features(name)
        parts = layers.get(name)
        if parts is None:
            parts = (_session().empty("u32", (out_features, in_features * case["bits"] // 32)),
                     _session().empty(case["param"], (out_features, in_features // case["group"])),
                     _session().empty(case["param"], (out_features, in_features // case["group"])))
        linear[name] = QuantizedLinear(name, *parts, bits=case["bits"], group_size=case["group"])
    return QuantizedDecoderBlock(shape, linear, biases)


def prepare(case, seed):
    inputs, kind = _inputs(case, seed), case["kind"]
    if kind == "matmul":
        out = _session().empty("f32", (case["M"], case["N"]))
        return {"kind": kind, "args": (out, _upload(inputs[0]), *map(_upload, inputs[1])), "out": _look(out),
                "options": {"bits": case["bits"], "group_size": case["group"], "policy": case["policy"]}}
    if kind == "attention":
        layers = {n: tuple(map(_upload, w)) for n, (w, _) in inputs[1].items()}
        block = _block(case, layers, {n: _upload(b) for n, (_, b) in inputs[1].items()})
        return {"kind": kind, "block": block, "x": _upload(inputs[0])}
    if kind == "feed_forward":
        block = _block(case, {n: tuple(map(_upload, w)) for n, w in inputs[1].items()}, {})
        return {"kind": kind, "block": block, "x": _upload(inputs[0])}
    if kind == "quantize":
        return {"kind": kind, "w": _upload(inputs), "options": {"bits": case["bits"], "group_size": case["group"],
                                                                "param_dtype": case["param"]}}
    if kind == "dequantize":
        return {"kind": kind, "w": tuple(map(_upload, inputs)),
                "options": {"bits": case["bits"], "group_size": case["group"], "dtype": case["w"]}}
    return {"kind": kind, "parts": tuple(map(_upload, inputs))}


def run(state):
    kind = state["kind"]
    if kind == "matmul":
        A.quantized_matmul_into(*state["args"], **state["options"])
        return state["out"]
    if kind == "attention":
        return [_look(t) for t in state["block"].attention(state["x"])]
    if kind == "feed_forward":
        return _look(state["block"].feed_forward(state["x"]))
    if kind == "quantize":
        return [_look(t) for t in A.quantize(state["w"], **state["options"])]
    if kind == "dequantize":
        return _look(A.dequantize(*state["w"], **state["options"]))
    table, index, hidden, logits = state["parts"]
    return [_look(A.index_select(table, 0, index)), _look(A.rms_norm(hidden, -1)), _look(A.softmax(logits, -1))]


# ---- what is measured against ----

def _weight_bytes(N, K, case):
    return N * K * case["bits"] // 8 + 2 * N * (K // case["group"]) * _BYTES[case["param"]]


def work(case):
    kind = case["kind"]
    if kind == "matmul":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": M * K * _BYTES[case["x"]] + _weight_bytes(N, K, case) + 4 * M * N, "flops": 2 * M * N * K}
    if kind == "attention":
        M, K, N = case["M"], case["width"], case["width"] + 2 * case["kv"]
        return {"bytes": M * K * _BYTES[case["x"]] + _weight_bytes(N, K, case) + N * _BYTES[case["param"]] + 4 * M * N,
                "flops": 2 * M * N * K}
    if kind == "feed_forward":
        M, K, N = case["M"], case["width"], case["inner"]
        return {"bytes": M * K * _BYTES[case["x"]] + 2 * _weight_bytes(N, K, case) + _weight_bytes(K, N, case) +
                4 * M * K, "flops": 6 * M * N * K}
    if kind in ("quantize", "dequantize"):
        N, K = case["N"], case["K"]
        return {"bytes": N * K * _BYTES[case["w"]] + _weight_bytes(N, K, case), "flops": 2 * N * K}
    M, width, vocab = case["M"], case["width"], case["vocab"]
    return {"bytes": (4 * M * width + 2 * M * vocab) * _BYTES[case["x"]] + 8 * M, "flops": 3 * M * (width + vocab)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("quantize", "dequantize"):
        return "exact"
    if kind == "row_ops":
        # f32: the sum over a vocabulary row and expf, measured 1.9e-6 off 64
        # bits; bf16: one rounding of each result.
        return {"rel": 8e-6 if case["x"] == "f32" else 8e-3}
    if case.get("policy") == "approximate":
        # Decoded weights rounded to bf16 where the rounded class takes the
        # shape: measured 1.5e-3 off 64 bits.
        return {"rel": 6e-3}
    # f32 sums in any order: measured up to 7e-7 off 64 bits.
    return {"rel": 5e-6}


def exact(case, seed):
    inputs, kind = _inputs(case, seed), case["kind"]
    if kind == "quantize":
        w = inputs.double().reshape(case["N"], -1, case["group"])
        low = w.amin(-1)
        return [None, (w.amax(-1) - low) / ((1 << case["bits"]) - 1), low]
    if kind == "dequantize":
        return _dense64(*inputs, case["bits"], case["group"])
    if kind == "row_ops":
        table, index, hidden, logits = (t.double() if t.is_floating_point() else t for t in inputs)
        rows = torch.where((index >= 0)[:, None], table[index.clamp(min=0)], 0.0)
        return [rows, hidden / (hidden.square().mean(-1, keepdim=True) + 1e-5).sqrt(), torch.softmax(logits, -1)]
    bits, group = case["bits"], case["group"]
    x = inputs[0].double()
    if kind == "matmul":
        return x @ _dense64(*inputs[1], bits, group).T.contiguous()
    if kind == "attention":
        return [x @ _dense64(*w, bits, group).T.contiguous() + b.double() for w, b in inputs[1].values()]
    gate, up, down = (_dense64(*inputs[1][n], bits, group).T.contiguous() for n in ("gate", "up", "down"))
    return (torch.nn.functional.silu(x @ gate) * (x @ up)) @ down

"""The work this framework is used for, as cases to time: BSI-linear layers from one token to thousands, dots on prebuilt
operands, the quantisation of weight matrices, query batches encoded as EWAH streams, whole decoder stacks, and the
reference's scalar entry point on decimal slices.

Every case goes through the package's public entry points in its default configuration (queries 7 bits with chunk
scales, keys 6 bits, two decimal places).  ``listed()`` holds representative sizes, ``draw(rng)`` gives more of the
same ranges."""
import math

import torch
import torch.nn as nn
import torch.nn.functional as F

from bsipytorch_amd import bsi_ops
from bsipytorch_amd.linear import BSIQuantizedLinear, quantize_model_bsi

DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
DECIMALS, THRESHOLD = 2, 0.5
MOST_MACS = 4096 * 4096 * 16384  # the largest listed layer
MOST_WEIGHTS = 16384 * 4096      # the largest listed weight matrix


def listed():
    return [
        # one token through an attention projection of the smallest model: latency and launches
        {"name": "linear_1x768x768", "kind": "linear", "rows": 1, "d": 768, "out": 768, "dtype": "float32", "bias": True},
        # one token through the widest layer: the packed keys are streamed once
        {"name": "linear_1x4096x16384_f16", "kind": "linear", "rows": 1, "d": 4096, "out": 16384, "dtype": "float16", "bias": True},
        # a batch of 16 sequences decoding together
        {"name": "linear_16x4096x4096_bf16", "kind": "linear", "rows": 16, "d": 4096, "out": 4096, "dtype": "bfloat16", "bias": True},
        # a short prompt through a width that is not a multiple of 256: row scales instead of chunk scales
        {"name": "linear_77x1600x4800", "kind": "linear", "rows": 77, "d": 1600, "out": 4800, "dtype": "float32", "bias": True},
        # a prompt of an odd length in half precision
        {"name": "linear_333x2048x2048_f16", "kind": "linear", "rows": 333, "d": 2048, "out": 2048, "dtype": "float16", "bias": True},
        # the FC1 shape of the benchmark, query build included
        {"name": "linear_512x2048x8192", "kind": "linear", "rows": 512, "d": 2048, "out": 8192, "dtype": "float32", "bias": True},
        # many prompts prefilled together through the widest layer
        {"name": "linear_4096x4096x16384_bf16", "kind": "linear", "rows": 4096, "d": 4096, "out": 16384, "dtype": "bfloat16", "bias": False},
        # the FC2 shape of the benchmark on prebuilt operands: activations behind a ReLU
        {"name": "dot_512x8192x2048_relu", "kind": "dot", "rows": 512, "d": 8192, "out": 2048, "dtype": "float32", "relu": True},
        # quantising the weights of the widest layer
        {"name": "keys_16384x4096", "kind": "keys", "d": 4096, "out": 16384, "dtype": "float32"},
        # a query batch kept as EWAH streams, and its dot
        {"name": "hybrid_64x2048x2048_relu", "kind": "hybrid", "rows": 64, "d": 2048, "out": 2048, "dtype": "float32", "relu": True},
        # one token through a stack of decoder layers, eager
        {"name": "decoder_12x768_1", "kind": "decoder", "rows": 1, "layers": 12, "d": 768, "heads": 12, "dtype": "float32"},
        # the scalar entry point: one vector, quantised in decimal mode, against prebuilt keys
        {"name": "scalar_1024x2048", "kind": "scalar", "d": 2048, "out": 1024, "dtype": "float32"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A layer width: mostly multiples of 256 or 64, as models have them, sometimes odd."""
    n, p = _log(rng, lo, hi), rng.random()
    step = 256 if p < 0.65 else (64 if p < 0.9 else 1)
    return min(hi, max(lo, (n + step // 2) // step * step))


def draw(rng):
    kind = rng.choice(["linear"] * 6 + ["dot", "keys", "hybrid", "decoder", "scalar", "dot"])
    dtype = rng.choice(["float32", "float16", "bfloat16"])
    d, out = _width(rng, 256, 8192), _width(rng, 256, 16384)
    out = min(out, MOST_WEIGHTS // d)
    if kind == "keys":
        return {"kind": kind, "d": d, "out": out, "dtype": dtype}
    if kind == "scalar":
        return {"kind": kind, "d": min(d, 4096), "out": min(out, 4096), "dtype": "float32"}
    if kind == "decoder":
        heads = rng.choice([4, 8, 12, 16])
        return {"kind": kind, "rows": _log(rng, 1, 512), "layers": rng.randint(2, 12), "d": heads * 64, "heads": heads, "dtype": "float32"}
    if kind == "hybrid":
        return {"kind": kind, "rows": _log(rng, 1, 512), "d": d, "out": min(out, 8192), "dtype": dtype, "relu": rng.random() < 0.5}
    rows = max(1, min(_log(rng, 1, 4096), MOST_MACS // (d * out)))
    if kind == "dot":
        return {"kind": kind, "rows": rows, "d": d, "out": out, "dtype": dtype, "relu": rng.random() < 0.5}
    return {"kind": kind, "rows": rows, "d": d, "out": out, "dtype": dtype, "bias": rng.random() < 0.7}


class Attention(nn.Module):
    def __init__(self, d, heads):
        super().__init__()
        self.heads = heads
        self.q_proj, self.k_proj, self.v_proj, self.out_proj = (nn.Linear(d, d) for _ in range(4))

    def forward(self, x):
        t, d = x.shape
        q, k, v = (p(x).view(t, self.heads, d // self.heads).transpose(0, 1) for p in (self.q_proj, self.k_proj, self.v_proj))
        a = F.scaled_dot_product_attention(q[None], k[None], v[None], is_causal=True)[0]
        return self.out_proj(a.transpose(0, 1).reshape(t, d))


class DecoderLayer(nn.Module):
    def __init__(self, d, heads):
        super().__init__()
        self.self_attn, self.self_attn_layer_norm = Attention(d, heads), nn.LayerNorm(d)
        self.fc1, self.fc2, self.final_layer_norm = nn.Linear(d, 4 * d), nn.Linear(4 * d, d), nn.LayerNorm(d)

    def forward(self, x):
        x = x + self.self_attn(self.self_attn_layer_norm(x))
        return x + self.fc2(F.relu(self.fc1(self.final_layer_norm(x))))


def _weights(gen, out, d, dtype):
    return (torch.randn(out, d, generator=gen, device="cuda") * 0.02).to(dtype)


def _activations(gen, rows, d, dtype, relu=False):
    """N(0, 1) with one column in a thousand twenty times as large, as transformer activations have them."""
    x = torch.randn(rows, d, generator=gen, device="cuda")
    x[:, torch.rand(d, generator=gen, device="cuda") < 0.001] *= 20.0
    return (torch.relu(x) if relu else x).to(dtype)


@torch.no_grad()
def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind, d, dtype = case["kind"], case["d"], DTYPES[case["dtype"]]
    if kind == "decoder":
        with torch.device("cuda"):
            model = nn.Sequential(*(DecoderLayer(d, case["heads"]) for _ in range(case["layers"])))
        for name, p in model.named_parameters():
            if p.dim() == 2 or (name.endswith("bias") and "norm" not in name):
                p.normal_(0.0, 0.02, generator=gen)
        model = quantize_model_bsi(model.eval(), DECIMALS, compress_threshold=THRESHOLD, verbose=False)
        return {"kind": kind, "model": model, "x": torch.randn(case["rows"], d, generator=gen, device="cuda")}
    if kind == "keys":
        return {"kind": kind, "weights": _weights(gen, case["out"], d, dtype)}
    weights = _weights(gen, case["out"], d, dtype)
    if kind == "scalar":
        keys = bsi_ops.build_bsi_keys(weights, DECIMALS, THRESHOLD)[0]
        return {"kind": kind, "keys": keys, "x": _activations(gen, 1, d, dtype)[0]}
    x = _activations(gen, case["rows"], d, dtype, case.get("relu", False))
    if kind == "linear":
        dense = nn.Linear(d, case["out"], bias=case["bias"], device="meta")
        dense.weight = nn.Parameter(weights, requires_grad=False)
        if case["bias"]:
            dense.bias = nn.Parameter((torch.randn(case["out"], generator=gen, device="cuda") * 0.1).to(dtype), requires_grad=False)
        return {"kind": kind, "layer": BSIQuantizedLinear(dense, DECIMALS, THRESHOLD), "x": x}
    keys = bsi_ops.build_bsi_keys_cuda(weights, DECIMALS, THRESHOLD)[0]
    if kind == "dot":
        return {"kind": kind, "keys": keys, "queries": bsi_ops.build_bsi_queries_cuda_batch_packed(x, DECIMALS, THRESHOLD)}
    return {"kind": kind, "keys": keys, "x": x}


@torch.no_grad()
def run(state):
    kind = state["kind"]
    if kind == "linear":
        return state["layer"](state["x"])
    if kind == "decoder":
        return state["model"](state["x"])
    if kind == "dot":
        return bsi_ops.batch_dot_product_multiquery_cuda_batch_caps(state["queries"], state["keys"])[0]
    if kind == "keys":
        keys = bsi_ops.build_bsi_keys_cuda(state["weights"], DECIMALS, THRESHOLD)[0]
        return {"planes": keys.words, "image": keys.ints8, "slice_weights": keys.slice_weights, "shifts": keys.shifts}
    if kind == "hybrid":
        streams = bsi_ops.build_bsi_queries_cuda_batch_hybrid(state["x"], DECIMALS, THRESHOLD)
        out = bsi_ops.batch_dot_product_multiquery_cuda_batch_caps(streams, state["keys"])[0]
        return {"streams": streams.comp_words, "lengths": streams.comp_len, "out": out}
    out, _total_ns, _build_ns, _dot_ns, query_bytes = bsi_ops.batch_dot_product_prebuilt(state["x"], state["keys"])
    return {"out": out, "query_bytes": query_bytes}


def work(case):
    """Bytes: activations and packed keys (6 planes, 3/4 byte a weight) in, outputs out.  Operations: 2 a multiply-add of
    the quantised values."""
    kind, d = case["kind"], case["d"]
    size = DTYPES[case["dtype"]].itemsize
    if kind == "keys":  # weights in; planes, int8 image, slice weights and shift of a row out
        return {"bytes": case["out"] * (d * (size + 1.75) + 28), "flops": 0.0}
    if kind == "decoder":
        t, n = case["rows"], case["layers"]
        return {"bytes": n * (12 * d * d * 0.75 + 13 * d * 4) + 2 * t * d * 4, "flops": n * (24.0 * t * d * d + 4.0 * t * t * d)}
    out = case["out"]
    if kind == "scalar":  # one slice count for all decimal keys: about 6 planes
        return {"bytes": d * 4 + out * d * 0.75 + out * 8, "flops": 2.0 * d * out}
    rows = case["rows"]
    keys = out * d * 0.75 + out * 4
    macs = 2.0 * rows * d * out
    if kind == "dot":  # seven planes of the queries and their chunk scales in
        return {"bytes": rows * (d * 0.875 + d / 64) + keys + rows * out * 4, "flops": macs}
    if kind == "hybrid":  # the streams go out too
        return {"bytes": rows * (d * size + d * 0.875) + keys + rows * out * 4, "flops": macs}
    return {"bytes": rows * d * size + keys + (out * 4 if case["bias"] else 0) + rows * out * size, "flops": macs}


def tolerance(case):
    """Sums of 32-bit products in any order; a half-precision layer rounds its output (and the bias sum) to its type."""
    kind = case["kind"]
    if kind == "decoder":
        return {"rel": 1e-3}  # a last-bit difference before a quantiser moves single values by a step
    if kind == "linear" and case["dtype"] != "float32":
        return {"rel": 1e-2 if case["dtype"] == "bfloat16" else 2e-3}
    return {"rel": 1e-12} if kind == "scalar" else {"rel": 1e-5}

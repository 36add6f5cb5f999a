"""Performance cases: the quantized Linear path as a model that serves requests calls it.

A case is one forward pass, through the public modules, of either
  * ``kind = "linear"``: one quantized Linear module, or
  * ``kind = "layer"``:  the four Linear modules of a decoder layer (qkv, o, gate_up, down) and its two RMSNorms in the
    order in which the layer runs them (attention and activation function are not part of this package, so ``o`` and
    ``down`` get their inputs from the case).
The methods are the registry's classes (``method_to_linear``) with their options:
  sq            SqW8A8BBF16OBF16PerTensor, the registry's SmoothQuant class (dynamic per-tensor activation scale)
  sq_channel    SqW8A8BBF16OBF16PerChannel (dynamic per-token scales; in a layer its norms feed it quantized rows)
  fp8_dynamic   FP8DynamicLinear, per-tensor scales (its default)
  fp8_token     FP8DynamicLinear, per-token x per-channel scales (in a layer its norms feed it quantized rows)
  fp8_static    FP8StaticLinear, calibrated input scale; ``quantize_output`` as for layers with an fp8 KV cache
  awq           WQLinear_GEMM, group 128 (32 and 64 are drawn too), fp16 activations or a bf16 model's

Sizes: the 7B-class layer of the benchmark (hidden 3584, qkv 4608, feed-forward 18944), the 0.5B-class one whose MLP
projection is the smallest benchmark configuration (hidden 896, feed-forward 4864), and generic ones in between; token
counts from one decoding sequence to a long prompt.
"""
from __future__ import annotations

import math

import torch

from llmqrt_amd.linear import (FP8DynamicLinear, FP8StaticLinear, SqW8A8BBF16OBF16PerChannel,
                               SqW8A8BBF16OBF16PerTensor, WQLinear_GEMM)
from llmqrt_amd.norm import RMSNorm

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
LAYER_7B = {"hidden": 3584, "qkv": 4608, "ffn": 18944}
LAYER_05B = {"hidden": 896, "qkv": 1152, "ffn": 4864}


def _linear(name, method, tokens, k, n, dtype, bias=False, group=128, quantize_output=False):
    return {"name": name, "kind": "linear", "method": method, "tokens": tokens, "k": k, "n": n, "dtype": dtype,
            "bias": bias, "group": group, "quantize_output": quantize_output}


def _layer(name, method, tokens, sizes, dtype, group=128):
    return {"name": name, "kind": "layer", "method": method, "tokens": tokens, **sizes, "dtype": dtype, "group": group}


def listed():
    return [
        # one sequence decoding, the narrowest projection of the 7B layer: launches and host work
        _linear("decode1_o_sq", "sq", 1, 3584, 3584, "bf16"),
        # sixteen sequences decoding on a small model: every launch is a few microseconds
        _layer("decode16_small_layer_fp8_dynamic", "fp8_dynamic", 16, LAYER_05B, "bf16"),
        # one sequence decoding on 4-bit weights: the weights cross HBM once per token
        _layer("decode1_layer_awq", "awq", 1, LAYER_7B, "fp16"),
        # a decode batch on int8 weights
        _layer("decode32_layer_sq_channel", "sq_channel", 32, LAYER_7B, "bf16"),
        # a larger decode batch on 4-bit weights inside a bf16 model, the widest projection
        _linear("decode64_gate_up_awq_bf16", "awq", 64, 3584, 37888, "bf16"),
        # a short prompt through a key projection whose output goes to an fp8 KV cache
        _linear("prompt200_k_fp8_static_out", "fp8_static", 200, 3584, 512, "bf16", bias=True, quantize_output=True),
        # a mid-sized prompt of no round length on 4-bit weights, the longest reduction
        _linear("prompt777_down_awq", "awq", 777, 18944, 3584, "fp16"),
        # a mid-sized prompt or a chunk of one, all projections
        _layer("prompt512_layer_fp8_token", "fp8_token", 512, LAYER_7B, "bf16"),
        # a prompt of a round decimal length (no multiple of any tile), projection with bias, fp16 model
        _linear("prompt1000_qkv_sq", "sq", 1000, 3584, 4608, "fp16", bias=True),
        # a long prompt, fp8, the longest reduction
        _linear("prompt4096_down_fp8_dynamic", "fp8_dynamic", 4096, 18944, 3584, "bf16"),
        # a long prompt through a whole layer
        _layer("prompt2048_layer_sq_channel", "sq_channel", 2048, LAYER_7B, "bf16"),
        # the largest call: the longest prompt through the widest projection
        _linear("prompt8192_gate_up_sq_channel", "sq_channel", 8192, 3584, 37888, "bf16"),
    ]


def _projections(case):
    """(name, in, out, bias) of the Linear modules of a case."""
    if case["kind"] == "linear":
        return [("out", case["k"], case["n"], case["bias"])]
    h, q, f = case["hidden"], case["qkv"], case["ffn"]
    return [("qkv", h, q, True), ("o", h, h, False), ("gate_up", h, 2 * f, False), ("down", f, h, False)]


def work(case):
    """Activations in, weights with their scales, outputs: each once."""
    m, nbytes, flops = case["tokens"], 0, 0
    for _, k, n, bias in _projections(case):
        weights = k * n // 2 + (k // case["group"]) * (2 * n + n // 2) if case["method"] == "awq" else k * n
        scales = 4 * n if case["method"] in ("sq_channel", "fp8_token") else 4
        out = (4 if case.get("quantize_output") else 2) * m * n
        nbytes += 2 * m * k + weights + scales + (2 * n if bias else 0) + out
        flops += 2 * m * n * k
    return {"bytes": nbytes, "flops": flops}


def _cost(case):
    """Seconds on the card, roughly: 8-bit operands at 2 POP/s, 4-bit weights on the fp16 cores at half of that."""
    w = work(case)
    return max(w["flops"] / (1e15 if case["method"] == "awq" else 2e15), w["bytes"] / 5e12)


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    methods = ("sq", "sq_channel", "fp8_dynamic", "fp8_token", "fp8_static", "awq")
    case = {"kind": "layer" if rng.random() < 0.35 else "linear", "method": rng.choice(methods)}
    case["tokens"] = _log_int(rng, 1, 8192)
    # the per-token fp8 op writes bf16 only
    case["dtype"] = "bf16" if case["method"] == "fp8_token" else rng.choice(("bf16", "bf16", "fp16"))
    case["group"] = rng.choice((128, 128, 128, 64, 32)) if case["method"] == "awq" else 128
    if case["kind"] == "layer":
        if rng.random() < 0.5:
            case.update(rng.choice((LAYER_7B, LAYER_05B)))
        else:
            hidden = 128 * _log_int(rng, 7, 28)
            case.update(hidden=hidden, qkv=hidden + 128 * rng.randint(2, 8), ffn=128 * _log_int(rng, 20, 148))
    else:
        step = 128 if case["method"] == "awq" else rng.choice((128, 128, 16))
        case["k"] = step * _log_int(rng, 896 // step, 18944 // step)
        case["n"] = 8 * _log_int(rng, 64, 37888 // 8) if rng.random() < 0.3 else 128 * _log_int(rng, 4, 296)
        case["bias"] = rng.random() < 0.4
        case["quantize_output"] = case["method"] == "fp8_static" and rng.random() < 0.3
    most = _cost(listed()[-1])
    while _cost(case) > most:
        case["tokens"] = max(1, int(0.8 * case["tokens"]))
    return case


def _module(case, k, n, bias, gen):
    """A quantized module made from a dense layer, as when a model is converted."""
    dtype = DTYPES[case["dtype"]]
    dense = torch.nn.Linear(k, n, bias=bias, device="meta")
    dense.weight = torch.nn.Parameter(0.02 * torch.randn(n, k, device="cuda", generator=gen), requires_grad=False)
    if bias:
        dense.bias = torch.nn.Parameter(0.5 * torch.randn(n, device="cuda", generator=gen), requires_grad=False)
    method = case["method"]
    if method == "sq":
        return SqW8A8BBF16OBF16PerTensor.from_linear(dense, 8, 0, init_only=False, dtype=dtype)
    if method == "sq_channel":
        return SqW8A8BBF16OBF16PerChannel.from_linear(dense, 8, 0, init_only=False, dtype=dtype)
    if method in ("fp8_dynamic", "fp8_token"):
        return FP8DynamicLinear.from_linear(dense, init_only=False, dtype=dtype, per_tensor=method == "fp8_dynamic")
    if method == "fp8_static":
        lin = FP8StaticLinear.from_linear(dense, init_only=False, dtype=dtype,
                                          quantize_output=case.get("quantize_output", False))
        # scales as a calibration run leaves them: the largest activation / output seen, over the largest e4m3 value
        lin.input_scale.data.fill_(90.0 / 448.0)
        lin.output_scale.data.fill_(0.02 * math.sqrt(5.0 * k) * 5.5 / 448.0)
        return lin
    group = case["group"]
    w = dense.weight.t().reshape(k // group, group, n)
    hi, lo = w.amax(dim=1), w.amin(dim=1)
    scales = ((hi - lo) / 15).clamp_(min=1e-5).half()
    zeros = (-lo / scales.float()).round_().clamp_(0, 15)
    return WQLinear_GEMM.from_linear(dense, 4, group, scales=scales, zeros=zeros)


def _activations(case, k, gen):
    """N(0, 1) with one channel in a hundred scaled by 20: the outlier channels activation quantizers have to live with.
    Decoding sequences come as [batch, 1, k], a prompt as [1, tokens, k]."""
    m = case["tokens"]
    x = torch.randn(m, k, device="cuda", generator=gen)
    x[:, torch.randperm(k, device="cuda", generator=gen)[: math.ceil(0.01 * k)]] *= 20.0
    if case["method"] == "fp8_static":
        x.clamp_(-90.0, 90.0)
    x = x.to(DTYPES[case["dtype"]])
    return x.view(m, 1, k) if m <= 64 else x.view(1, m, k)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    state = {"case": case, "mods": {}, "x": {}, "norms": {}}
    for name, k, n, bias in _projections(case):
        state["mods"][name] = _module(case, k, n, bias, gen)
        state["x"][name] = _activations(case, k, gen)
        if case["kind"] == "layer" and name in ("qkv", "gate_up"):
            # the norm weight of a smoothed layer carries 1 / smoothing factor: one channel scale each
            g = (1.0 + 0.1 * torch.randn(k, device="cuda", generator=gen)).to(DTYPES[case["dtype"]])
            state["norms"][name] = RMSNorm(g, 1e-6)
    return state


@torch.no_grad()
def run(state):
    case, mods, x, norms = state["case"], state["mods"], state["x"], state["norms"]
    if case["kind"] == "linear":
        return mods["out"](x["out"])
    out = {}
    for name, mod in mods.items():
        h = x[name]
        if name not in norms:
            out[name] = mod(h)
        elif case["method"] == "sq_channel":
            q, s = norms[name].forward_quantized(h)
            out[name] = mod.forward_quantized(q, s, h.dtype)
        elif case["method"] == "fp8_token":
            q, s = norms[name].forward_quantized(h, fp8=True)
            out[name] = mod.forward_quantized(q, s)
        else:
            out[name] = mod(norms[name](h))
    return out


def tolerance(case):
    """Four times the distance to the same computation with its products, sums and epilogue in 64 bits (codes and scales
    as the quantizers define them), measured over the methods above: relative 1.7e-3 / largest 4.0e-3 for bf16 results,
    2.1e-4 / 6.6e-4 for fp16 ones, 3.4e-4 / 1.2e-3 where 4-bit weights may or may not be rounded to fp16 first."""
    if case.get("quantize_output"):
        return {"rel": 9e-3, "max": 0.13}  # a result at a tie of the e4m3 grid may land on either side: one step is 1/8
    return {"rel": 6.7e-3, "max": 1.6e-2} if case["dtype"] == "bf16" else {"rel": 1.4e-3, "max": 5e-3}

"""What a program that serves quantised models has this framework do, as cases that can be timed.

Three kinds of work, all through the public entry points:

* "linear": one quantised linear layer on a batch of M token rows.  The 8-bit activation formats quantise the bf16 rows
  and multiply (`act_quant` + `fp8_gemm`, `int8_gemm`, `int8_gemm_per_token`, `w4a8_gemm`); the 16-bit activation formats
  multiply directly (`mul` on Marlin words, `w4a16_gemm` on bit-packed rows).
* "moe": one mixture-of-experts layer, router logits in, token rows out (`softmax_topk_router` + `ep_moe_forward`).
* "weights": one weight matrix on its way into a format, or back out of it, as when a model is loaded.

A case gives M, N, K (or the expert set's sizes) and the format; inputs are N(0, 1) activations and N(0, 0.02) weights.
"""
import math

import torch

from llm_kernels_amd.fast_dequant import w4a16
from llm_kernels_amd.fast_dequant.simple_marlin.marlin import mul
from llm_kernels_amd.fast_dequant.simple_marlin.utils import QuantUtils
from llm_kernels_amd.moe.ep_moe import ep_moe_forward, softmax_topk_router
from llm_kernels_amd.quantization import fp8_kernel, int8_kernel, w4a8_kernel

# the GEMMs return torch's default dtype: a bf16 inference program sets it once, when it starts
torch.set_default_dtype(torch.bfloat16)

FORMATS = ("fp8", "int8", "int8_per_token", "w4a8", "w4a16_marlin", "w4a16_rows")
# (N, K) of the attention and MLP projections that bench.py times (4096 wide, 14336 in the MLP, gate and up together)
PROJECTIONS = ((4096, 4096), (6144, 4096), (14336, 4096), (28672, 4096), (4096, 14336))
# (experts, experts per token, hidden, intermediate): eight large experts, and generic sets of more and smaller ones
EXPERT_SETS = ((8, 2, 4096, 14336), (16, 4, 4096, 2048), (64, 8, 2048, 1408))


def _linear(name, fmt, M, N, K, dtype="bf16"):
    return {"name": name, "kind": "linear", "format": fmt, "dtype": dtype, "M": M, "N": N, "K": K}


def _moe(name, fmt, tokens, experts=8, topk=2, hidden=4096, inter=14336):
    return {"name": name, "kind": "moe", "format": fmt, "tokens": tokens, "experts": experts, "topk": topk,
            "hidden": hidden, "inter": inter}


def listed():
    return [
        # one token of one request through the smallest projection: latency, launches and host time
        _linear("fp8 1 row", "fp8", 1, 4096, 4096),
        # a decode batch of 16 through the largest projection (gate and up together): streams the weights
        _linear("fp8 16 rows wide", "fp8", 16, 28672, 4096),
        # a prefill of 4096 tokens through the same projection: matrix cores
        _linear("fp8 prefill", "fp8", 4096, 28672, 4096),
        # an odd number of rows, as a batch of decoding requests with a chunk of a prompt gives, down projection
        _linear("int8 250 rows down", "int8", 250, 4096, 14336),
        # a prefill chunk with one scale per token and per output channel
        _linear("int8 per token prefill", "int8_per_token", 2048, 14336, 4096),
        # 4-bit weights, 8-bit activations: a decode batch, and a prefill chunk
        _linear("w4a8 16 rows", "w4a8", 16, 14336, 4096),
        _linear("w4a8 prefill", "w4a8", 1024, 4096, 4096),
        # 4-bit weights, 16-bit activations: a decode batch on Marlin words, and a ragged chunk on bit-packed rows
        _linear("w4a16 marlin 16 rows", "w4a16_marlin", 16, 4096, 4096, "fp16"),
        _linear("w4a16 rows 300 rows", "w4a16_rows", 300, 14336, 4096, "bf16"),
        # the Mixtral-shaped expert layer: a decode batch (streams the experts' weights) and a prefill (matrix cores)
        _moe("moe 16 tokens", "fp8", 16),
        _moe("moe prefill", "fp8", 4096),
        # loading a model: one MLP weight matrix into the two-level 4-bit format
        {"name": "w4a8 weights", "kind": "weights", "format": "w4a8", "to": "quantised", "N": 14336, "K": 4096},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _ragged(rng, fmt):
    """A weight shape off the projections' list: K in whole 128-blocks, N as fine as the format takes it."""
    K = 128 * _log_int(rng, 8, 112)
    N = _log_int(rng, 1024, 28672)
    step = {"w4a16_marlin": 64, "w4a8": 8, "w4a16_rows": 8}.get(fmt, rng.choice((1, 8, 8, 64)))
    return max(step, N // step * step), K


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "linear", "moe", "weights"))
    if kind == "moe":
        experts, topk, hidden, inter = rng.choice(EXPERT_SETS)
        case = _moe("", rng.choice(("fp8", "fp8", "int8")), _log_int(rng, 1, 4096), experts, topk, hidden, inter)
    elif kind == "weights":
        fmt = rng.choice(("fp8", "int8", "w4a8", "w4a16_rows"))
        N, K = rng.choice(PROJECTIONS) if rng.random() < 0.5 else _ragged(rng, "w4a8")
        to = "quantised" if fmt == "w4a16_rows" else rng.choice(("quantised", "dense"))
        case = {"name": "", "kind": kind, "format": fmt, "to": to, "N": N, "K": K}
    else:
        fmt = rng.choice(FORMATS)
        N, K = rng.choice(PROJECTIONS) if rng.random() < 0.5 else _ragged(rng, fmt)
        M = _log_int(rng, 1, 4096)
        dtype = "bf16"
        if fmt == "w4a16_marlin":
            M, dtype = -(-M // 16) * 16, "fp16"                  # `mul` takes whole 16-row tiles of fp16
        elif fmt == "w4a16_rows":
            dtype = rng.choice(("bf16", "fp16"))
        case = _linear("", fmt, M, N, K, dtype)
    del case["name"]
    return case


_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
_WEIGHT_QUANT = {"fp8": fp8_kernel.weight_quant, "int8": int8_kernel.weight_quant, "w4a8": w4a8_kernel.weight_quant}
_WEIGHT_DEQUANT = {"fp8": fp8_kernel.weight_dequant, "int8": int8_kernel.weight_dequant,
                   "w4a8": w4a8_kernel.weight_dequant}


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)

    def normal(*shape, scale=1.0, dtype=torch.bfloat16):
        return (torch.randn(*shape, generator=gen, device=dev, dtype=torch.float32) * scale).to(dtype)

    kind, fmt = case["kind"], case["format"]
    state = {"kind": kind, "format": fmt}
    if kind == "moe":
        T, E, H, I = case["tokens"], case["experts"], case["hidden"], case["inter"]
        quant = _WEIGHT_QUANT[fmt]
        experts = [(quant(normal(2 * I, H, scale=0.02)), quant(normal(H, I, scale=0.02))) for _ in range(E)]
        state["w13"] = torch.stack([e[0][0].view(torch.uint8) for e in experts]).view(experts[0][0][0].dtype)
        state["w13_scale"] = torch.stack([e[0][1] for e in experts])
        state["w2"] = torch.stack([e[1][0].view(torch.uint8) for e in experts]).view(experts[0][1][0].dtype)
        state["w2_scale"] = torch.stack([e[1][1] for e in experts])
        state["x"] = normal(T, H)
        state["logits"] = normal(T, E, dtype=torch.float32)
        state["topk"] = case["topk"]
        return state
    N, K = case["N"], case["K"]
    if kind == "weights":
        w = normal(N, K, scale=0.02, dtype=torch.float16 if fmt.startswith("w4") else torch.float32)
        state["to"] = case["to"]
        state["w"] = w if case["to"] == "quantised" else _WEIGHT_QUANT[fmt](w)
        return state
    state["x"] = normal(case["M"], K, dtype=_DTYPES[case["dtype"]])
    if fmt == "w4a16_marlin":
        _, q, s = QuantUtils.fake_quantize(normal(K, N, scale=0.02, dtype=torch.float16), 128)
        state["w"] = QuantUtils.pack(q, s, 128)
        state["out"] = torch.empty(case["M"], N, dtype=torch.float16, device=dev)
        state["workspace"] = torch.zeros(max(16, N // 128 * 16), dtype=torch.int32, device=dev)
    elif fmt == "w4a16_rows":
        state["w"] = w4a16.quantize_nk(normal(N, K, scale=0.02), 128)[:2]
    elif fmt == "int8_per_token":
        state["w"] = int8_kernel.weight_quant_per_channel(normal(N, K, scale=0.02))
    else:
        state["w"] = _WEIGHT_QUANT[fmt](normal(N, K, scale=0.02, dtype=torch.float16))
    return state


def run(state):
    kind, fmt = state["kind"], state["format"]
    if kind == "moe":
        ids, weights = softmax_topk_router(state["logits"], state["topk"])
        return ep_moe_forward(state["x"], ids, weights, state["w13"], state["w2"], state["w13_scale"], state["w2_scale"],
                              block_shape=[128, 128])
    w = state["w"]
    if kind == "weights":
        if state["to"] == "dense":
            return _WEIGHT_DEQUANT[fmt](*w)
        return w4a16.quantize_nk(w, 128) if fmt == "w4a16_rows" else _WEIGHT_QUANT[fmt](w)
    x = state["x"]
    if fmt == "fp8":
        return fp8_kernel.fp8_gemm(*fp8_kernel.act_quant(x), *w)
    if fmt == "int8":
        return int8_kernel.int8_gemm(*int8_kernel.act_quant(x), *w)
    if fmt == "int8_per_token":
        return int8_kernel.int8_gemm_per_token(*int8_kernel.act_quant_per_token(x), *w)
    if fmt == "w4a8":
        return w4a8_kernel.w4a8_gemm(*w4a8_kernel.act_quant(x), *w)
    if fmt == "w4a16_marlin":
        mul(x, w[0], state["out"], w[1], state["workspace"])
        return state["out"]
    return w4a16.w4a16_gemm(x, w[0], w[1], 128)


def _weight_bytes(fmt, N, K):
    """Bytes of a quantised [N, K] weight matrix with its scales."""
    blocks = -(-N // 128) * (K // 128)
    return {"fp8": N * K + 4 * blocks, "int8": N * K + 2 * blocks, "int8_per_token": N * K + 4 * N,
            "w4a8": N * K // 2 + 2 * blocks + 2 * N * (K // 128),
            "w4a16_marlin": N * K // 2 + 2 * N * (K // 128), "w4a16_rows": N * K // 2 + 2 * N * (K // 128)}[fmt]


def work(case):
    fmt = case["format"]
    if case["kind"] == "moe":
        T, E, H, I = case["tokens"], case["experts"], case["hidden"], case["inter"]
        rows = T * case["topk"]
        # experts that some token is routed to: the expected number under random logits
        routed = E * (1.0 - (1.0 - case["topk"] / E) ** T)
        per_expert = _weight_bytes(fmt, 2 * I, H) + _weight_bytes(fmt, H, I)
        return {"bytes": routed * per_expert + 4 * T * H + 4 * T * E, "flops": 6.0 * rows * H * I}
    N, K = case["N"], case["K"]
    if case["kind"] == "weights":
        dense = (4 if fmt in ("fp8", "int8") else 2) if case["to"] == "quantised" else 2
        codes = N * K if fmt == "w4a16_rows" else 0              # quantize_nk returns the unpacked codes too
        return {"bytes": N * K * dense + _weight_bytes(fmt, N, K) + codes, "flops": 2.0 * N * K}
    M = case["M"]
    return {"bytes": 2 * M * K + _weight_bytes(fmt, N, K) + 2 * M * N, "flops": 2.0 * M * N * K}


def tolerance(case):
    if case["kind"] == "weights":
        return "exact"                                           # codes, scales and products rounded once: one right answer
    # outputs are rounded to bf16 or fp16, sums over K are kept in 32 bits
    return {"rel": 1e-2 if case["kind"] == "moe" or case["dtype"] == "bf16" else 2e-3}

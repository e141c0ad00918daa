"""Blockwise W8A8 int8 quantisation and GEMM on MI355X.

Same functions as the reference quantization/int8_kernel.py: act_quant (:34), weight_quant (:91),
weight_dequant (:145), int8_gemm (:233).  act_quant_per_token / weight_quant_per_channel /
int8_gemm_per_token add the per-token x per-channel scheme with one full-K int32 accumulation.
"""
from typing import Tuple

import torch

try:
    from .. import _lib
except ImportError:  # this directory itself is on sys.path (the reference's top-level module layout)
    import _lib


def act_quant(x: torch.Tensor, block_size: int = 128) -> Tuple[torch.Tensor, torch.Tensor]:
    """1 x block_size groups: s = max|x| / 127 (fp32), y = round-half-away(x / s) int8, s stored fp16."""
    return _lib.host.act_quant(x, block_size, 1)


def weight_quant(x: torch.Tensor, block_size: int = 128) -> Tuple[torch.Tensor, torch.Tensor]:
    """block x block tiles of W [N, K]: s = blockmax / 127, half-away rounding, fp16 scales."""
    return _lib.host.weight_quant(x, block_size, False)


def weight_dequant(x: torch.Tensor, s: torch.Tensor, block_size: int = 128) -> torch.Tensor:
    """y = fp32(x) * s[block] in torch's default dtype."""
    return _lib.host.weight_dequant(x, s, block_size, False)


def int8_gemm(a: torch.Tensor, a_s: torch.Tensor, b: torch.Tensor, b_s: torch.Tensor):
    """c[..., n] = sum_kb fp32(int32 a_kb . b_kb[n]) * a_s[..., kb] * b_s[n // 128, kb]; default dtype out."""
    return _lib.host.int8_gemm(a, a_s, b, b_s)


# ----------------------------------------------------------------------------- per-token x per-channel
def act_quant_per_token(x: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
    """Per-token symmetric int8: s = max|row| / 127 (fp32) over the last dimension, y = round-half-away(x / s)."""
    return _lib.host.rowwise_quant(x)


def weight_quant_per_channel(w: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
    """Per-output-channel symmetric int8 of W [N, K], the same arithmetic with fp32 scales [N]."""
    return _lib.host.rowwise_quant(w)


def int8_gemm_per_token(a, a_s, b, b_s, return_int32: bool = False):
    """c[m, n] = int32(sum_k a[m,k] b[n,k]) * a_s[m] * b_s[n]; optionally also the raw int32 accumulators."""
    return _lib.host.int8_gemm_per_token(a, a_s, b, b_s, bool(return_int32))

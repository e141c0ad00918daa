"""DeepSeek-V3 style blockwise FP8 (OCP e4m3) quantisation and GEMM on MI355X.

Same functions as the reference quantization/fp8_kernel.py: act_quant (:33), weight_dequant (:84),
fp8_gemm (:170); weight_quant is the 128x128 weight analogue the reference lacks.  The bodies
validate like the reference (AssertionError), allocate the outputs and call the HIP kernels.
"""
from typing import Tuple

import torch

try:
    from .. import _lib
except ImportError:  # this directory itself is on sys.path (the reference's top-level module layout)
    import _lib


def act_quant(x: torch.Tensor, block_size: int = 128) -> Tuple[torch.Tensor, torch.Tensor]:
    """1 x block_size groups: s = max|x| / 448 (fp32), y = (x / s) as float8_e4m3fn."""
    return _lib.host.act_quant(x, block_size, 0)


def weight_quant(x: torch.Tensor, block_size: int = 128) -> Tuple[torch.Tensor, torch.Tensor]:
    """block x block tiles of W [N, K]: s = blockmax / 448 (fp32), y = (x / s) as float8_e4m3fn."""
    return _lib.host.weight_quant(x, block_size, True)


def weight_dequant(x: torch.Tensor, s: torch.Tensor, block_size: int = 128) -> torch.Tensor:
    """y = fp32(x) * s[block] in torch's default dtype."""
    return _lib.host.weight_dequant(x, s, block_size, True)


def fp8_gemm(a: torch.Tensor, a_s: torch.Tensor, b: torch.Tensor, b_s: torch.Tensor):
    """c[..., n] = sum_kb (a_kb . b_kb[n]) * a_s[..., kb] * b_s[n // 128, kb], fp32 accumulate,
    returned in torch's default dtype.  a [..., K] e4m3fn, b [N, K] e4m3fn, K % 128 == 0."""
    return _lib.host.fp8_gemm(a, a_s, b, b_s)

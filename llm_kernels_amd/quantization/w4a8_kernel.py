"""W4A8 (QServe-style two-level) weight quantisation and GEMM on MI355X.

Same functions as the reference quantization/w4a8_kernel.py: act_quant (:171), weight_quant (:265),
weight_dequant (:104), w4a8_gemm (:406).  Level 1: 128x128 blocks, s = absmax/119, clamp +-119;
level 2: per (row, 128-col group) asymmetric uint4 with int8 scale s4 and zero z4; eight rows are
packed per int32 word (nibble i of word [r, k] is row 8r + i).
"""
from typing import Tuple

import torch

try:
    from .. import _lib
except ImportError:  # this directory itself is on sys.path (the reference's top-level module layout)
    import _lib
from .bitpack import pack_weights_over_rows

PACKING_BITS = 32
W_BITS = 4


def act_quant(x: torch.Tensor, block_size: int = 128) -> Tuple[torch.Tensor, torch.Tensor]:
    """1 x block_size groups: s = max|x| / 127 (fp32), y = floor(x / s + 0.5) int8, s stored fp16."""
    return _lib.host.act_quant(x, block_size, 2)


def weight_quant(x: torch.Tensor, block_size: int = 128, group_size_int4: int = 128,
                 pack_direction: str = "row") -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor]:
    """W [N, K] -> (packed int32 [N/8, K], s fp16 [N/128, K/128], s4 int8 [N, K/g], z4 int8 [N, K/g])."""
    assert x.is_contiguous(), 'Input tensor must be contiguous'
    assert x.dim() == 2, 'Input tensors must have 2 dimensions'
    assert x.size(-1) % block_size == 0, f'Last dimension size must be divisible by block_size (block_size={block_size})'
    assert block_size % group_size_int4 == 0, 'block_size must be divisible by group_size_int4'
    _lib.require_gpu(x)
    assert pack_direction == "row", "Only row packing is supported"
    M, N = x.size()
    assert M % (PACKING_BITS // W_BITS) == 0, f'row nums must be divisible by {PACKING_BITS // W_BITS}'
    # The reference checks the nibble range 0..15 on the host between the levels and the packing.  The second level ends
    # in a clamp to that range which maps a NaN to 0 as well, so the check cannot fail here and no device is waited for.
    if block_size == 128 and 8 <= group_size_int4 <= 128 and group_size_int4 & (group_size_int4 - 1) == 0 and x.data_ptr() % 16 == 0:
        return _lib.host.w4a8_weight_quant(x, group_size_int4)
    y = torch.empty_like(x, dtype=torch.int8)
    s = x.new_empty(((M + block_size - 1) // block_size, (N + block_size - 1) // block_size), dtype=torch.float16)
    ng = (N + group_size_int4 - 1) // group_size_int4
    s4 = x.new_empty(M, ng, dtype=torch.int8)
    z4 = x.new_empty(M, ng, dtype=torch.int8)
    st = _lib.stream(x)
    _lib.call("llmk_weight_quant_i8_block", _lib.ptr(x), _lib.dt(x.dtype), _lib.ptr(y), _lib.ptr(s),
              M, N, block_size, 119.0, _lib.ROUND_HALF_UP, 1, st)
    _lib.call("llmk_weight_quant_w4a8_level2", _lib.ptr(y), _lib.ptr(s4), _lib.ptr(z4), M, N, group_size_int4, st)
    y_packed, _ = pack_weights_over_rows(y, W_BITS, PACKING_BITS, transpose=False)
    return y_packed, s, s4, z4


def weight_dequant(y: torch.Tensor, s: torch.Tensor, s4: torch.Tensor, z4: torch.Tensor,
                   block_size: int = 128, group_size_int4: int = 128, pack_direction: str = "row") -> torch.Tensor:
    """packed [N/8, K] -> fp16 [N, K]: ((q - z4) * s4 evaluated in int8) * s."""
    assert y.is_contiguous(), 'Input tensor must be contiguous'
    assert y.dim() == 2, 'Input tensors must have 2 dimensions'
    assert y.size(-1) % block_size == 0, f'Last dimension size must be divisible by block_size (block_size={block_size})'
    assert block_size % group_size_int4 == 0, 'block_size must be divisible by group_size_int4'
    assert pack_direction == "row", "Only row packing is supported for dequantization"
    return _lib.host.w4a8_weight_dequant(y, s, s4, z4, block_size, group_size_int4)


def w4a8_gemm(a: torch.Tensor, a_s: torch.Tensor, b: torch.Tensor,
              b_s: torch.Tensor, b_s4: torch.Tensor, b_z4: torch.Tensor,
              GROUP_SIZE_INT4: int = 128, elements_per_sample: int = 8,
              pack_direction: str = "row") -> torch.Tensor:
    """c = a(int8) x dequant_int8(b)^T with per-128-K a_s * b_s scaling; default dtype out."""
    assert pack_direction == "row", "Only row packing is supported for dequantization"
    assert elements_per_sample == PACKING_BITS // W_BITS, 'weights must be packed 8 nibbles per int32'
    return _lib.host.w4a8_gemm(a, a_s, b, b_s, b_s4, b_z4, GROUP_SIZE_INT4)

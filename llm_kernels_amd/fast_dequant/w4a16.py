"""W4A16 GEMM for weights kept in the plain [N, K] bit-packed layout.

W [N, K] is quantised symmetrically along K in groups (s = absmax / 7, q = clamp(rne(w / s), -8, 7) + 8)
and stored with quantization.bitpack.pack_weights_over_cols as int32 [N, K/8] (nibble i of a word is
k = 8*word + i).  The simple-Marlin layout has its own entry point (simple_marlin.marlin.mul).
"""
import torch

try:
    from .. import _lib
except ImportError:  # this directory itself is on sys.path (the reference's top-level module layout)
    import _lib


def quantize_nk(w: torch.Tensor, group_size: int = 128):
    """W [N, K] float -> (packed int32 [N, K/8], scales fp16 [N, K/group_size], q uint8 [N, K]).

    One pass over W on the GPU: s = absmax / 7 rounded to fp16, q = clamp(rne(w / s), -8, 7) + 8 with the
    quotient by the rounded scale in fp32, nibble i of a packed word is k = 8 * word + i (the layout of
    quantization.bitpack.pack_weights_over_cols(q, 4, 32, transpose=False))."""
    return _lib.host.w4_quantize_nk(w, group_size)


def w4a16_gemm(x: torch.Tensor, w_packed: torch.Tensor, scales: torch.Tensor, group_size: int = 128):
    """y[..., n] = sum_k x[..., k] * (nibble(n, k) - 8) * scales[n, k // group_size]; fp16 or bf16 in / out
    (the dtype of x), fp16 scales."""
    return _lib.host.w4a16_gemm(x, w_packed, scales, group_size)

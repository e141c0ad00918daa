"""EP-MoE device ops on MI355X (reference moe/group_gemm_kernel.py).

run_moe_ep_preproess (:48), grouped_gemm_triton (:442) keep their names and signatures.  The four
Triton kernels of the reference (pre_reorder :81, silu_and_mul :120, gelu_and_mul :176,
post_reorder :238) are exposed twice: as plain functions, and as `*_triton_kernel` objects that
accept the reference's `kernel[grid](args..., BLOCK_SIZE=...)` call form, so that a caller written
against the reference runs unchanged.
"""
from typing import List, Optional

import torch

try:
    from .. import _lib
    from ..quantization import fp8_kernel as _fp8_kernel, int8_kernel as _int8_kernel
except ImportError:  # this directory itself is on sys.path (the reference's top-level module layout)
    import _lib
    from quantization import fp8_kernel as _fp8_kernel, int8_kernel as _int8_kernel


def _cdiv(a, b):
    return (a + b - 1) // b


# limits of the one-launch sort behind llmk_moe_ep_preprocess (LLMK_MOE_PREPROCESS_MAX_* of the C header)
PREPROCESS_MAX_IDS = 32768
PREPROCESS_MAX_EXPERTS = 512


def run_moe_ep_preproess(topk_ids: torch.Tensor, num_experts: int):
    """Stable sort of the flattened expert ids -> (sorted ids, src2dst int32 [T*topk], seg_indptr int64 [E+1])."""
    _lib.require_gpu(topk_ids)
    n = topk_ids.numel()
    if (n <= PREPROCESS_MAX_IDS and num_experts <= PREPROCESS_MAX_EXPERTS and topk_ids.is_contiguous()
            and topk_ids.dtype in (torch.int32, torch.int64)):
        # the id counts of one forward pass: one launch instead of the eight of sort + pointers + map
        return _lib.host.ep_preprocess(topk_ids, int(num_experts))
    st = _lib.stream(topk_ids)
    reorder_topk_ids, reorder_ids = torch.sort(topk_ids.view(-1), stable=True)
    seg_indptr = torch.zeros(num_experts + 1, device=topk_ids.device, dtype=torch.int64)
    src2dst = torch.empty(n, device=topk_ids.device, dtype=torch.int32)
    sorted64 = reorder_topk_ids if reorder_topk_ids.dtype == torch.int64 else reorder_topk_ids.to(torch.int64)
    _lib.call("llmk_moe_seg_indptr", _lib.ptr(sorted64), _lib.ptr(seg_indptr), n, num_experts, st)
    _lib.call("llmk_moe_src2dst", _lib.ptr(reorder_ids), _lib.ptr(src2dst), n, st)
    return reorder_topk_ids, src2dst, seg_indptr


def _ids_bytes(t):
    if t.dtype == torch.int64:
        return 8
    if t.dtype == torch.int32:
        return 4
    raise TypeError("expert id tensors must be int32 or int64, got %s" % t.dtype)


def _f32_or_none(t):
    return None if t is None else t.float().contiguous()


def pre_reorder(input, gateup_input, src2dst, topk_ids, a1_scales, start_expert_id, end_expert_id, topk,
                hidden_size):
    """gateup_input[src2dst[t, j]] = input[t] * (1 / a1_scales[e] or 1) for every local expert e of token t."""
    _lib.require_gpu(input, gateup_input, src2dst, topk_ids)
    assert input.is_contiguous() and gateup_input.is_contiguous() and src2dst.is_contiguous() and topk_ids.is_contiguous()
    sc = _f32_or_none(a1_scales)
    T = input.numel() // hidden_size
    _lib.call("llmk_moe_pre_reorder", _lib.ptr(input), _lib.dt(input.dtype), _lib.ptr(gateup_input),
              _lib.dt(gateup_input.dtype), _lib.ptr(src2dst), _lib.ptr(topk_ids), _ids_bytes(topk_ids), _lib.ptr(sc),
              int(start_expert_id), int(end_expert_id), int(topk), T, int(hidden_size), _lib.stream(input))
    return gateup_input


def _act_and_mul(act, gateup_output, down_input, hidden_size, reorder_topk_ids, scales, start_expert_id,
                 end_expert_id):
    _lib.require_gpu(gateup_output, down_input, reorder_topk_ids)
    assert gateup_output.is_contiguous() and down_input.is_contiguous() and reorder_topk_ids.is_contiguous()
    sc = _f32_or_none(scales)
    M = gateup_output.numel() // hidden_size
    _lib.call("llmk_moe_act_and_mul", _lib.ptr(gateup_output), _lib.dt(gateup_output.dtype), _lib.ptr(down_input),
              _lib.dt(down_input.dtype), _lib.ptr(reorder_topk_ids), _ids_bytes(reorder_topk_ids), _lib.ptr(sc),
              int(start_expert_id), int(end_expert_id), M, int(hidden_size), act, _lib.stream(gateup_output))
    return down_input


def silu_and_mul(gateup_output, down_input, hidden_size, reorder_topk_ids, scales, start_expert_id, end_expert_id):
    """down_input[r] = dtype(silu_fp32(gate)) * up * (1/scale[e]); gate = cols [0, I), up = [I, 2I)."""
    return _act_and_mul(0, gateup_output, down_input, hidden_size, reorder_topk_ids, scales, start_expert_id,
                        end_expert_id)


def gelu_and_mul(gateup_output, down_input, hidden_size, reorder_topk_ids, scales, start_expert_id, end_expert_id):
    return _act_and_mul(1, gateup_output, down_input, hidden_size, reorder_topk_ids, scales, start_expert_id,
                        end_expert_id)


def post_reorder(down_output, output, src2dst, topk_ids, topk_weights, start_expert_id, end_expert_id, topk,
                 hidden_size):
    """output[t] = sum_j down_output[src2dst[t, j]] * dtype(topk_weights[t, j]), summed in the tensor dtype."""
    return _lib.host.post_reorder(down_output, output, src2dst, topk_ids, topk_weights, int(start_expert_id),
                                  int(end_expert_id), int(topk), int(hidden_size))


def _is_fp8(quant_dtype):
    """Which 1 x 128 activation format goes with a weight dtype: e4m3 with fp32 scales, or int8 with fp16 scales."""
    fp8 = quant_dtype == torch.float8_e4m3fn
    assert fp8 or quant_dtype == torch.int8, 'quant_dtype must be torch.int8 or torch.float8_e4m3fn'
    return fp8


_ACTS = {"silu": 0, "gelu": 1}


def pre_reorder_quant(input, src2dst, topk_ids, a1_scales, start_expert_id, end_expert_id, topk, hidden_size,
                      quant_dtype):
    """pre_reorder followed by the 1 x 128 activation quantizer, in one pass (the reference's TODO at
    sglang_moe_all_gather_all_reduce.py:295-296).  Returns (q [T*topk, hidden], s [T*topk, hidden/128]); equal
    bit for bit to act_quant(pre_reorder(...)).  Rows of non-local experts are left unwritten."""
    return _lib.host.pre_reorder_quant(input, src2dst, topk_ids, a1_scales, int(start_expert_id), int(end_expert_id),
                                       int(topk), int(hidden_size), _is_fp8(quant_dtype))


def act_and_mul_quant(gateup_output, hidden_size, reorder_topk_ids, scales, start_expert_id, end_expert_id, quant_dtype,
                      activation="silu"):
    """silu_and_mul / gelu_and_mul followed by the 1 x 128 activation quantizer, in one pass (the reference's TODO
    at sglang_moe_all_gather_all_reduce.py:365,407-408).  `hidden_size` is the gate+up width 2I as in
    silu_and_mul.  Returns (q [M, I], s [M, I/128]); equal bit for bit to act_quant(silu_and_mul(...))."""
    return _lib.host.act_and_mul_quant(gateup_output, int(hidden_size), reorder_topk_ids, scales, int(start_expert_id),
                                       int(end_expert_id), _is_fp8(quant_dtype), _ACTS[activation])


def grouped_gemm_swiglu_quant_fused(a, b, batch_size):
    """True when `grouped_gemm_swiglu_quant` runs this gate / up projection in one kernel (shapes that the 256-column
    tile kernel takes); otherwise run grouped_gemm_triton and act_and_mul_quant."""
    return _lib.host.swiglu_fused(a, b, int(batch_size))


def grouped_gemm_swiglu_quant(a, scale_a, b, scale_b, batch_size, seg_indptr, weight_indices, mid_dtype, activation="silu"):
    """Gate / up projection of a gated MLP over expert segments with the gated activation and the 1 x 128 quantiser of
    the down projection in the GEMM's epilogue: equal bit for bit to
    act_and_mul_quant(grouped_gemm_triton(a, b, c of `mid_dtype`, ...)), without the [M, 2I] tensor (the reference runs
    the three kernels one after the other, sglang_moe_all_gather_all_reduce.py:330-408).  a [M, K] and b [E, 2I, K]
    int8 or float8_e4m3fn with 1 x 128 / 128 x 128 block scales.  Returns (q [M, I], s [M, I/128]); rows outside every
    segment are left unwritten.  Only for shapes for which grouped_gemm_swiglu_quant_fused() is true."""
    assert mid_dtype in (torch.float16, torch.bfloat16)
    return _lib.host.swiglu_quant(a, scale_a, b, scale_b, int(batch_size), seg_indptr, weight_indices, _lib.dt(mid_dtype),
                                  _ACTS[activation])


class _GridCall:
    """Accepts `obj[grid](*args, BLOCK_SIZE=...)`; the grid and the tile size are chosen by the HIP launcher."""

    def __init__(self, fn):
        self._fn = fn
        self.__doc__ = fn.__doc__

    def __getitem__(self, grid):
        def launch(*args, BLOCK_SIZE=None, **kw):
            return self._fn(*args, **kw)
        return launch

    def __call__(self, *args, BLOCK_SIZE=None, **kw):
        return self._fn(*args, **kw)


pre_reorder_triton_kernel = _GridCall(pre_reorder)
silu_and_mul_triton_kernel = _GridCall(silu_and_mul)
gelu_and_mul_triton_kernel = _GridCall(gelu_and_mul)
post_reorder_triton_kernel = _GridCall(post_reorder)


def grouped_gemm_triton(
    a: torch.Tensor,
    b: torch.Tensor,
    c: torch.Tensor,
    batch_size: int,
    weight_column_major: bool,
    seg_indptr: Optional[torch.Tensor] = None,
    weight_indices: Optional[torch.Tensor] = None,
    use_fp8_w8a8: bool = False,
    scale_a: torch.Tensor = None,
    scale_b: torch.Tensor = None,
    block_shape: Optional[List[int]] = None,
):
    """c[seg[e]:seg[e+1]] = a[seg[e]:seg[e+1]] @ b[weight_indices[e]]^T for e < batch_size; c is written in place.

    With `block_shape` and quantised weights the activations are quantised here per 1 x block_k group:
    int8 weights -> int8 activations (the reference behaviour), float8_e4m3fn weights -> e4m3 activations.
    """
    assert weight_column_major == True  # noqa: E712  (same precondition as the reference)
    if use_fp8_w8a8 and block_shape is None:
        assert scale_a is not None and scale_b is not None
    _lib.require_gpu(a, b, c)
    assert seg_indptr is not None, 'seg_indptr is required'
    quantised_w = b.dtype in (torch.int8, torch.float8_e4m3fn)
    if block_shape is not None and quantised_w:
        assert len(block_shape) == 2
        block_n, block_k = block_shape[0], block_shape[1]
        assert block_n == 128 and block_k == 128, 'block-scaled grouped GEMM uses 128 x 128 weight blocks'
        if a.dtype == b.dtype:
            # extension: activations already in the 1 x block_k format of the weights (from pre_reorder_quant /
            # act_and_mul_quant); scale_a is theirs
            assert scale_a is not None, 'quantised activations need scale_a'
            scale_a = scale_a.contiguous()
        else:
            per_token_group_quant = (_int8_kernel if b.dtype == torch.int8 else _fp8_kernel).act_quant
            a, scale_a = per_token_group_quant(a.contiguous(), block_k)
        assert _cdiv(a.shape[-1], block_k) == scale_a.shape[-1]
        assert _cdiv(b.shape[-2], block_n) == scale_b.shape[-2]
        assert _cdiv(b.shape[-1], block_k) == scale_b.shape[-1]
    elif quantised_w and use_fp8_w8a8:
        # per-expert scalar scales (the branch the reference keeps commented out, group_gemm_kernel.py:417-420):
        # c = (a . b^T) * scale_a[e] * scale_b[e] with operands already quantised.  Run as block scales that are
        # constant per expert: a scalar factor commutes with the per-block accumulation.
        assert a.dtype == b.dtype, 'per-expert scaling takes activations already in the weight dtype'
        assert a.shape[-1] % 128 == 0, 'K must be a multiple of 128'
        kb = a.shape[-1] // 128
        nb = _cdiv(b.shape[1], 128)
        sdt = torch.float32 if b.dtype == torch.float8_e4m3fn else torch.float16
        seg64 = (seg_indptr if seg_indptr.dtype == torch.int64 else seg_indptr.to(torch.int64)).contiguous()
        sa = scale_a.to(torch.float32).flatten().contiguous()
        sb = scale_b.to(torch.float32).flatten().contiguous()
        assert sa.numel() >= batch_size and sb.numel() >= b.shape[0], 'one activation scale per segment, one weight scale per expert'
        scale_a = torch.empty(a.shape[0], kb, device=a.device, dtype=sdt)
        scale_b = torch.empty(b.shape[0], nb, kb, device=a.device, dtype=sdt)
        # one launch, nothing read back (usable under graph capture)
        _lib.call("llmk_moe_expert_scales", _lib.ptr(sa), _lib.ptr(sb), _lib.ptr(seg64), int(batch_size), b.shape[0],
                  a.shape[0], b.shape[1], b.shape[2], _lib.ptr(scale_a), _lib.ptr(scale_b), _lib.dt(sdt), _lib.stream(a))
    elif quantised_w:
        raise AssertionError('quantised weights need block_shape=[128, 128] and scale_b, or use_fp8_w8a8 with per-expert scales')
    return _lib.host.grouped_gemm(a, b, c, int(batch_size), seg_indptr, weight_indices, scale_a, scale_b)

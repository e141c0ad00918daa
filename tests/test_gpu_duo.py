"""The tile kernel whose two wave groups take turns (gemm_duo.hpp), on every tile height that is built: numbers of 128-byte sub-blocks around its
loop of four and below it, one to six K slices, ragged rows and columns."""
import ctypes

import pytest
import torch

from llm_kernels_amd import _lib
from llm_kernels_amd.fast_dequant import w4a16
from llm_kernels_amd.quantization import fp8_kernel, int8_kernel
from helpers import announce, assert_close_scaled, default_dtype

# (M, N, K): tile rows, K slices
FP8 = {(257, 6768, 128): (96, 1), (196, 8957, 256): (96, 1), (232, 8288, 384): (96, 1), (200, 8336, 640): (96, 1), (197, 8640, 768): (96, 1),
       (210, 8311, 896): (96, 1), (289, 6864, 1024): (96, 1), (201, 8648, 1152): (96, 1), (198, 8312, 1280): (96, 1), (257, 6616, 1408): (96, 1),
       (593, 224, 3072): (96, 4), (1450, 287, 4224): (96, 4), (301, 8280, 1536): (128, 1), (298, 8776, 1152): (128, 1), (290, 8435, 1280): (128, 1),
       (290, 8224, 1408): (128, 1), (1351, 648, 6144): (128, 3)}
INT8 = {(193, 8264, 896): (96, 1), (201, 8285, 1152): (96, 1), (257, 6824, 1408): (96, 1), (749, 1288, 6144): (96, 2), (582, 216, 3072): (96, 4),
        (294, 8288, 4096): (128, 1), (307, 8287, 4224): (128, 1), (704, 1320, 6144): (128, 3)}
PER_TOKEN = {(524, 3632, 1536): (96, 1), (519, 3607, 1152): (96, 1), (526, 248, 3072): (96, 4), (1011, 375, 4224): (96, 3), (289, 8424, 3072): (128, 1),
             (291, 8344, 4224): (128, 1), (2042, 407, 6144): (128, 4), (450, 8256, 640): (160, 1), (451, 8888, 768): (160, 1), (452, 8391, 1152): (160, 1),
             (590, 6536, 1408): (160, 1)}
W4 = {(1081, 224, 128): (96, 1), (1465, 208, 256): (96, 1), (1054, 224, 384): (96, 1), (566, 216, 1152): (96, 3), (537, 240, 1280): (96, 3),
      (659, 208, 2176): (96, 4), (850, 280, 4224): (96, 6), (1849, 1552, 384): (128, 1), (1080, 2704, 512): (128, 1), (865, 1104, 4224): (128, 4),
      (1029, 3664, 128): (160, 1), (1538, 2456, 256): (160, 1), (1160, 3208, 384): (160, 1), (300, 14336, 4096): (160, 1), (148, 6672, 4224): (160, 4),
      (1605, 2952, 128): (192, 1), (979, 4728, 256): (192, 1), (983, 4688, 384): (192, 1), (990, 4688, 512): (192, 1), (169, 6408, 6144): (192, 4)}


def shape(entry, *args):
    out = (ctypes.c_int32 * 2)()
    return (out[0], out[1]) if getattr(_lib.load(), entry)(*args, ctypes.cast(out, ctypes.c_void_p)) else None


def shape8(kind, per_token, M, N, K):
    return shape("llmk_gemm_8bit_duo_shape", kind, per_token, M, N, K, _lib.load().llmk_gemm_workspace_bytes(M, N, K))


def test_the_cases_reach_every_tile():
    for cases, kind, per_token, heights in ((FP8, _lib.KIND_FP8, 0, {96, 128}), (INT8, _lib.KIND_I8, 0, {96, 128}), (PER_TOKEN, _lib.KIND_I8, 1, {96, 128, 160})):
        assert {rows for rows, _ in cases.values()} == heights
        for call, want in cases.items():
            assert shape8(kind, per_token, *call) == want, (kind, per_token, call)
    assert {rows for rows, _ in W4.values()} == {96, 128, 160, 192}
    for (M, N, K), want in W4.items():
        assert shape("llmk_gemm_w4a16_duo_shape", _lib.F16, M, N, K, 128, 1 << 50) == want, (M, N, K)


def test_scratch_of_its_slices_is_reported_and_small():
    """What is reported holds the planes of the slices, and never more than the array that serves calls without scratch of their own."""
    for (M, N, K), (_, z) in {**FP8, **INT8, **PER_TOKEN}.items():
        assert 4 * z * M * N * (z > 1) <= _lib.load().llmk_gemm_workspace_bytes(M, N, K) <= 32 << 20, (M, N, K)


def _ints(gen, dev, lo, hi, *size):
    return torch.randint(lo, hi + 1, size, device=dev, generator=gen)


def _call8(name, a, a_s, b, b_s, M, N, K, scratch, out):
    ws = torch.empty(scratch, dtype=torch.uint8, device=a.device) if scratch else None
    args = [_lib.ptr(a), _lib.ptr(a_s), _lib.ptr(b), _lib.ptr(b_s)] + ([_lib.dt(a_s.dtype)] if name == "llmk_gemm_i8_block" else [])
    _lib.call(name, *args, _lib.ptr(out), _lib.dt(out.dtype), M, N, K, _lib.ptr(ws) if scratch else None, scratch, _lib.stream(a))
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("kind,M,N,K,scales", [("fp8", *c, torch.float32) for c in FP8] +
                         [("int8", *c, (torch.float16, torch.bfloat16, torch.float32)[i % 3]) for i, c in enumerate(INT8)])
def test_block_scales_exact(dev, kind, M, N, K, scales):
    """Small integers under powers of two of their own in every row, column block and K step: the fp32 result is exact in any order; with the
    reported scratch, with none, and with room for one plane."""
    announce("duo", kind, M, N, K, scales)
    gen = torch.Generator(device=dev).manual_seed(M + K)
    kb, nb = K // 128, -(-N // 128)
    a, b = _ints(gen, dev, -3, 3, M, K), _ints(gen, dev, -3, 3, N, K)
    a_s, b_s = (2.0 ** _ints(gen, dev, 0, 3, M, kb)).to(scales), (2.0 ** _ints(gen, dev, 0, 3, nb, kb)).to(scales)
    ref = (a.double() * a_s.double().repeat_interleave(128, 1)) @ (b.double() * b_s.double().repeat_interleave(128, 1).repeat_interleave(128, 0)[:N]).t()
    dt, name = (torch.float8_e4m3fn, "llmk_gemm_fp8_block") if kind == "fp8" else (torch.int8, "llmk_gemm_i8_block")
    a8, b8 = a.float().to(dt), b.float().to(dt)
    with default_dtype(torch.float32):
        c = fp8_kernel.fp8_gemm(a8, a_s, b8, b_s) if kind == "fp8" else int8_kernel.int8_gemm(a8, a_s, b8, b_s)
    assert torch.equal(c.double(), ref)
    for scratch in (0, 4 * M * N + 256):
        out = torch.full((M, N), float("nan"), device=dev)
        assert torch.equal(_call8(name, a8, a_s, b8, b_s, M, N, K, scratch, out).double(), ref), scratch
    out = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
    assert_close_scaled(_call8(name, a8, a_s, b8, b_s, M, N, K, _lib.load().llmk_gemm_workspace_bytes(M, N, K), out), ref, rtol=2 ** -8, atol=0)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", PER_TOKEN)
def test_per_token_exact(dev, M, N, K):
    announce("duo per token", M, N, K)
    gen = torch.Generator(device=dev).manual_seed(M + K)
    a, b = _ints(gen, dev, -128, 127, M, K).to(torch.int8), _ints(gen, dev, -128, 127, N, K).to(torch.int8)
    a_s, b_s = torch.rand(M, device=dev, generator=gen) + 0.5, torch.rand(N, device=dev, generator=gen) + 0.5
    ref = a.double() @ b.double().t()
    with default_dtype(torch.float32):
        c, acc = int8_kernel.int8_gemm_per_token(a, a_s, b, b_s, return_int32=True)
    assert torch.equal(acc.double(), ref)
    assert torch.equal(c, acc.float() * a_s[:, None] * b_s[None, :])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", W4)
def test_row_packed_weights(dev, M, N, K, dtype):
    """One element of a row: the output row is a column of the rounded weights, to the bit.  Random rows: fp32 sums of exact products, one rounding."""
    announce("duo w4", dtype, M, N, K)
    gen = torch.Generator(device=dev).manual_seed(M + K)
    w = torch.randn(N, K, device=dev, generator=gen, dtype=torch.float32) * 0.02
    packed, scales, codes = w4a16.quantize_nk(w, 128)
    weights = ((codes.float() - 8) * scales.float().repeat_interleave(128, 1)).to(dtype)
    k = (7 * torch.arange(M, device=dev) + 3) % K
    x = torch.zeros(M, K, dtype=dtype, device=dev)
    x[torch.arange(M, device=dev), k] = 1
    assert torch.equal(w4a16.w4a16_gemm(x, packed, scales, 128), weights[:, k].t())
    x = torch.randn(M, K, device=dev, generator=gen, dtype=torch.float32).to(dtype)
    ref = x.double() @ weights.double().t()
    assert_close_scaled(w4a16.w4a16_gemm(x, packed, scales, 128), ref, rtol=2 ** -8 if dtype == torch.bfloat16 else 2 ** -11, atol=2e-5)

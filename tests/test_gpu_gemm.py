"""HIP block-scaled GEMMs vs the float64 oracle.

Tolerance: |c - ref| <= 1e-2 * rms(ref) + 1e-2 * |ref| (rtol 1e-2 / atol 1e-2 relative to the output
scale).  Integer accumulators are checked bit-exactly.
"""
import ctypes

import pytest
import torch

from oracle import gemm_ref as g, quant_ref as q, bitpack_ref as bp
from llm_kernels_amd import _lib
from llm_kernels_amd.fast_dequant import w4a16
from llm_kernels_amd.quantization import fp8_kernel, int8_kernel, w4a8_kernel
from helpers import announce, assert_close_scaled, default_dtype

pytestmark = pytest.mark.gpu

SMALL = [(1, 128, 128), (16, 256, 512), (5, 130, 256), (33, 200, 384), (70, 64, 1024), (128, 512, 256)]


def _quant_inputs_fp8(M, N, K, seed):
    torch.manual_seed(seed)
    x = torch.randn(M, K).bfloat16()
    w = torch.randn(N, K) * 0.02
    a, a_s = q.act_quant_fp8(x)
    b, b_s = q.weight_quant_fp8(w)
    return a, a_s, b, b_s


@pytest.mark.parametrize("M,N,K", SMALL)
@pytest.mark.parametrize("out", [torch.bfloat16, torch.float16, torch.float32])
def test_fp8_gemm_small(dev, M, N, K, out):
    announce("fp8_gemm", M, N, K, out)
    a, a_s, b, b_s = _quant_inputs_fp8(M, N, K, M + N)
    with default_dtype(out):
        c = fp8_kernel.fp8_gemm(a.to(dev), a_s.to(dev), b.to(dev), b_s.to(dev))
    assert c.dtype == out and c.shape == (M, N)
    assert_close_scaled(c, g.gemm_blockwise(a, a_s, b, b_s), what="fp8_gemm")


def test_fp8_gemm_batched_leading_dims_and_asserts(dev):
    announce("fp8_gemm leading dims")
    a, a_s, b, b_s = _quant_inputs_fp8(6, 256, 256, 3)
    with default_dtype(torch.bfloat16):
        c = fp8_kernel.fp8_gemm(a.view(2, 3, 256).to(dev), a_s.view(2, 3, 2).to(dev), b.to(dev), b_s.to(dev))
    assert c.shape == (2, 3, 256)
    assert_close_scaled(c.view(6, 256), g.gemm_blockwise(a, a_s, b, b_s))
    with pytest.raises(AssertionError):
        fp8_kernel.fp8_gemm(a.to(dev).t(), a_s.to(dev), b.to(dev), b_s.to(dev))


@pytest.mark.parametrize("M,N,K", [(1, 4096, 4096), (16, 4096, 4096), (16, 6144, 4096), (256, 4096, 4096)])
def test_fp8_gemm_llama_shapes(dev, M, N, K):
    announce("fp8_gemm llama", M, N, K)
    a, a_s, b, b_s = _quant_inputs_fp8(M, N, K, 11)
    with default_dtype(torch.bfloat16):
        c = fp8_kernel.fp8_gemm(a.to(dev), a_s.to(dev), b.to(dev), b_s.to(dev))
    assert_close_scaled(c, g.gemm_blockwise(a, a_s, b, b_s), what="fp8 llama")


def test_fp8_gemm_quantize_on_device_end_to_end(dev):
    """act_quant + weight_quant + fp8_gemm on the GPU against the unquantised product (reference-style check)."""
    announce("fp8 end to end 64x4096x14336")
    torch.manual_seed(5)
    x = torch.randn(64, 14336, device=dev).bfloat16()
    w = (torch.randn(4096, 14336, device=dev) * 0.02)
    a, a_s = fp8_kernel.act_quant(x)
    b, b_s = fp8_kernel.weight_quant(w)
    with default_dtype(torch.bfloat16):
        c = fp8_kernel.fp8_gemm(a, a_s, b, b_s)
    ref = x.float() @ w.t()
    cos = torch.nn.functional.cosine_similarity(c.float().flatten(), ref.flatten(), dim=0)
    assert cos > 0.999
    assert_close_scaled(c, g.gemm_blockwise(a.cpu(), a_s.cpu(), b.cpu(), b_s.cpu()), what="fp8 e2e")


# ------------------------------------------------------------------------------------------- int8
@pytest.mark.parametrize("M,N,K", SMALL + [(16, 4096, 4096), (128, 14336, 4096)])
def test_int8_gemm(dev, M, N, K):
    announce("int8_gemm", M, N, K)
    torch.manual_seed(M * 7 + N)
    a, a_s = q.act_quant_int8(torch.randn(M, K))
    b, b_s = q.weight_quant_int8(torch.randn(N, K) * 0.02)
    with default_dtype(torch.bfloat16):
        c = int8_kernel.int8_gemm(a.to(dev), a_s.to(dev), b.to(dev), b_s.to(dev))
    assert c.dtype == torch.bfloat16
    assert_close_scaled(c, g.gemm_blockwise(a, a_s, b, b_s), what="int8_gemm")


@pytest.mark.parametrize("M,N,K", [(1, 128, 128), (16, 256, 4096), (37, 130, 512), (128, 512, 14336), (3850, 4110, 640)])
def test_int8_block_accumulators_bit_exact(dev, M, N, K):
    """Unit scales and fp32 output: the result is the exact integer product (every 128-K int32 partial
    and their sum stay below 2^24 for |values| <= 15)."""
    announce("int8 exact", M, N, K)
    torch.manual_seed(K)
    a = torch.randint(-15, 16, (M, K), dtype=torch.int8)
    b = torch.randint(-15, 16, (N, K), dtype=torch.int8)
    a_s = torch.ones(M, K // 128, dtype=torch.float16)
    b_s = torch.ones((N + 127) // 128, K // 128, dtype=torch.float16)
    with default_dtype(torch.float32):
        c = int8_kernel.int8_gemm(a.to(dev), a_s.to(dev), b.to(dev), b_s.to(dev))
    assert torch.equal(c.cpu().long(), a.long() @ b.long().T)
    # full-range values, one K block: a single int32 partial (|sum| <= 128*127*127 < 2^24) is exact in fp32
    a1 = torch.randint(-127, 128, (M, 128), dtype=torch.int8)
    b1 = torch.randint(-127, 128, (N, 128), dtype=torch.int8)
    with default_dtype(torch.float32):
        c1 = int8_kernel.int8_gemm(a1.to(dev), a_s[:, :1].contiguous().to(dev), b1.to(dev), b_s[:, :1].contiguous().to(dev))
    assert torch.equal(c1.cpu().long(), a1.long() @ b1.long().T)


@pytest.mark.parametrize("M,N,K", [(1, 4096, 4096), (16, 4096, 4096), (130, 200, 1024), (128, 4096, 14336),
                                   (65, 136, 128), (300, 264, 640), (1000, 521, 1152), (2048, 4096, 2048),
                                   (4096, 4096, 1024), (3850, 4110, 640),
                                   (300, 1000, 8192), (70, 1001, 8192), (100, 2050, 4096)])   # K split into 7, 8, 4
def test_int8_per_token_int32_bit_exact(dev, M, N, K):
    announce("int8 rowcol", M, N, K)
    torch.manual_seed(M + K)
    a, a_s = q.int8_quant_rowwise(torch.randn(M, K))
    b, b_s = q.int8_quant_rowwise(torch.randn(N, K) * 0.02)
    with default_dtype(torch.bfloat16):
        c, acc = int8_kernel.int8_gemm_per_token(a.to(dev), a_s.to(dev), b.to(dev), b_s.to(dev), return_int32=True)
    assert acc.dtype == torch.int32 and torch.equal(acc.cpu(), g.int8_gemm_int32(a, b))
    assert_close_scaled(c, g.int8_gemm_rowcol(a, a_s, b, b_s), what="int8 rowcol")
    # without scratch the entry point cannot split K: the slices' integer sums must give the same bits
    ad, bd, asd, bsd = a.to(dev), b.to(dev), a_s.to(dev).float().contiguous(), b_s.to(dev).float().contiguous()
    c0 = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
    _lib.call("llmk_gemm_i8_rowcol", _lib.ptr(ad), _lib.ptr(asd), _lib.ptr(bd), _lib.ptr(bsd), _lib.ptr(c0),
              _lib.dt(c0.dtype), None, M, N, K, None, 0, _lib.stream(ad))
    assert torch.equal(c0, c), "int8 rowcol: split and unsplit K differ"
    with default_dtype(torch.float32):     # scaled output alone (no accumulator buffer), full-range operands
        a2 = torch.randint(-128, 128, (M, K), dtype=torch.int8)
        b2 = torch.randint(-128, 128, (N, K), dtype=torch.int8)
        c2 = int8_kernel.int8_gemm_per_token(a2.to(dev), a_s.to(dev), b2.to(dev), b_s.to(dev))
    assert_close_scaled(c2, g.int8_gemm_rowcol(a2, a_s, b2, b_s), what="int8 rowcol full range")
    ag, asg = int8_kernel.act_quant_per_token(torch.randn(M, K, device=dev))
    assert ag.dtype == torch.int8 and asg.shape == (M,)


@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 13])
@pytest.mark.parametrize("M", [2000, 4000])            # the 128 x 256 and the 256 x 256 tile, the last tile row ragged
@pytest.mark.parametrize("kind", ["fp8", "int8", "int8 fp16 scales", "int8 bf16 scales"])
def test_scales_of_every_k_step_on_large_tiles(dev, kind, M, steps):
    """Small integers under scales that are powers of two of their own in every row, column block and K step: every product and sum is
    a whole number below 2^24, so the fp32 result is exact in any order, and a scale taken from another step or row shows."""
    announce("scales on large tiles", kind, M, steps)
    check_scales_of_every_k_step(dev, kind.split()[0], M, 4096, steps, torch.float16 if " fp16" in kind else torch.bfloat16 if "bf16" in kind else torch.float32)


@pytest.mark.parametrize("steps", [1, 3, 4, 6, 9, 31, 62])
@pytest.mark.parametrize("M,N", [(40, 1024), (70, 4096), (129, 2048), (250, 3968), (251, 1920)])
@pytest.mark.parametrize("kind", ["fp8", "int8", "int8 fp16 scales"])
def test_scales_of_every_k_step_on_mid_size_tiles(dev, kind, M, N, steps):
    """The same where K steps of 512 bytes end inside a step, in 32- and 64-row tiles, ragged rows, 64 and 128 columns and K slices."""
    announce("scales on mid-size tiles", kind, M, N, steps)
    check_scales_of_every_k_step(dev, kind.split()[0], M, N, steps, torch.float16 if "fp16" in kind else torch.float32)


@pytest.mark.parametrize("scales", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("extra", [-16, 0, 256, 1 << 30])
@pytest.mark.parametrize("M,N,steps", [(861, 2801, 200), (520, 264, 9), (918, 8219, 64)])
def test_int8_scales_at_scratch_limits(dev, M, N, steps, extra, scales):
    """16-bit activation scales where the split last round of 256-column tiles fits in the scratch, but not behind fp32 scales (861 x 2801 x 25600 is one of the
    shapes that go to another tile with it, 918 x 8219 x 8192 splits its last round with fp16 scales as they are): the scales are read as what they are, whatever
    scratch there is, and nothing behind it is written."""
    announce("int8 scales, scratch", M, N, steps, extra, str(scales))
    nbytes = min((64 << 20) + extra, _lib.load().llmk_gemm_workspace_bytes(M, N, 128 * steps))
    check_scales_of_every_k_step(dev, "int8", M, N, steps, scales, nbytes)


@pytest.mark.parametrize("scratch", [None, 0])
@pytest.mark.parametrize("steps", [84, 85, 86, 87])
def test_int8_fp16_scales_on_both_sides_of_the_widening_line(dev, steps, scratch):
    """4000 x 4096: up to 85 K steps the 256-column tiles take fp16 scales as they are, from 86 on a pass widens them if there is scratch for it."""
    announce("int8 fp16 scales, widened or not", steps, scratch)
    check_scales_of_every_k_step(dev, "int8", 4000, 4096, steps, torch.float16, scratch)


def check_scales_of_every_k_step(dev, kind, M, N, steps, scales, scratch=None):
    K = 128 * steps
    gen = torch.Generator(device=dev).manual_seed(100 * steps + M)

    def ints(lo, hi, *shape):
        return torch.randint(lo, hi + 1, shape, device=dev, generator=gen)

    a, b = ints(-3, 3, M, K), ints(-3, 3, N, K)
    a_s, b_s = 2.0 ** ints(0, 4, M, steps).float(), 2.0 ** ints(0, 4, -(-N // 128), steps).float()
    ref = (a.double() * a_s.double().repeat_interleave(128, 1)) @ (b.double() * b_s.double().repeat_interleave(128, 1).repeat_interleave(128, 0)[:N]).t()
    a_s, b_s = a_s.to(scales), b_s.to(scales)
    with default_dtype(torch.float32):
        if scratch is not None:
            a, b = a.to(torch.int8), b.to(torch.int8)
            c = torch.full((M, N), float("nan"), device=dev)
            ws = torch.full((scratch + 256,), 0x5A, dtype=torch.uint8, device=dev)
            _lib.call("llmk_gemm_i8_block", _lib.ptr(a), _lib.ptr(a_s), _lib.ptr(b), _lib.ptr(b_s), _lib.dt(scales), _lib.ptr(c), _lib.dt(torch.float32), M, N, K,
                      _lib.ptr(ws), scratch, None)
            assert (ws[scratch:] == 0x5A).all()
        elif kind == "fp8":
            c = fp8_kernel.fp8_gemm(a.float().to(torch.float8_e4m3fn), a_s, b.float().to(torch.float8_e4m3fn), b_s)
        else:
            c = int8_kernel.int8_gemm(a.to(torch.int8), a_s, b.to(torch.int8), b_s)
    assert torch.equal(c.double(), ref)


# ------------------------------------------------------------------------------------------- w4a8
@pytest.mark.parametrize("M,N,K", [(1, 128, 128), (16, 256, 512), (37, 136, 256), (16, 4096, 4096), (128, 1024, 7168),
                                   (5, 8, 128), (33, 264, 2048), (64, 4096, 4096), (17, 1032, 2176), (16, 14336, 4096),
                                   (16, 512, 4224), (16, 4096, 14336), (64, 520, 12416)])
def test_w4a8_gemm(dev, M, N, K):
    announce("w4a8_gemm", M, N, K)
    torch.manual_seed(N + K)
    wq, s, s4, z4 = q.w4a8_weight_quant_levels(torch.randn(N, K) * 0.02)
    a, a_s = q.act_quant_int8(torch.randn(M, K).bfloat16(), rounding="up")
    packed, _ = bp.pack_rows(wq.numpy(), 4, 32)
    with default_dtype(torch.bfloat16):
        c = w4a8_kernel.w4a8_gemm(a.to(dev), a_s.to(dev), torch.from_numpy(packed).to(dev), s.to(dev),
                                  s4.to(dev), z4.to(dev), 128, 8, "row")
    assert c.shape == (M, N) and c.dtype == torch.bfloat16
    assert_close_scaled(c, g.w4a8_gemm(a, a_s, wq, s, s4, z4), what="w4a8_gemm")


def test_w4a8_exact_and_wrap(dev):
    """Unit block scales + fp32 out: exact integers, including out-of-contract s4/z4 that wrap in int8."""
    announce("w4a8 exact/wrap")
    torch.manual_seed(9)
    M, N, K = 8, 64, 256
    wq = torch.randint(0, 16, (N, K), dtype=torch.uint8)
    s4 = torch.randint(1, 4, (N, K // 128), dtype=torch.int8)
    z4 = torch.randint(0, 16, (N, K // 128), dtype=torch.int8)
    s4[0, 0], z4[0, 0] = 20, 2            # (15 - 2) * 20 = 260 wraps
    s4[1, 1], z4[1, 1] = -9, 15           # negative scale
    a = torch.randint(-7, 8, (M, K), dtype=torch.int8)
    ones_a = torch.ones(M, K // 128, dtype=torch.float16)
    ones_b = torch.ones(1, K // 128, dtype=torch.float16)
    packed, _ = bp.pack_rows(wq.numpy(), 4, 32)
    with default_dtype(torch.float32):
        c = w4a8_kernel.w4a8_gemm(a.to(dev), ones_a.to(dev), torch.from_numpy(packed).to(dev), ones_b.to(dev),
                                  s4.to(dev), z4.to(dev))
    b8 = q.w4a8_dequant_int8(wq, s4, z4)
    assert torch.equal(c.cpu().long(), a.long() @ b8.long().T)


@pytest.mark.parametrize("M,N,K,sdt", [(16, 5000, 1024, torch.float16), (16, 4104, 128, torch.float32),
                                       (3, 264, 1408, torch.bfloat16), (30, 1040, 1920, torch.float16),
                                       (16, 72, 3072, torch.float32), (1, 8, 2176, torch.float16), (40, 8192, 4096, torch.float32),
                                       (3, 312, 384, torch.bfloat16), (16, 1032, 8320, torch.float16),
                                       (50, 264, 14336, torch.float32)])
def test_w4a8_decode_exact_mixed_wrap(dev, M, N, K, sdt):
    """Decode-size shapes over many column tiles with a sprinkle of out-of-contract (s4, z4): exact integers."""
    announce("w4a8 decode exact", M, N, K, sdt)
    torch.manual_seed(M + N)
    wq = torch.randint(0, 16, (N, K), dtype=torch.uint8)
    s4 = torch.randint(1, 9, (N, K // 128), dtype=torch.int8)
    z4 = torch.randint(0, 16, (N, K // 128), dtype=torch.int8)
    wild = torch.rand(N, K // 128) < 0.02
    s4[wild] = torch.randint(-128, 128, (int(wild.sum()),), dtype=torch.int8)
    z4[wild] = torch.randint(-128, 128, (int(wild.sum()),), dtype=torch.int8)
    a = torch.randint(-3, 4, (M, K), dtype=torch.int8)
    ones_a = torch.ones(M, K // 128, dtype=sdt)
    ones_b = torch.ones((N + 127) // 128, K // 128, dtype=sdt)
    packed, _ = bp.pack_rows(wq.numpy(), 4, 32)
    with default_dtype(torch.float32):
        c = w4a8_kernel.w4a8_gemm(a.to(dev), ones_a.to(dev), torch.from_numpy(packed).to(dev), ones_b.to(dev),
                                  s4.to(dev), z4.to(dev))
    b8 = q.w4a8_dequant_int8(wq, s4, z4)
    assert torch.equal(c.cpu().long(), a.long() @ b8.long().T)


@pytest.mark.parametrize("M,N,K,sdt", [(160, 4096, 1024, torch.float16), (200, 520, 3200, torch.float32),
                                       (256, 1032, 2176, torch.bfloat16), (161, 8, 128, torch.float16),
                                       (250, 2048, 8192, torch.float16), (256, 264, 14336, torch.float32),
                                       (130, 4104, 4096, torch.bfloat16),
                                       (17, 14336, 1536, torch.float16), (33, 8, 128, torch.float32), (64, 2048, 7168, torch.float16),
                                       (32, 1600, 16384, torch.bfloat16), (48, 15368, 1408, torch.float32),
                                       # more than 256 tiles of 64 columns, up to 128 rows: the 128-column tile kernel
                                       (97, 9000, 4096, torch.float16), (128, 8200, 4224, torch.float32)])
def test_w4a8_mid_m_fused_tiles_exact_mixed_wrap(dev, M, N, K, sdt):
    """Mid-size M: the tile kernels unpack and dequantise the packed words inside their K loop (no int8 copy of
    W).  Unit block scales, fp32 out, 2 % out-of-contract (s4, z4) pairs: exact integers with the int8 wrap,
    over ragged row and column tiles, K tails, split K (few tiles, long K) and every scale dtype."""
    announce("w4a8 fused tiles exact", M, N, K, sdt)
    lib = _lib.load()
    # these shapes take the fused tile path: their scratch is that of the int8 tile kernels (activation scales,
    # split-K partial sums) with no int8 copy of the weights in front
    assert lib.llmk_gemm_w4a8_workspace_bytes(M, N, K, 128) == lib.llmk_gemm_workspace_bytes(M, N, K)
    torch.manual_seed(M + N)
    wq = torch.randint(0, 16, (N, K), dtype=torch.uint8)
    s4 = torch.randint(1, 9, (N, K // 128), dtype=torch.int8)
    z4 = torch.randint(0, 16, (N, K // 128), dtype=torch.int8)
    wild = torch.rand(N, K // 128) < 0.02
    s4[wild] = torch.randint(-128, 128, (int(wild.sum()),), dtype=torch.int8)
    z4[wild] = torch.randint(-128, 128, (int(wild.sum()),), dtype=torch.int8)
    a = torch.randint(-3, 4, (M, K), dtype=torch.int8)
    ones_a = torch.ones(M, K // 128, dtype=sdt)
    ones_b = torch.ones((N + 127) // 128, K // 128, dtype=sdt)
    packed, _ = bp.pack_rows(wq.numpy(), 4, 32)
    with default_dtype(torch.float32):
        c = w4a8_kernel.w4a8_gemm(a.to(dev), ones_a.to(dev), torch.from_numpy(packed).to(dev), ones_b.to(dev),
                                  s4.to(dev), z4.to(dev))
    b8 = q.w4a8_dequant_int8(wq, s4, z4)
    assert torch.equal(c.cpu().long(), (a.double() @ b8.double().T).long())      # exact: every sum is far below 2^53


WAVE_W4A8 = [
    # every tile shape of the kernel whose waves stream their own K share, with ragged rows and columns and K steps that do
    # not divide by the waves: 16 rows x 16, 32 and 64 columns, then 32, 48 and 64 rows
    (7, 1048, 1152, torch.float16), (16, 4104, 2176, torch.float32), (5, 14344, 1280, torch.bfloat16),
    (31, 6152, 896, torch.float16), (32, 14344, 1152, torch.float32), (47, 4104, 1280, torch.bfloat16),
    (48, 14344, 1152, torch.float16), (64, 6152, 1280, torch.float32), (64, 14344, 1152, torch.bfloat16),
    # four waves, more than one round of workgroups
    (50, 24008, 1152, torch.float16), (95, 28680, 640, torch.float32), (256, 4104, 1152, torch.bfloat16),
    # K slices; tables of more than one round of loads; more K steps than one workgroup takes
    (1, 72, 16384, torch.float16), (40, 264, 33024, torch.float32), (20, 136, 65664, torch.float16), (300, 4104, 1024, torch.float16),
    # 16 rows x 32 columns, one stage; 32 to 64 rows x 16, 48 rows x 32
    (1, 4184, 128, torch.bfloat16), (90, 1352, 256, torch.float32), (34, 4096, 2176, torch.float16), (49, 3096, 2176, torch.bfloat16),
    (33, 31960, 1664, torch.float32)]


@pytest.mark.parametrize("M,N,K,sdt", WAVE_W4A8)
@pytest.mark.parametrize("scratch", [True, False])
def test_w4a8_wave_kernel_exact(dev, M, N, K, sdt, scratch):
    """Unit block scales, fp32 out, wild (s4, z4): exact integers (every sum is below 2^24), with the reported scratch and without."""
    announce("w4a8 wave kernel", M, N, K, sdt, scratch)
    if not scratch and K > 32768:
        pytest.skip("beyond 256 K steps the slices need their sums")
    torch.manual_seed(M * 7 + N)
    wq = torch.randint(0, 16, (N, K), dtype=torch.uint8)
    s4 = torch.randint(-128, 128, (N, K // 128), dtype=torch.int8)
    z4 = torch.randint(-128, 128, (N, K // 128), dtype=torch.int8)
    a = (torch.rand(M, K) < 64.0 / K).to(torch.int8) * torch.randint(-128, 128, (M, K), dtype=torch.int8)   # about 64 nonzeros a row
    ad, packed = a.to(dev), torch.from_numpy(bp.pack_rows(wq.numpy(), 4, 32)[0]).to(dev)
    ones_a, ones_b = torch.ones(M, K // 128, dtype=sdt, device=dev), torch.ones((N + 127) // 128, K // 128, dtype=sdt, device=dev)
    s4d, z4d = s4.to(dev), z4.to(dev)
    c = torch.full((M, N), 7.0, device=dev)
    lib = _lib.load()
    nbytes = lib.llmk_gemm_w4a8_workspace_bytes(M, N, K, 128) if scratch else 0
    ws = torch.empty(max(1, nbytes), dtype=torch.uint8, device=dev)
    _lib.call("llmk_gemm_w4a8", _lib.ptr(ad), _lib.ptr(ones_a), _lib.ptr(packed), _lib.ptr(ones_b), _lib.dt(sdt), _lib.ptr(s4d), _lib.ptr(z4d),
              _lib.ptr(c), _lib.dt(torch.float32), M, N, K, 128, _lib.ptr(ws) if nbytes else None, nbytes, None)
    b8 = q.w4a8_dequant_int8(wq, s4, z4)
    ref = ad.double() @ b8.to(dev).double().T
    assert ref.abs().max() < 2 ** 24
    assert torch.equal(c.double(), ref)


W4A8_ANY_WORDS = [(300, 4104, 1024), (200, 8200, 512), (512, 520, 2048), (100, 264, 33024)]


@pytest.mark.parametrize("M,N,K", W4A8_ANY_WORDS)
def test_w4a8_words_at_any_offset(dev, M, N, K):
    """A view of packed words that starts on 4 bytes only: the two passes, in the scratch that the operator allocates."""
    announce("w4a8 words at any offset", M, N, K)
    torch.manual_seed(M + N)
    wq = torch.randint(0, 16, (N, K), dtype=torch.uint8)
    s4, z4 = (torch.randint(-128, 128, (N, K // 128), dtype=torch.int8) for _ in range(2))
    a = (torch.rand(M, K) < 64.0 / K).to(torch.int8) * torch.randint(-128, 128, (M, K), dtype=torch.int8)
    packed = torch.from_numpy(bp.pack_rows(wq.numpy(), 4, 32)[0])
    words = torch.zeros(packed.numel() + 1, dtype=torch.int32, device=dev)[1:].view(packed.shape)
    words.copy_(packed)
    assert words.data_ptr() % 16 == 4
    ones_a, ones_b = torch.ones(M, K // 128, dtype=torch.float16, device=dev), torch.ones((N + 127) // 128, K // 128, dtype=torch.float16, device=dev)
    with default_dtype(torch.float32):
        c = w4a8_kernel.w4a8_gemm(a.to(dev), ones_a, words, ones_b, s4.to(dev), z4.to(dev))
    ref = a.to(dev).double() @ q.w4a8_dequant_int8(wq, s4, z4).to(dev).double().T
    assert ref.abs().max() < 2 ** 24 and torch.equal(c.double(), ref)


WAVE_8BIT = [
    # every tile shape of the kernel whose waves stream their own K share (eight waves 16 to 64 rows x 16 to 64 columns, four waves
    # 32 to 64 rows x 64), with ragged rows and columns and K steps that do not divide by the waves
    (1, 72, 128), (7, 1051, 1152), (5, 14344, 1280), (16, 28680, 1152), (17, 41, 384), (31, 6152, 896), (33, 2051, 2432), (50, 40, 256),
    (97, 41, 1792), (228, 528, 1536), (509, 144, 1536), (261, 936, 1280), (350, 360, 1408), (495, 328, 1152), (495, 744, 2944),
    (492, 968, 1408), (331, 1392, 2688), (452, 624, 1280), (423, 1232, 1280), (446, 872, 1280), (355, 1104, 1920), (372, 2696, 2688),
    (509, 1712, 1536), (467, 1720, 1920), (508, 792, 6656), (344, 2704, 1792), (504, 4320, 1536), (357, 3424, 3584), (351, 5424, 1280),
    # two stages in flight; K slices (without scratch: a scale table of more than one round of loads, and one that leaves room for one
    # stage only)
    (9, 264, 8192), (40, 136, 66688), (2, 24, 3276800),
    # 48 and 64 rows x 64 columns with eight and with four waves, 48 rows x 32
    (33, 8225, 768), (49, 8203, 3072), (33, 57445, 128), (49, 90485, 128), (33, 5443, 640)]


@pytest.mark.parametrize("M,N,K", WAVE_8BIT)
@pytest.mark.parametrize("kind,sdt", [("fp8", torch.float32), ("i8", torch.float32), ("i8", torch.float16), ("i8", torch.bfloat16),
                                      ("rowcol", torch.float32)])
def test_8bit_wave_kernel_exact(dev, M, N, K, kind, sdt):
    """Whole numbers up to 8, at most 64 of them a row, and power-of-two scales from 1/4 to 4: every sum is a multiple of 2^-4 of at
    most 2^16, exact in fp32 in any order."""
    announce("8-bit wave kernel", M, N, K, kind, sdt)
    gen = torch.Generator(dev).manual_seed(M * 7 + N)
    a = torch.randint(-8, 9, (M, K), generator=gen, device=dev, dtype=torch.int8)
    a *= torch.rand(M, K, generator=gen, device=dev) < 64.0 / K
    a *= a.ne(0).cumsum(1, dtype=torch.int32) <= 64
    b = torch.randint(-8, 9, (N, K), generator=gen, device=dev, dtype=torch.int8)
    pow2 = lambda *shape: torch.exp2(torch.randint(-2, 3, shape, generator=gen, device=dev).float())
    c = torch.full((M, N), 7.0, device=dev)
    nbytes = _lib.load().llmk_gemm_workspace_bytes(M, N, K)
    ws = torch.empty(max(1, nbytes), dtype=torch.uint8, device=dev)
    head, tail = (_lib.ptr(c), _lib.dt(torch.float32)), (M, N, K, _lib.ptr(ws), nbytes, None)
    if kind == "rowcol":
        a_s, b_s, c32 = pow2(M), pow2(N), torch.full((M, N), 7, dtype=torch.int32, device=dev)
        _lib.call("llmk_gemm_i8_rowcol", _lib.ptr(a), _lib.ptr(a_s), _lib.ptr(b), _lib.ptr(b_s), *head, _lib.ptr(c32), *tail)
        sums = torch.zeros(M, N, dtype=torch.float64, device=dev)
        for k in range(0, K, 1 << 17):
            sums += a[:, k:k + (1 << 17)].double() @ b[:, k:k + (1 << 17)].double().T
        assert torch.equal(c32.double(), sums)
        ref = sums * a_s[:, None].double() * b_s.double()
    else:
        a_s, b_s = pow2(M, K // 128), pow2((N + 127) // 128, K // 128)
        ref = torch.zeros(M, N, dtype=torch.float64, device=dev)
        for k in range(0, K, 1 << 17):
            part = slice(k, k + (1 << 17))
            ks = slice(k // 128, (k + (1 << 17)) // 128)
            ref += (a[:, part].double() * a_s[:, ks].double().repeat_interleave(128, 1)) @ \
                   (b[:, part].double() * b_s[:, ks].double().repeat_interleave(128, 1).repeat_interleave(128, 0)[:N]).T
        if kind == "fp8":
            a8, b8 = a.float().to(torch.float8_e4m3fn), b.float().to(torch.float8_e4m3fn)
            call = lambda tail: _lib.call("llmk_gemm_fp8_block", _lib.ptr(a8), _lib.ptr(a_s), _lib.ptr(b8), _lib.ptr(b_s), *head, *tail)
        else:
            a_t, b_t = a_s.to(sdt), b_s.to(sdt)
            call = lambda tail: _lib.call("llmk_gemm_i8_block", _lib.ptr(a), _lib.ptr(a_t), _lib.ptr(b), _lib.ptr(b_t), _lib.dt(sdt), *head, *tail)
        if K > 16384:
            call((M, N, K, None, 0, None))
            assert torch.equal(c.double(), ref)
            c.fill_(7.0)
        call(tail)
    assert torch.equal(c.double(), ref)


@pytest.mark.parametrize("M,N,K", [(5, 1051, 256), (200, 6146, 1024), (96, 4099, 4096), (600, 517, 1024), (700, 4093, 1024),
                                   (1030, 10243, 512), (560, 2053, 8192), (400, 1027, 4096)])
@pytest.mark.parametrize("out", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("kind", ["fp8", "i8", "rowcol"])
def test_8bit_outputs_at_any_alignment(dev, M, N, K, out, kind):
    """Outputs that start one element behind an aligned address, with rows of odd lengths, in every kernel and with K slices: what the
    fp32 sums (exact: see above) round to, and not an element outside."""
    announce("8-bit unaligned outputs", M, N, K, out, kind)
    gen = torch.Generator(dev).manual_seed(M + N)
    a = torch.randint(-8, 9, (M, K), generator=gen, device=dev, dtype=torch.int8)
    a *= torch.rand(M, K, generator=gen, device=dev) < 48.0 / K
    a *= a.ne(0).cumsum(1, dtype=torch.int32) <= 64
    b = torch.randint(-8, 9, (N, K), generator=gen, device=dev, dtype=torch.int8)
    ref = a.double() @ b.double().T
    guard = 32
    buf = torch.full((M * N + 2 * guard,), 77.0, dtype=out, device=dev)
    c = buf[guard + 1:guard + 1 + M * N].view(M, N)
    nbytes = _lib.load().llmk_gemm_workspace_bytes(M, N, K)
    ws = torch.empty(max(1, nbytes), dtype=torch.uint8, device=dev)
    tail = (M, N, K, _lib.ptr(ws), nbytes, None)
    if kind == "rowcol":
        ibuf = torch.full((M * N + 2 * guard,), 77, dtype=torch.int32, device=dev)
        c32 = ibuf[guard + 1:guard + 1 + M * N].view(M, N)
        one_a, one_b = torch.ones(M, device=dev), torch.ones(N, device=dev)
        _lib.call("llmk_gemm_i8_rowcol", _lib.ptr(a), _lib.ptr(one_a), _lib.ptr(b), _lib.ptr(one_b), _lib.ptr(c), _lib.dt(out), _lib.ptr(c32), *tail)
        assert torch.equal(c32.double(), ref)
        assert (ibuf[:guard + 1] == 77).all() and (ibuf[guard + 1 + M * N:] == 77).all()
    else:
        one_a, one_b = torch.ones(M, K // 128, device=dev), torch.ones((N + 127) // 128, K // 128, device=dev)
        if kind == "fp8":
            a8, b8 = a.float().to(torch.float8_e4m3fn), b.float().to(torch.float8_e4m3fn)
            _lib.call("llmk_gemm_fp8_block", _lib.ptr(a8), _lib.ptr(one_a), _lib.ptr(b8), _lib.ptr(one_b), _lib.ptr(c), _lib.dt(out), *tail)
        else:
            _lib.call("llmk_gemm_i8_block", _lib.ptr(a), _lib.ptr(one_a), _lib.ptr(b), _lib.ptr(one_b), _lib.dt(torch.float32), _lib.ptr(c),
                      _lib.dt(out), *tail)
    assert torch.equal(c, ref.to(out))
    assert (buf[:guard + 1] == 77).all() and (buf[guard + 1 + M * N:] == 77).all()


@pytest.mark.parametrize("M,N", [(1290, 16904), (1800, 8456), (2300, 8456), (2811, 8456), (4000, 2048), (900, 28672), (640, 16904)])
def test_large_tile_order_exact(dev, M, N):
    """Tile rows of 256 or 128 that are and are not a multiple of four, several rounds of workgroups and a part of one: every tile
    is computed, and computed once."""
    announce("large tile order", M, N)
    gen = torch.Generator(dev).manual_seed(M + N)
    a = torch.randint(-8, 9, (M, 128), generator=gen, device=dev, dtype=torch.int8)
    b = torch.randint(-8, 9, (N, 128), generator=gen, device=dev, dtype=torch.int8)
    one_a, one_b = torch.ones(M, device=dev), torch.ones(N, device=dev)
    ref = (a.float() @ b.float().T)
    c = torch.full((M, N), 7.5, device=dev)
    _lib.call("llmk_gemm_i8_rowcol", _lib.ptr(a), _lib.ptr(one_a), _lib.ptr(b), _lib.ptr(one_b), _lib.ptr(c), _lib.dt(torch.float32), None, M, N,
              128, None, 0, None)
    assert torch.equal(c, ref)


@pytest.mark.parametrize("M,N,K", [(128, 4096, 4096), (256, 1024, 7168), (512, 4096, 4096), (384, 14336, 4096),
                                   (96, 2056, 14336)])
def test_w4a8_mid_m_fused_tiles(dev, M, N, K):
    """The same path on quantised operands with real scales, against the float64 oracle."""
    announce("w4a8 fused tiles", M, N, K)
    torch.manual_seed(N + K)
    wq, s, s4, z4 = q.w4a8_weight_quant_levels(torch.randn(N, K) * 0.02)
    a, a_s = q.act_quant_int8(torch.randn(M, K).bfloat16(), rounding="up")
    packed, _ = bp.pack_rows(wq.numpy(), 4, 32)
    with default_dtype(torch.bfloat16):
        c = w4a8_kernel.w4a8_gemm(a.to(dev), a_s.to(dev), torch.from_numpy(packed).to(dev), s.to(dev),
                                  s4.to(dev), z4.to(dev), 128, 8, "row")
    assert_close_scaled(c, g.w4a8_gemm(a, a_s, wq, s, s4, z4), what="w4a8 fused tiles")


@pytest.mark.parametrize("sdt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("M,N,K", [(128, 4096, 4096), (200, 520, 3200), (257, 1032, 8192)])
def test_int8_mid_m_scale_dtypes(dev, M, N, K, sdt):
    """Mid-size M, int8 blocks: the kernel stages 16-bit activation scales as they are; every scale dtype gives the
    oracle's result on the same (rounded) scales."""
    announce("int8 mid-M scale dtype", M, N, K, sdt)
    torch.manual_seed(M + K)
    a, a_s = q.act_quant_int8(torch.randn(M, K).bfloat16() * 3)
    b, b_s = q.weight_quant_int8(torch.randn(N, K) * 0.02)
    a_s, b_s = a_s.to(sdt), b_s.to(sdt)
    with default_dtype(torch.float32):
        c = int8_kernel.int8_gemm(a.to(dev), a_s.to(dev), b.to(dev), b_s.to(dev))
    assert_close_scaled(c, g.gemm_blockwise(a, a_s, b, b_s), what="int8 mid-M scales " + str(sdt))


def _random_mid_shapes(n, seed):
    import random
    rnd = random.Random(seed)
    shapes = []
    for _ in range(n):
        M = rnd.choice([65, 66, 96, 127, 128, 129, 160, 255, 256, 257, 300, 384, 511, 512, 513, 700, 1024])
        N = rnd.choice([8, 24, 64, 72, 128, 136, 520, 1000, 2048, 2056, 4096, 4104, 6144])
        K = 128 * rnd.choice([1, 2, 3, 4, 5, 7, 8, 12, 16, 17, 32, 40, 64])
        shapes.append((M, N, K))
    return shapes


@pytest.mark.parametrize("M,N,K", _random_mid_shapes(28, 7) + [
    # 17 to 64 rows: the first rows and both tile heights of the mid-size kernels, K slices, ragged columns, and the shapes
    # on either side of the row and weight-size rules that stay on the weight-streaming kernel or the 64-row tiles
    (17, 14336, 1536), (32, 16384, 1280), (17, 14344, 1408), (32, 4096, 4096), (33, 8, 128), (33, 4104, 4096), (48, 520, 8192),
    (64, 2048, 7168), (64, 15368, 3072), (64, 16392, 1280), (20, 3000, 14336), (64, 1030, 8320), (40, 72, 16384),
    # decode sizes on short K: one to four K steps per wave, whole and partial
    (2, 8, 128), (1, 1000, 1024), (16, 4104, 1152), (5, 520, 2048), (16, 72, 2176), (1, 1000, 3072), (20, 264, 3200), (16, 28680, 1408)])
def test_mid_and_small_tile_kernels_exact_integers(dev, M, N, K):
    """Random mid-size shapes (ragged row and column tiles, K tails, split K, one or more rounds of tiles) with small
    integer operands, unit block scales of a random dtype and fp32 output: the block-scaled int8 and fp8 GEMMs and the
    per-token int8 GEMM must return the exact integer product (every partial sum is below 2^24)."""
    announce("mid-size exact", M, N, K)
    torch.manual_seed(M * 7 + N + K)
    a = torch.randint(-7, 8, (M, K), dtype=torch.int8)
    b = torch.randint(-7, 8, (N, K), dtype=torch.int8)
    ref = (a.double() @ b.double().T).long()
    sdt = [torch.float16, torch.bfloat16, torch.float32][(M + N + K // 128) % 3]
    a_s = torch.ones(M, K // 128, dtype=sdt)
    b_s = torch.ones((N + 127) // 128, K // 128, dtype=sdt)
    with default_dtype(torch.float32):
        c = int8_kernel.int8_gemm(a.to(dev), a_s.to(dev), b.to(dev), b_s.to(dev))
        assert torch.equal(c.cpu().long(), ref), "int8 block"
        # the same integers are exact in e4m3 (|v| <= 7)
        c8 = fp8_kernel.fp8_gemm(a.float().to(torch.float8_e4m3fn).to(dev), a_s.float().to(dev),
                                 b.float().to(torch.float8_e4m3fn).to(dev), b_s.float().to(dev))
        assert torch.equal(c8.cpu().long(), ref), "fp8 block"
        _, acc = int8_kernel.int8_gemm_per_token(a.to(dev), torch.ones(M).to(dev), b.to(dev), torch.ones(N).to(dev),
                                                 return_int32=True)
        assert torch.equal(acc.cpu().long(), ref), "int8 per token"


# shapes that the mid-size kernels run in blocks of tiles an XCD, by the kinds that take them there: two to eight tile rows, both tile heights, 64 and 128
# columns, K slices
MID_BLOCKS = {("fp8", "int8", "per token"): [(97, 5560, 2176), (131, 3312, 1280), (197, 3104, 1280), (270, 3080, 1280), (130, 3904, 1152), (70, 12353, 1280), (506, 3133, 3328)],
              ("fp8", "int8"): [(398, 3352, 5504), (384, 2496, 3840), (145, 5056, 3840), (237, 3384, 7808)],
              ("fp8",): [(65, 8336, 2176), (130, 6616, 640), (261, 3384, 1152), (131, 1048, 12800), (236, 14024, 2176), (259, 10712, 384), (391, 6224, 640), (120, 11331, 4224)],
              ("fp16", "bf16"): [(33, 5360, 1536), (33, 2608, 3072), (68, 7016, 1152), (149, 4400, 2176), (261, 2824, 2176), (65, 13504, 1152), (163, 6632, 1152), (202, 11040, 1152),
                                 (389, 6696, 1152), (33, 8321, 2048)]}


@pytest.mark.parametrize("M,N,K", [(223, 1872, 11392), (97, 5504, 10368), (200, 9473, 2176)] + [c for cases in MID_BLOCKS.values() for c in cases])
def test_mid_size_tiles_in_the_order_of_the_xcds(dev, M, N, K):
    """Column tiles that are no multiple of eight and operands beyond 4 MB: the tiles are dealt to the XCDs in blocks, with one to eight tile rows,
    a ragged last one and K slices.  Small integers: every partial sum is exact, also with fp16 and bf16 activations on 4-bit weights."""
    announce("mid-size tile order", M, N, K)
    gen = torch.Generator(device=dev).manual_seed(M + N + K)
    a = torch.randint(-7, 8, (M, K), device=dev, generator=gen)
    b = torch.randint(-7, 8, (N, K), device=dev, generator=gen)
    ref = a.double() @ b.double().T
    ones, wones = torch.ones(M, K // 128, device=dev), torch.ones((N + 127) // 128, K // 128, device=dev)
    with default_dtype(torch.float32):
        assert torch.equal(int8_kernel.int8_gemm(a.to(torch.int8), ones.half(), b.to(torch.int8), wones.half()).double(), ref), "int8"
        assert torch.equal(fp8_kernel.fp8_gemm(a.float().to(torch.float8_e4m3fn), ones, b.float().to(torch.float8_e4m3fn), wones).double(), ref), "fp8"
        _, acc = int8_kernel.int8_gemm_per_token(a.to(torch.int8), torch.ones(M, device=dev), b.to(torch.int8), torch.ones(N, device=dev), return_int32=True)
        assert torch.equal(acc.double(), ref), "per token"
    nib = (b + 8).view(N, K // 8, 8)                         # element i of a word in bits 4 i .. 4 i + 3
    words = torch.zeros(N, K // 8, dtype=torch.int64, device=dev)
    for i in range(8):
        words |= nib[:, :, i] << (4 * i)
    words = torch.where(words >= 1 << 31, words - (1 << 32), words).to(torch.int32)
    scales = torch.full((N, K // 128), 2.0 ** -10, dtype=torch.float16, device=dev)
    # half a last place of the rounded sum: 11 significant bits in fp16, 8 in bf16, so at most 2^-11 and 2^-8 of the value
    for dt, half in ((torch.float16, 2.0 ** -11), (torch.bfloat16, 2.0 ** -8)):
        y = w4a16.w4a16_gemm(a.to(dt), words, scales, 128).double() * 1024
        assert bool(((y - ref).abs() <= half * ref.abs()).all()), dt


MID_128_COLUMNS = [(130, 9000, 640), (300, 5000, 1152), (500, 3208, 384), (100, 16000, 256), (128, 20000, 640), (236, 14024, 2176), (391, 6224, 640), (65, 8336, 2176)]


@pytest.mark.parametrize("M,N,K", MID_128_COLUMNS + [(256, 14336, 4096), (512, 6144, 8192)])
def test_fp8_one_round_of_128_column_tiles(dev, M, N, K):
    """fp8 block GEMM on weights too wide for the 64-column mid-size kernel that fit one round of 64- or 128-row by
    128-column tiles (the 128-column form of the producer / consumer kernel): ragged rows and columns, odd numbers of
    K blocks.  Small integers with unit scales must come out exactly; quantised random operands within 1e-2 of the
    oracle."""
    announce("fp8 128-column mid-size", M, N, K)
    torch.manual_seed(M + N + K)
    a = torch.randint(-7, 8, (M, K), dtype=torch.int8)
    b = torch.randint(-7, 8, (N, K), dtype=torch.int8)
    with default_dtype(torch.float32):
        c = fp8_kernel.fp8_gemm(a.float().to(torch.float8_e4m3fn).to(dev), torch.ones(M, K // 128).to(dev),
                                b.float().to(torch.float8_e4m3fn).to(dev), torch.ones((N + 127) // 128, K // 128).to(dev))
    assert torch.equal(c.cpu().long(), (a.double() @ b.double().T).long())
    x = torch.randn(M, K).bfloat16()
    w = torch.randn(N, K) * 0.02
    aq, a_s = q.act_quant_fp8(x)
    bq, b_s = q.weight_quant_fp8(w)
    with default_dtype(torch.bfloat16):
        c = fp8_kernel.fp8_gemm(aq.to(dev), a_s.to(dev), bq.to(dev), b_s.to(dev))
    assert_close_scaled(c, g.gemm_blockwise(aq, a_s, bq, b_s), what="fp8 128-column mid-size")


@pytest.mark.parametrize("kind", ["fp8", "int8"])
@pytest.mark.parametrize("M,N,K,out", [(128, 1024, 4096, torch.bfloat16), (200, 520, 3200, torch.float32),
                                       (70, 136, 1152, torch.float16), (300, 2048, 8192, torch.bfloat16),
                                       (48, 2560, 16384, torch.bfloat16), (64, 14336, 4096, torch.float16),
                                       (256, 4096, 14336, torch.bfloat16),
                                       # fp8: K slices of the 128-column form of the mid-size kernel (rows beyond 8 KB on few tiles)
                                       (128, 4096, 14336, torch.bfloat16), (100, 3000, 10240, torch.float32),
                                       (256, 14336, 14336, torch.float16)])
def test_mid_m_split_k_shapes(dev, kind, M, N, K, out):
    """Mid-size M with few column tiles: the K range is split over workgroups (uneven slices included)."""
    announce("split-K", kind, M, N, K, out)
    torch.manual_seed(M + N + K)
    x = torch.randn(M, K).bfloat16()
    w = torch.randn(N, K) * 0.02
    with default_dtype(out):
        if kind == "fp8":
            a, a_s = q.act_quant_fp8(x)
            b, b_s = q.weight_quant_fp8(w)
            c = fp8_kernel.fp8_gemm(a.to(dev), a_s.to(dev), b.to(dev), b_s.to(dev))
        else:
            a, a_s = q.act_quant_int8(x)
            b, b_s = q.weight_quant_int8(w)
            c = int8_kernel.int8_gemm(a.to(dev), a_s.to(dev), b.to(dev), b_s.to(dev))
    assert c.dtype == out
    assert_close_scaled(c, g.gemm_blockwise(a, a_s, b, b_s), what="split-K " + kind)


@pytest.mark.parametrize("kind", ["fp8", "int8"])
@pytest.mark.parametrize("M,N,K,out", [(16, 4096, 14336, torch.bfloat16), (1, 1000, 8192, torch.float32),
                                       (13, 264, 4224, torch.float16), (50, 520, 12416, torch.bfloat16),
                                       (16, 28672, 4224, torch.bfloat16), (33, 136, 16384, torch.float32)])
def test_decode_k_ranges(dev, kind, M, N, K, out):
    """Decode-sized M with K > 4096: the weight-streaming kernel runs on K ranges side by side and a second
    kernel adds the fp32 partial sums (ragged last range, ragged rows and columns included)."""
    announce("K ranges", kind, M, N, K, out)
    torch.manual_seed(M + N + K)
    x = torch.randn(M, K).bfloat16()
    w = torch.randn(N, K) * 0.02
    with default_dtype(out):
        if kind == "fp8":
            a, a_s = q.act_quant_fp8(x)
            b, b_s = q.weight_quant_fp8(w)
            c = fp8_kernel.fp8_gemm(a.to(dev), a_s.to(dev), b.to(dev), b_s.to(dev))
        else:
            a, a_s = q.act_quant_int8(x)
            b, b_s = q.weight_quant_int8(w)
            c = int8_kernel.int8_gemm(a.to(dev), a_s.to(dev), b.to(dev), b_s.to(dev))
    assert c.dtype == out
    assert_close_scaled(c, g.gemm_blockwise(a, a_s, b, b_s), what="K ranges " + kind)


def test_int8_decode_k_ranges_exact(dev):
    """Unit scales, small integers: the sum over K ranges is the exact integer product."""
    announce("K ranges exact")
    torch.manual_seed(9)
    M, N, K = 16, 1032, 12416
    a = torch.randint(-15, 16, (M, K), dtype=torch.int8)
    b = torch.randint(-15, 16, (N, K), dtype=torch.int8)
    a_s = torch.ones(M, K // 128, dtype=torch.float32)
    b_s = torch.ones((N + 127) // 128, K // 128, dtype=torch.float32)
    with default_dtype(torch.float32):
        c = int8_kernel.int8_gemm(a.to(dev), a_s.to(dev), b.to(dev), b_s.to(dev))
    assert torch.equal(c.cpu().long(), a.long() @ b.long().T)


def test_fp8_gemm_without_scratch_takes_the_streaming_kernel(dev):
    """The scratch is optional: the same call without it runs another kernel and agrees with the oracle too."""
    announce("fp8 no scratch")
    torch.manual_seed(5)
    M, N, K = 48, 2560, 8192
    a, a_s = q.act_quant_fp8(torch.randn(M, K).bfloat16())
    b, b_s = q.weight_quant_fp8(torch.randn(N, K) * 0.02)
    ad, asd, bd, bsd = a.to(dev), a_s.to(dev), b.to(dev), b_s.to(dev)
    c = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
    _lib.call("llmk_gemm_fp8_block", _lib.ptr(ad), _lib.ptr(asd), _lib.ptr(bd), _lib.ptr(bsd), _lib.ptr(c),
              _lib.dt(c.dtype), M, N, K, None, 0, _lib.stream(ad))
    ref = g.gemm_blockwise(a, a_s, b, b_s)
    assert_close_scaled(c, ref, what="fp8 without scratch")
    with default_dtype(torch.bfloat16):
        c2 = fp8_kernel.fp8_gemm(ad, asd, bd, bsd)
    assert_close_scaled(c2, ref, what="fp8 with scratch")


@pytest.mark.parametrize("kind", ["fp8", "int8"])
@pytest.mark.parametrize("M,N,K", [(65, 128, 128), (130, 200, 256), (300, 384, 512), (520, 256, 384), (1100, 130, 256)])
def test_tiled_kernels_ragged_shapes(dev, kind, M, N, K):
    """Shapes that exercise every tile height of the large-M kernel, with ragged M and N."""
    announce("tiled ragged", kind, M, N, K)
    torch.manual_seed(M + N + K)
    x = torch.randn(M, K).bfloat16()
    w = torch.randn(N, K) * 0.02
    if kind == "fp8":
        a, a_s = q.act_quant_fp8(x)
        b, b_s = q.weight_quant_fp8(w)
        fn = fp8_kernel.fp8_gemm
    else:
        a, a_s = q.act_quant_int8(x)
        b, b_s = q.weight_quant_int8(w)
        fn = int8_kernel.int8_gemm
    for out in (torch.bfloat16, torch.float32):
        with default_dtype(out):
            c = fn(a.to(dev), a_s.to(dev), b.to(dev), b_s.to(dev))
        assert_close_scaled(c, g.gemm_blockwise(a, a_s, b, b_s), what="tiled %s" % kind)


@pytest.mark.parametrize("kind", ["fp8", "int8", "int8_f32scales"])
@pytest.mark.parametrize("M,N,K", [(4000, 4100, 256), (4096, 4096, 384), (3900, 4352, 128)])
def test_wide_tile_kernel_ragged_shapes(dev, kind, M, N, K):
    """Shapes large enough for the 256 x 256 tile, with ragged M and N, odd and single K step counts."""
    announce("wide ragged", kind, M, N, K)
    torch.manual_seed(M + N + K)
    x = torch.randn(M, K).bfloat16()
    w = torch.randn(N, K) * 0.02
    if kind == "fp8":
        a, a_s = q.act_quant_fp8(x)
        b, b_s = q.weight_quant_fp8(w)
        fn = fp8_kernel.fp8_gemm
    else:
        a, a_s = q.act_quant_int8(x)
        b, b_s = q.weight_quant_int8(w)
        if kind == "int8_f32scales":
            a_s, b_s = a_s.float(), b_s.float()
        fn = int8_kernel.int8_gemm
    ref = g.gemm_blockwise(a, a_s, b, b_s)
    for out in (torch.bfloat16, torch.float32):
        with default_dtype(out):
            c = fn(a.to(dev), a_s.to(dev), b.to(dev), b_s.to(dev))
        assert_close_scaled(c, ref, what="wide %s" % kind)


@pytest.mark.parametrize("kind", ["fp8", "int8"])
@pytest.mark.parametrize("M,N,K,out", [(5120, 10240, 8192, torch.bfloat16), (4096, 4608, 8192, torch.float32),
                                       (5000, 10200, 8192, torch.float16), (1100, 1300, 8192, torch.bfloat16)])
def test_large_tiles_split_last_round(dev, kind, M, N, K, out):
    """Long K and a tile count that leaves a short last round of 256 workgroups: 800 tiles of 256 x 256 (three
    rounds and 32 tiles, split eight ways), 576 tiles of 128 x 256 (two rounds and 64 tiles, split four ways), the
    first again with ragged rows and columns, and a small problem on smaller tiles for contrast.  The tiles of the
    short round are split along K and a second kernel adds the fp32 partial sums.  Every output dtype."""
    announce("split last round", kind, M, N, K, out)
    torch.manual_seed(M + N + K)
    x = torch.randn(M, K).bfloat16()
    w = torch.randn(N, K) * 0.02
    with default_dtype(out):
        if kind == "fp8":
            a, a_s = q.act_quant_fp8(x)
            b, b_s = q.weight_quant_fp8(w)
            c = fp8_kernel.fp8_gemm(a.to(dev), a_s.to(dev), b.to(dev), b_s.to(dev))
        else:
            a, a_s = q.act_quant_int8(x)
            b, b_s = q.weight_quant_int8(w)
            c = int8_kernel.int8_gemm(a.to(dev), a_s.to(dev), b.to(dev), b_s.to(dev))
    assert c.dtype == out
    rows = torch.randperm(M)[:96].sort().values                     # 96 random rows, all columns; every element finite
    assert bool(torch.isfinite(c).all())
    assert_close_scaled(c[rows.to(dev)], g.gemm_blockwise(a[rows], a_s[rows], b, b_s), what="split last round " + kind)
    # all rows: column sums against a one-row oracle GEMM of the scale-weighted column sums of A
    wsum = (a.float().double().reshape(M, K // 128, 128) * a_s.double()[:, :, None]).sum(0).reshape(1, K)
    want = g.gemm_blockwise(wsum, torch.ones(1, K // 128, dtype=torch.float64), b.float(), b_s)[0]
    got = c.double().sum(0).cpu()
    ref_rms = g.gemm_blockwise(a[rows], a_s[rows], b, b_s).pow(2).mean().sqrt().item()
    assert bool(((got - want).abs() <= 1e-2 * ref_rms * (M ** 0.5) + 1e-2 * want.abs()).all()), "column sums"


@pytest.mark.parametrize("M", [1, 40, 65, 600])
def test_empty_sums_are_zero(dev, M):
    """K = 0 through the C ABI: nothing is read, the outputs are zeros (grouped: of the segments' rows)."""
    announce("K = 0", M)
    N = 200
    pad = torch.zeros(1 << 16, dtype=torch.uint8, device=dev)     # operands of no elements, somewhere in memory
    mid = ctypes.c_void_p(pad.data_ptr() + (1 << 15))
    st = _lib.stream(pad)
    for dt in (torch.float32, torch.bfloat16):
        for name, scales in (("llmk_gemm_fp8_block", ()), ("llmk_gemm_i8_block", (_lib.F16,))):
            c = torch.full((M, N), 7.0, dtype=dt, device=dev)
            _lib.call(name, mid, mid, mid, mid, *scales, _lib.ptr(c), _lib.dt(dt), M, N, 0, None, 0, st)
            assert (c == 0).all()
        c, acc = torch.full((M, N), 7.0, dtype=dt, device=dev), torch.full((M, N), 7, dtype=torch.int32, device=dev)
        _lib.call("llmk_gemm_i8_rowcol", mid, mid, mid, mid, _lib.ptr(c), _lib.dt(dt), _lib.ptr(acc), M, N, 0, None, 0, st)
        assert (c == 0).all() and (acc == 0).all()
        for kind, sdt in ((_lib.KIND_I8, _lib.F16), (_lib.KIND_FP8, _lib.F32), (_lib.KIND_BF16, 0)):
            c = torch.full((M + 2, N), 7.0, dtype=dt, device=dev)
            seg = torch.tensor([1, 1 + M // 2, 1 + M // 2, 1 + M], dtype=torch.int64, device=dev)
            _lib.call("llmk_grouped_gemm", mid, mid, _lib.ptr(c), kind, _lib.dt(dt), 3, M + 2, N, 0, _lib.ptr(seg), None, mid, mid, sdt,
                      None, 0, st)
            assert (c[1:-1] == 0).all() and (c[0] == 7).all() and (c[-1] == 7).all()

"""W4A16 GEMMs (simple-Marlin layout `mul`, and the [N, K/8] bit-packed layout) vs the oracle."""
import pytest
import torch

from oracle import gemm_ref as g, marlin_ref as mr, quant_ref as q, bitpack_ref as bp
from llm_kernels_amd.fast_dequant.simple_marlin.utils import QuantUtils
from llm_kernels_amd.fast_dequant.simple_marlin.marlin import mul
from llm_kernels_amd.fast_dequant import w4a16
from llm_kernels_amd import _lib
from helpers import announce, assert_close_scaled

pytestmark = pytest.mark.gpu

# the 14 shapes of the reference's own accuracy test (fast_dequant/simple_marlin/test.py:139-157)
REFERENCE_CASES = [
    (16, 64, 128, 128), (16, 128, 128, 128), (16, 64, 512, 128), (16, 64, 1024, 128),
    (256, 512, 1024, 128), (512, 256, 1024, 128), (1024, 1024, 512, 128), (128, 2048, 1024, 128),
    (1024, 2048, 2048, 128), (2048, 1024, 1024, 128), (512, 4096, 2048, 128),
    (256, 512, 1024, 64), (256, 512, 1024, 256), (512, 512, 512, 512),
]


@pytest.mark.parametrize("M,N,K,groupsize", REFERENCE_CASES)
def test_mul_reference_recipe(dev, M, N, K, groupsize):
    """Recipe of the reference test: seed 42, inputs randn * 0.1, pass = every |diff| <= 0.05."""
    announce("marlin mul", M, N, K, groupsize)
    torch.manual_seed(42)
    A = (torch.randn(M, K) * 0.1).half()
    W = (torch.randn(K, N) * 0.1).half()
    ref_deq, W_int4, scales = mr.fake_quantize(W, groupsize)
    B, sp = mr.pack(W_int4, scales, groupsize)
    C = torch.zeros(M, N, dtype=torch.half, device=dev)
    workspace = torch.zeros(N // 128 * 16 + 16, dtype=torch.int32, device=dev)
    ret = mul(A.to(dev), B.to(dev), C, sp.to(dev), workspace)
    assert ret is None
    ref = g.w4a16_gemm(A, W_int4, scales, groupsize)
    assert (C.cpu().double() - ref).abs().max() <= 0.05            # the reference's acceptance threshold
    assert_close_scaled(C, ref, what="marlin mul")
    assert torch.allclose(ref, A.double() @ ref_deq.double())


def test_mul_quantize_and_pack_on_device(dev):
    announce("marlin device-side pack")
    torch.manual_seed(1)
    M, N, K, g_ = 16, 4096, 4096, 128
    A = torch.randn(M, K, device=dev).half()
    W = (torch.randn(K, N, device=dev) * 0.02).half()
    ref_deq, W_int4, scales = QuantUtils.fake_quantize(W, g_)
    B, sp = QuantUtils.pack(W_int4, scales, g_)
    assert B.shape == (K // 16, 2 * N) and B.dtype == torch.int32 and B.device == W.device
    oB, osp = mr.pack(W_int4.cpu(), scales.cpu(), g_)
    assert torch.equal(B.cpu(), oB) and torch.equal(sp.cpu(), osp)
    C = torch.zeros(M, N, dtype=torch.half, device=dev)
    mul(A, B, C, sp, torch.zeros(512, dtype=torch.int32, device=dev))
    assert_close_scaled(C, A.double().cpu() @ ref_deq.double().cpu(), what="marlin 16x4096x4096")


@pytest.mark.parametrize("M,N,K,groupsize", [(16, 64, 16, 16), (16, 192, 48, 16), (32, 64, 256, 32), (48, 320, 128, -1)])
def test_mul_edge_shapes(dev, M, N, K, groupsize):
    announce("marlin edge", M, N, K, groupsize)
    torch.manual_seed(M + N + K)
    A = (torch.randn(M, K) * 0.5).half()
    W = (torch.randn(K, N) * 0.1).half()
    _, W_int4, scales = mr.fake_quantize(W, groupsize)
    # the kernel reads scales in the grouped permutation; pack with an explicit group size of K for -1
    B, sp = mr.pack(W_int4, scales, K if groupsize == -1 else groupsize)
    C = torch.full((M, N), 7.0, dtype=torch.half, device=dev)
    mul(A.to(dev), B.to(dev), C, sp.to(dev), torch.zeros(64, dtype=torch.int32, device=dev))
    assert_close_scaled(C, g.w4a16_gemm(A, W_int4, scales, groupsize), what="marlin edge")


def test_mul_error_behaviour(dev):
    announce("marlin errors")
    A = torch.zeros(16, 64, dtype=torch.half, device=dev)
    B = torch.zeros(4, 128, dtype=torch.int32, device=dev)
    C = torch.zeros(16, 64, dtype=torch.half, device=dev)
    s = torch.ones(1, 64, dtype=torch.half, device=dev)
    ws = torch.zeros(16, dtype=torch.int32, device=dev)
    with pytest.raises(RuntimeError):
        mul(A[:15], B, C[:15], s, ws)                       # M % 16
    with pytest.raises(RuntimeError):
        mul(A.float(), B, C, s, ws)                         # dtype
    with pytest.raises(RuntimeError):
        mul(A, B.long(), C, s, ws)
    with pytest.raises(RuntimeError):
        mul(A, B, C, s[:, :32].contiguous(), ws)            # scale N mismatch
    with pytest.raises(RuntimeError):
        mul(A, B, C.cpu(), s, ws)                           # device mismatch


# ----------------------------------------------------------------------------- [N, K/8] layout (config 1)
@pytest.mark.parametrize("M,N,K,gs", [(16, 4096, 4096, 128), (1, 64, 128, 128), (7, 100, 256, 64), (16, 256, 512, 32),
                                      (40, 512, 1024, 128), (16, 128, 384, -1), (16, 28672, 4096, 128), (16, 1000, 14336, 128),
                                      (3, 8200, 4096, 256), (32, 4100, 2048, 128), (64, 520, 8192, 128), (33, 4096, 512, 512),
                                      (300, 1000, 512, 64), (4096, 4096, 256, 128), (48, 1000, 12416, 128), (1, 4096, 14336, 128),
                                      (64, 264, 8448, 256), (20, 129, 4224, 128), (16, 264, 8320, 128)])
def test_w4a16_nk(dev, M, N, K, gs):
    announce("w4a16 nk", M, N, K, gs)
    torch.manual_seed(0)
    x = torch.randn(M, K).half()
    w = torch.randn(N, K) * 0.02
    grp = K if gs == -1 else gs
    qn, s = q.w4a16_quant_nk(w, grp)
    packed, _ = bp.pack_cols(qn.numpy(), 4, 32)
    y = w4a16.w4a16_gemm(x.to(dev), torch.from_numpy(packed).to(dev), s.to(dev), gs)
    assert y.dtype == torch.half and y.shape == (M, N)
    ref = g.w4a16_gemm(x, qn.t().int().contiguous(), s.t().contiguous(), grp)
    assert_close_scaled(y, ref, what="w4a16 nk")


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("N,K,gs", [(4096, 4096, 128), (257, 1024, 64), (96, 512, 32), (33, 1024, 512), (5, 64, 8)])
def test_w4a16_nk_device_quantize_round_trip(dev, dtype, N, K, gs):
    """One-pass quantiser of the [N, K/8] layout: codes, scales and packed words bit-exact against the oracle's
    absmax/7 rule and the bit-packing oracle (every division is an IEEE fp32 division on both sides)."""
    announce("w4a16 nk quantize on device", dtype, N, K, gs)
    torch.manual_seed(3)
    from llm_kernels_amd.quantization.bitpack import unpack_over_cols
    w = (torch.randn(N, K) * 0.02).to(dtype)
    w[N // 2, :gs] = 0                                              # a group of zeros: scale 0, codes 8
    packed, s, qd = w4a16.quantize_nk(w.to(dev), gs)
    oq, os_ = q.w4a16_quant_nk(w, gs)
    oq[N // 2, :gs] = 8
    assert packed.shape == (N, K // 8) and packed.dtype == torch.int32
    assert torch.equal(s.cpu(), os_)
    assert torch.equal(qd.cpu(), oq)
    opacked, _ = bp.pack_cols(oq.numpy(), 4, 32)
    assert torch.equal(packed.cpu(), torch.from_numpy(opacked))
    assert torch.equal(unpack_over_cols(packed, 4, K), qd)          # pack/unpack round trip, bit exact


def test_w4a16_nk_device_quantize_refuses_bad_shapes(dev):
    w = torch.randn(16, 256, device=dev)
    with pytest.raises(AssertionError):
        w4a16.quantize_nk(w, 96)                                    # not a divisor of K
    with pytest.raises(AssertionError):
        w4a16.quantize_nk(w[:, :48].contiguous(), 48)               # not a power of two
    with pytest.raises(AssertionError):
        w4a16.quantize_nk(w.double(), 128)


@pytest.mark.parametrize("M,N,K", [(16, 4096, 4096), (32, 1024, 4096), (64, 512, 8192), (16, 256, 14336)])
def test_mul_split_k_is_deterministic_and_rearms(dev, M, N, K):
    """Decode shapes split K over workgroups inside one launch; repeated launches must give identical bits
    (fixed summation order) and leave the ticket counters re-armed."""
    announce("marlin split-k repeat", M, N, K)
    torch.manual_seed(7)
    A = (torch.randn(M, K) * 0.3).half()
    W = (torch.randn(K, N) * 0.05).half()
    _, q, s = mr.fake_quantize(W, 128)
    B, sp = mr.pack(q, s, 128)
    Ag, Bg, sg = A.to(dev), B.to(dev), sp.to(dev)
    ws = torch.zeros(64, dtype=torch.int32, device=dev)
    outs = []
    for _ in range(20):
        C = torch.empty(M, N, dtype=torch.half, device=dev)
        mul(Ag, Bg, C, sg, ws)
        outs.append(C)
    torch.cuda.synchronize()
    for o in outs[1:]:
        assert torch.equal(o, outs[0])
    assert_close_scaled(outs[0], g.w4a16_gemm(A, q, s, 128), what="marlin split-k")


# ------------------------------------------------- compute-bound shapes: dequantise to fp16, then the 256 x 256 tile kernel
@pytest.mark.parametrize("M,N,K,gs", [(4096, 4096, 256, 128), (4000, 4032, 192, 64), (3856, 4160, 64, 16), (4096, 4096, 128, -1)])
def test_mul_large_tile_shapes(dev, M, N, K, gs):
    announce("marlin large tiles", M, N, K, gs)
    torch.manual_seed(M + K)
    A = (torch.randn(M, K) * 0.3).half()
    W = (torch.randn(K, N) * 0.05).half()
    _, q4, s = mr.fake_quantize(W, gs)
    B, sp = mr.pack(q4, s, K if gs == -1 else gs)          # the kernel reads scales in the grouped permutation
    C = torch.zeros(M, N, dtype=torch.half, device=dev)
    mul(A.to(dev), B.to(dev), C, sp.to(dev), torch.zeros(64, dtype=torch.int32, device=dev))
    assert_close_scaled(C, g.w4a16_gemm(A, q4, s, gs), what="marlin large tiles")


@pytest.mark.parametrize("M,N,K,gs", [(80, 192, 192, 64), (128, 4096, 4096, 128), (272, 1088, 8192, -1), (512, 320, 1024, 128),
                                      (96, 28672, 512, 128), (144, 64, 14336, 128), (256, 4160, 2048, 256),
                                      (48, 4096, 14336, 128), (64, 28672, 4096, 128)])
def test_mul_mid_m_fused_tiles(dev, M, N, K, gs):
    """64 < M <= 512, and 32 < M <= 64 with large weights: the tile kernels expand the Marlin units themselves
    (odd chunk counts, one or several K slices, group sizes from 64 to the whole column)."""
    announce("marlin fused tiles", M, N, K, gs)
    torch.manual_seed(M + N + K)
    A = (torch.randn(M, K) * 0.3).half()
    W = (torch.randn(K, N) * 0.05).half()
    _, q4, s = mr.fake_quantize(W, gs)
    B, sp = mr.pack(q4, s, K if gs == -1 else gs)
    C = torch.zeros(M, N, dtype=torch.half, device=dev)
    mul(A.to(dev), B.to(dev), C, sp.to(dev), torch.zeros(64, dtype=torch.int32, device=dev))
    assert_close_scaled(C, g.w4a16_gemm(A, q4, s, gs), what="marlin fused tiles")


@pytest.mark.parametrize("M,N,K,gs", [(65, 136, 128, 64), (128, 4096, 4096, 128), (200, 1000, 1152, 128), (256, 520, 8192, 256),
                                      (512, 264, 2048, 64), (100, 129, 14336, -1), (130, 4100, 4224, 128), (96, 28672, 1024, 128),
                                      (48, 4096, 14336, 128), (64, 28672, 4096, 128), (33, 2400, 14336, 256),
                                      # one round of 128-column tiles of the producer / consumer kernel: 64- and 128-row tiles,
                                      # ragged rows and columns, groups of 64 and of the whole row
                                      (130, 9000, 640, 64), (300, 5000, 1152, 128), (100, 16000, 256, -1), (128, 20000, 384, 64),
                                      (128, 14336, 4096, 128)])
def test_w4a16_nk_mid_m_fused_tiles(dev, M, N, K, gs):
    """64 < M <= 512, and 32 < M <= 64 with large weights: the tile kernels expand the packed words themselves
    (one or several K slices, ragged rows and columns, group sizes from 64 to the whole row)."""
    announce("w4a16 nk fused tiles", M, N, K, gs)
    torch.manual_seed(M + N + K)
    x = torch.randn(M, K).half()
    w = torch.randn(N, K) * 0.02
    grp = K if gs == -1 else gs
    qn, s = q.w4a16_quant_nk(w, grp)
    packed, _ = bp.pack_cols(qn.numpy(), 4, 32)
    y = w4a16.w4a16_gemm(x.to(dev), torch.from_numpy(packed).to(dev), s.to(dev), gs)
    assert y.dtype == torch.half and y.shape == (M, N)
    ref = g.w4a16_gemm(x, qn.t().int().contiguous(), s.t().contiguous(), grp)
    assert_close_scaled(y, ref, what="w4a16 nk fused tiles")


@pytest.mark.parametrize("M,N,K,gs", [(2300, 14400, 384, 128), (4100, 8200, 128, 64), (2560, 14336, 256, 128),
                                      (600, 61000, 640, 64)])
def test_w4a16_nk_fused_256_column_tiles(dev, M, N, K, gs):
    """More than 512 rows and two or more rounds of 256 x 256 tiles: the packed words are expanded inside the
    256-column tile kernel (two, four, six and ten K steps of 64: from no steady-state step to eight; ragged rows
    and columns; groups of one K step and of two)."""
    announce("w4a16 nk fused 256-column tiles", M, N, K, gs)
    torch.manual_seed(M + N + K)
    x = torch.randn(M, K).half()
    w = torch.randn(N, K) * 0.02
    qn, s = q.w4a16_quant_nk(w, gs)
    packed, _ = bp.pack_cols(qn.numpy(), 4, 32)
    y = w4a16.w4a16_gemm(x.to(dev), torch.from_numpy(packed).to(dev), s.to(dev), gs)
    assert y.dtype == torch.half and y.shape == (M, N)
    ref = g.w4a16_gemm(x, qn.t().int().contiguous(), s.t().contiguous(), gs)
    assert_close_scaled(y, ref, what="w4a16 nk fused 256-column tiles")


@pytest.mark.parametrize("M,N,K,gs", [(4096, 4096, 256, 128), (3990, 4100, 384, 64), (4096, 3848, 128, 32)])
def test_w4a16_nk_large_tile_shapes(dev, M, N, K, gs):
    announce("w4a16 nk large tiles", M, N, K, gs)
    torch.manual_seed(N + K)
    x = torch.randn(M, K).half()
    w = torch.randn(N, K) * 0.02
    qn, s = q.w4a16_quant_nk(w, gs)
    packed, _ = bp.pack_cols(qn.numpy(), 4, 32)
    y = w4a16.w4a16_gemm(x.to(dev), torch.from_numpy(packed).to(dev), s.to(dev), gs)
    ref = g.w4a16_gemm(x, qn.t().int().contiguous(), s.t().contiguous(), gs)
    assert_close_scaled(y, ref, what="w4a16 nk large tiles")


WITHOUT_SCRATCH = [(128, 1024, 4096), (48, 4096, 14336), (300, 520, 1152), (16, 264, 8320), (49, 4160, 9472)]


@pytest.mark.parametrize("M,N,K", WITHOUT_SCRATCH)
def test_w4a16_without_scratch(dev, M, N, K):
    """The scratch of both w4a16 entry points is optional: without it the kernels run with one K slice (or the
    weight-streaming variant) and must agree with the oracle all the same."""
    announce("w4a16 without scratch", M, N, K)
    torch.manual_seed(M + N)
    x = torch.randn(M, K).half()
    qn, s = q.w4a16_quant_nk(torch.randn(N, K) * 0.02, 128)
    packed, _ = bp.pack_cols(qn.numpy(), 4, 32)
    xd, pd, sd = x.to(dev), torch.from_numpy(packed).to(dev), s.to(dev)
    y = torch.empty(M, N, dtype=torch.half, device=dev)
    _lib.call("llmk_gemm_w4a16_nk", _lib.ptr(xd), _lib.ptr(pd), _lib.ptr(y), _lib.ptr(sd), _lib.dt(xd.dtype),
              M, N, K, 128, None, 0, _lib.stream(xd))
    assert_close_scaled(y, g.w4a16_gemm(x, qn.t().int().contiguous(), s.t().contiguous(), 128), what="nk without scratch")
    if M % 16 == 0 and N % 64 == 0:
        A = (torch.randn(M, K) * 0.3).half()
        W = (torch.randn(K, N) * 0.05).half()
        _, q4, sm = mr.fake_quantize(W, 128)
        B, sp = mr.pack(q4, sm, 128)
        Ad, Bd, spd = A.to(dev), B.to(dev), sp.to(dev)
        C = torch.zeros(M, N, dtype=torch.half, device=dev)
        _lib.call("llmk_gemm_w4a16_marlin", _lib.ptr(Ad), _lib.ptr(Bd), _lib.ptr(C), _lib.ptr(spd),
                  M, N, K, 128, None, 0, _lib.stream(Ad))
        assert_close_scaled(C, g.w4a16_gemm(A, q4, sm, 128), what="marlin without scratch")


@pytest.mark.parametrize("M,N,K,gs", [(16, 4096, 4096, 128), (1, 256, 512, 128), (7, 1000, 1024, 128), (40, 520, 2048, 128),
                                      (16, 28672, 4096, 128), (16, 1032, 14336, 128), (64, 264, 8192, 128),
                                      (16, 256, 384, 128), (33, 300, 4608, 128), (16, 512, 1024, 64), (20, 129, 512, 256),
                                      (300, 1000, 512, 128), (2048, 4096, 1024, 128),
                                      # K > 4096 with M * N not a multiple of 4: the ring kernel's summing pass does not take it
                                      (1, 1001, 8192, 128), (3, 50257, 8192, 128)])
def test_w4a16_nk_bf16(dev, M, N, K, gs):
    """bf16 activations / outputs for the [N, K/8] layout: the weight-streaming kernel at decode sizes (128-wide
    groups, whole four-step K shares), the bf16 copy of W plus the bf16 tile GEMM everywhere else."""
    announce("w4a16 nk bf16", M, N, K, gs)
    torch.manual_seed(2)
    x = torch.randn(M, K).bfloat16()
    w = torch.randn(N, K) * 0.02
    qn, s = q.w4a16_quant_nk(w, gs)
    packed, _ = bp.pack_cols(qn.numpy(), 4, 32)
    y = w4a16.w4a16_gemm(x.to(dev), torch.from_numpy(packed).to(dev), s.to(dev), gs)
    assert y.dtype == torch.bfloat16 and y.shape == (M, N)
    deq = (qn.double() - 8) * s.double().repeat_interleave(gs, 1)            # [N, K], exact
    assert_close_scaled(y, x.double() @ deq.T, what="w4a16 nk bf16")


def test_w4a16_nk_bf16_decode_is_exact_for_small_integers(dev):
    """Integer activations, unit scales: the bf16 decode kernel (nibbles as 128 + q, the -136 * sum(a) bias in the
    accumulator) returns the exact integer product wherever it is representable in bf16."""
    announce("w4a16 nk bf16 exact")
    torch.manual_seed(3)
    M, N, K = 16, 512, 1024
    x = torch.randint(-2, 3, (M, K)).float()
    qn = torch.randint(0, 16, (N, K), dtype=torch.uint8)
    s = torch.ones(N, K // 128, dtype=torch.float16)
    packed, _ = bp.pack_cols(qn.numpy(), 4, 32)
    y = w4a16.w4a16_gemm(x.bfloat16().to(dev), torch.from_numpy(packed).to(dev), s.to(dev), 128)
    ref = x.double() @ (qn.double() - 8).T
    assert torch.equal(y.cpu().double(), ref.bfloat16().double())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(1, 8, 512), (3, 40, 640), (16, 1000, 768), (17, 136, 896), (64, 264, 1408), (5, 5000, 3968),
                                   (4, 72, 4224), (64, 136, 8320), (3, 4672, 9088)])
def test_w4a16_nk_decode_any_number_of_steps(dev, dtype, M, N, K):
    """K ranges of the ring kernel that are no multiple of its waves' four-step shares, one range and several of unequal
    length, scale rows at every two-byte offset.  Small integers and power-of-two scales: every sum is exact in fp32, so the
    result is the rounded product (bf16 via -136 biases included).  fp16: an infinite activation reaches its own row only."""
    announce("w4a16 nk decode steps", dtype, M, N, K)
    torch.manual_seed(M + N + K)
    x = torch.randint(-2, 3, (M, K)).to(dtype)
    qn = torch.randint(0, 16, (N, K), dtype=torch.uint8)
    s = torch.exp2(torch.randint(-4, 1, (N, K // 128)).float()).half()
    packed = torch.from_numpy(bp.pack_cols(qn.numpy(), 4, 32)[0]).to(dev)
    w = (qn.double() - 8) * s.double().repeat_interleave(128, 1)
    y = w4a16.w4a16_gemm(x.to(dev), packed, s.to(dev), 128)
    assert torch.equal(y.cpu(), (x.double() @ w.T).to(dtype))
    if dtype == torch.float16:
        x[0, K - 1] = float("inf")
        y = w4a16.w4a16_gemm(x.to(dev), packed, s.to(dev), 128).cpu()
        ref = (x.double() @ w.T).to(dtype)
        assert torch.equal(y[1:], ref[1:]) and torch.equal(y[0].isnan(), ref[0].isnan())
        assert torch.equal(y[0].nan_to_num(0.0), ref[0].nan_to_num(0.0))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(1, 8, 4096), (17, 136, 4096), (64, 2600, 4096), (64, 5000, 4096), (16, 1000, 8192), (3, 72, 12288)])
def test_w4a16_nk_decode_full_ranges(dev, dtype, M, N, K):
    """Ranges of 32 steps, the form of the ring kernel without shares to move: every ring depth, one range and several."""
    test_w4a16_nk_decode_any_number_of_steps(dev, dtype, M, N, K)


# every tile shape of the kernels whose waves stream their own K share: 16 to 64 rows x 16 to 64 columns of a workgroup, four and
# eight waves, ragged rows and columns, fewer K steps than waves, K slices; then groups of several K steps
WAVE_NK = [(17, 8200, 4224, 128), (64, 8200, 128, 128), (33, 20008, 128, 128), (33, 8200, 8320, 128), (65, 8, 256, 128),
           (97, 1032, 1152, 128), (65, 3000, 640, 128), (128, 520, 256, 128), (65, 2056, 1152, 128), (70, 4104, 896, 128),
           (97, 1032, 384, 128), (250, 1032, 640, 128), (100, 4104, 1024, 128), (97, 3000, 896, 128), (49, 12296, 640, 128),
           (17, 12296, 128, 128), (33, 4104, 4224, 128), (31, 14344, 1152, 128), (40, 6152, 2176, 128), (49, 14344, 896, 128),
           (160, 1032, 640, 128), (100, 6152, 1024, 128), (97, 1000, 1152, 384), (80, 520, 2048, -1),
           # the tiles that only exact weights or only rounded ones of the two types get with shapes like these
           (34, 4096, 2176, 128), (33, 31960, 1664, 128), (17, 64, 4224, 128), (17, 2096, 4224, 128), (49, 7312, 512, 128),
           (33, 2112, 4224, 128), (49, 3096, 2176, 128), (49, 4248, 9344, 128), (66, 64, 2176, 128), (17, 34824, 128, 128),
           (162, 1352, 512, 128), (33, 2768, 4352, 128), (17, 8312, 4224, 128), (33, 4104, 4224, 128)]
WAVE_MARLIN = [(32, 8256, 128, 128), (16, 4160, 8320, 128), (64, 12352, 128, 128), (32, 4160, 8320, 128), (48, 14400, 128, 128),
               (48, 8256, 8320, 128), (16, 64, 128, 128), (16, 64, 8320, 128), (16, 4160, 128, 128), (48, 576, 8320, 128),
               (16, 8256, 1152, 128), (32, 2112, 1152, 128), (32, 4160, 1152, 128), (32, 14400, 128, 128), (48, 3008, 1152, 128),
               (256, 1088, 640, 128), (144, 576, 8320, 128), (48, 8256, 640, 128), (128, 1088, 8320, 128), (64, 8256, 640, 128),
               (512, 1088, 640, 128), (80, 320, 1152, 384), (32, 192, 2048, 2048)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,gs", WAVE_NK)
def test_w4a16_nk_wave_kernel(dev, dtype, M, N, K, gs):
    """Small integers and power-of-two scales: every sum is exact in fp32, so the result is the rounded product; then an
    infinite activation reaches its own row only (fp16)."""
    announce("w4a16 nk wave kernel", dtype, M, N, K, gs)
    torch.manual_seed(M + N + K)
    g_ = K if gs == -1 else gs
    x = torch.randint(-2, 3, (M, K), device=dev).to(dtype)
    qn = torch.randint(0, 16, (N, K), dtype=torch.uint8)
    s = torch.exp2(torch.randint(-4, 1, (N, K // g_)).float()).half().to(dev)
    packed = torch.from_numpy(bp.pack_cols(qn.numpy(), 4, 32)[0]).to(dev)
    w = ((qn.to(dev).double() - 8) * s.double().repeat_interleave(g_, 1)).T.contiguous()
    assert torch.equal(w4a16.w4a16_gemm(x, packed, s, gs), (x.double() @ w).to(dtype))
    if dtype == torch.float16:
        x[1, K - 1] = float("inf")
        y, ref = w4a16.w4a16_gemm(x, packed, s, gs), (x.double() @ w).to(dtype)
        assert torch.equal(y[:1], ref[:1]) and torch.equal(y[2:], ref[2:]) and torch.equal(y[1].isfinite(), ref[1].isfinite())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,gs", [(64, 8193, 128, 128), (33, 8193, 256, 256), (80, 1025, 256, 128), (97, 4097, 384, 128), (65, 33, 128, 128),
                                      (97, 1025, 1152, -1), (160, 1026, 640, 640), (65, 3001, 640, 128), (100, 2051, 128, 128)])
def test_w4a16_nk_wave_kernel_last_columns(dev, dtype, M, N, K, gs):
    """A last tile of one to three columns and one to five groups: its few scales, at the very end of the table, reach their columns."""
    test_w4a16_nk_wave_kernel(dev, dtype, M, N, K, gs)


@pytest.mark.parametrize("M,N,K,gs", WAVE_MARLIN)
@pytest.mark.parametrize("scratch", [True, False])
def test_mul_wave_kernel(dev, M, N, K, gs, scratch):
    """The same on Marlin words, with the scratch that is reported and without any."""
    announce("marlin wave kernel", M, N, K, gs, scratch)
    torch.manual_seed(M + N + K)
    A = torch.randint(-2, 3, (M, K), device=dev).half()
    qw = torch.randint(0, 16, (K, N), dtype=torch.int32, device=dev)
    s = torch.exp2(torch.randint(-4, 1, (K // gs, N), device=dev).float()).half()
    B, sp = QuantUtils.pack(qw, s, gs)
    C = torch.full((M, N), 7.0, dtype=torch.half, device=dev)
    nbytes = _lib.load().llmk_gemm_w4a16_marlin_workspace_bytes(M, N, K) if scratch else 0
    ws = torch.full((nbytes + 256,), 0x5A, dtype=torch.uint8, device=dev)
    _lib.call("llmk_gemm_w4a16_marlin", _lib.ptr(A), _lib.ptr(B), _lib.ptr(C), _lib.ptr(sp), M, N, K, gs, _lib.ptr(ws) if nbytes else None, nbytes,
              _lib.stream(A))
    ref = A.double() @ ((qw.double() - 8) * s.double().repeat_interleave(gs, 0))
    assert torch.equal(C, ref.half())
    assert (ws[nbytes:] == 0x5A).all()


@pytest.mark.parametrize("M,N,K,gs", [(16, 192, 1152, 384), (16, 64, 8576, 8576), (16, 1088, 3840, 640), (16, 128, 17024, 128), (16, 4160, 2304, 768),
                                      (48, 192, 1152, 384), (64, 576, 8960, 1280)])
def test_mul_wave_kernel_groups(dev, M, N, K, gs):
    """Groups of any number of K steps, cut by waves and by K slices: every step finds its group."""
    test_mul_wave_kernel(dev, M, N, K, gs, True)
    test_mul_wave_kernel(dev, M, N, K, gs, False)


def _row_differences(M, K, gs, dev, dtype):
    """One +1 and one -1 a row, in the same group of K: the product is the difference of two weights of a column, exact in fp32."""
    x = torch.zeros(M, K, dtype=dtype, device=dev)
    m, g0 = torch.arange(M, device=dev), torch.randint(0, K // gs, (M,), device=dev) * gs
    i = torch.randint(0, gs, (M,), device=dev)
    x[m, g0 + i] = 1.0
    x[m, g0 + (i + 1 + torch.randint(0, gs - 1, (M,), device=dev)) % gs] = -1.0
    return x


@pytest.mark.parametrize("M,N,K,gs", [(16, 4096, 4096, 128), (16, 64, 8320, 128), (48, 8256, 640, 128), (64, 12352, 128, 128), (80, 320, 1152, 384),
                                      (256, 1088, 640, 128), (512, 4096, 1024, 128), (528, 1088, 640, 128)])
def test_mul_multiplies_the_fake_quantised_weights(dev, M, N, K, gs):
    """Whatever the number of rows: (q - 8) * s rounded to fp16 once, as fake_quantize gives it and the reference's kernel forms it."""
    announce("marlin weights", M, N, K, gs)
    torch.manual_seed(M + N + K)
    W, qw, s = QuantUtils.fake_quantize((torch.randn(K, N, device=dev) * 0.02).half(), gs)
    A = _row_differences(M, K, gs, dev, torch.float16)
    C = torch.full((M, N), 7.0, dtype=torch.half, device=dev)
    B, sp = QuantUtils.pack(qw, s, gs)
    mul(A, B, C, sp, torch.zeros(N // 128 * 16 + 16, dtype=torch.int32, device=dev))
    assert torch.equal(C, (A.double() @ W.double()).half())


@pytest.mark.parametrize("M,N,K,gs", [(48, 4096, 8192, 128), (65, 2056, 1152, 128), (100, 4104, 1024, 128), (97, 1000, 1024, 256), (250, 1032, 640, 128),
                                      (512, 4096, 1024, 128), (520, 1032, 640, 128)])
def test_w4a16_nk_rounded_weights(dev, M, N, K, gs):
    """fp16 beyond 64 rows (and from 33 on large weights): the weights rounded to fp16 in whichever kernel is taken."""
    announce("w4a16 nk weights", M, N, K, gs)
    torch.manual_seed(M + N + K)
    packed, s, qn = w4a16.quantize_nk((torch.randn(N, K, device=dev) * 0.02).half(), gs)
    W = ((qn.float() - 8).half() * s.repeat_interleave(gs, 1)).T.contiguous()
    x = _row_differences(M, K, gs, dev, torch.float16)
    assert torch.equal(w4a16.w4a16_gemm(x, packed, s, gs), (x.double() @ W.double()).half())


@pytest.mark.parametrize("M,N,K,gs", [(33, 20008, 128, 128), (40, 14344, 256, 128), (64, 8200, 384, 128), (31, 4104, 1152, 384), (97, 1032, 640, 128)])
def test_w4a16_nk_bf16_infinite_activations(dev, M, N, K, gs):
    """bf16 calls outside the ring kernel's shapes (128-wide groups, at least 512 of K): an infinite activation is an infinite output
    of its sign, or NaN where the weight is zero, and reaches its own row only."""
    announce("w4a16 nk bf16 infinities", M, N, K, gs)
    torch.manual_seed(M + N + K)
    x = torch.randint(-2, 3, (M, K), device=dev).to(torch.bfloat16)
    qn = torch.randint(0, 16, (N, K), dtype=torch.uint8)
    s = torch.exp2(torch.randint(-4, 1, (N, K // gs)).float()).half().to(dev)
    packed = torch.from_numpy(bp.pack_cols(qn.numpy(), 4, 32)[0]).to(dev)
    w = ((qn.to(dev).double() - 8) * s.double().repeat_interleave(gs, 1)).T.contiguous()
    x[1, K - 1], x[2, 5] = float("inf"), float("-inf")
    ref = (x.double() @ w).to(torch.bfloat16)
    assert torch.allclose(w4a16.w4a16_gemm(x, packed, s, gs).float(), ref.float(), rtol=0, atol=0, equal_nan=True)


@pytest.mark.parametrize("M,N,K,gs", [(65, 72, 128, 64), (130, 4096, 1024, 128), (512, 264, 4096, 128), (300, 14344, 512, 128),
                                      (200, 20000, 640, 128), (500, 8192, 384, 192), (600, 10000, 1024, 128), (1024, 28672, 256, 128)])
def test_w4a16_nk_bf16_expanding_tiles(dev, M, N, K, gs):
    """bf16 on the tile kernels that expand the words: both column widths, K slices, groups that are no power of two, the
    256-column tiles, ragged rows and columns; single weights exactly (one activation per row, no sum to round)."""
    announce("w4a16 nk bf16 tiles", M, N, K, gs)
    torch.manual_seed(M + N)
    x = torch.randn(M, K).bfloat16()
    qn, s = q.w4a16_quant_nk(torch.randn(N, K) * 0.02, gs)
    packed, s = torch.from_numpy(bp.pack_cols(qn.numpy(), 4, 32)[0]).to(dev), s.to(dev)
    y = w4a16.w4a16_gemm(x.to(dev), packed, s, gs)
    deq = (qn.double() - 8) * s.cpu().double().repeat_interleave(gs, 1)
    # the weights this path multiplies are (q - 8) * s rounded to bf16: against those only the output's rounding (2^-9 of
    # it) and fp32 sums are left.  Against unrounded weights every product is off by up to 2^-9 too, and of 29 M sums of
    # 256 such errors (0.0011 of the output scale each) three lie nine deviations out, at the 1e-2 bound.
    assert_close_scaled(y, x.double() @ deq.bfloat16().double().T, rtol=2 ** -8, atol=1e-4, what="w4a16 nk bf16 tiles")
    one = torch.zeros(M, K)
    k = torch.randint(0, K, (M,))
    one[torch.arange(M), k] = 1.0
    y = w4a16.w4a16_gemm(one.bfloat16().to(dev), packed, s, gs)
    assert torch.equal(y.cpu(), deq.bfloat16().T[k])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M", [80, 300, 512])
def test_w4a16_nk_expanding_tiles_hold_no_copy_of_the_weights(dev, dtype, M):
    """The tiles that expand the packed words need room for split-K partial sums at most, not for a 16-bit copy of W."""
    N, K = 14336, 4096
    announce("w4a16_nk scratch", dtype, M, N, K)
    torch.manual_seed(0)
    packed, s, _ = w4a16.quantize_nk((torch.randn(N, K, device=dev) * 0.02).to(dtype), 128)
    _lib.release_workspaces()
    w4a16.w4a16_gemm(torch.randn(M, K, device=dev).to(dtype), packed, s, 128)
    torch.cuda.synchronize()
    assert sum(t.numel() for t in _lib._ws.values()) < N * K * 2


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,gs", [(16, 256, 4096, 128), (16, 256, 8192, 128), (40, 512, 4736, 128), (64, 9216, 4608, 128),
                                      (33, 25600, 4096, 128), (48, 4096, 14336, 128), (100, 384, 2048, 64), (80, 512, 1024, 32),
                                      (520, 1024, 1024, 128), (1300, 512, 512, 128)])
def test_w4a16_nk_reported_scratch_is_what_the_call_uses(dev, dtype, M, N, K, gs):
    """The reported number of bytes gives the bits that any larger workspace gives, and nothing behind it is written."""
    announce("w4a16_nk reported scratch", dtype, M, N, K, gs)
    torch.manual_seed(M + N)
    x = torch.randn(M, K, device=dev).to(dtype)
    packed, s, _ = w4a16.quantize_nk(torch.randn(N, K, device=dev) * 0.02, gs)
    need = _lib.load().llmk_gemm_w4a16_nk_workspace_bytes(M, N, K, gs, _lib.dt(dtype))
    room = max(need, N * K * 2 + 8 * M * N * 4) + 256
    guard = torch.full((room + 256,), 0x5A, dtype=torch.uint8, device=dev)
    outs = []
    for n in (need, room):
        y = torch.empty(M, N, dtype=dtype, device=dev)
        _lib.call("llmk_gemm_w4a16_nk", _lib.ptr(x), _lib.ptr(packed), _lib.ptr(y), _lib.ptr(s), _lib.dt(dtype), M, N, K, gs,
                  _lib.ptr(guard) if n else None, n, _lib.stream(x))
        torch.cuda.synchronize()
        assert (guard[n:] == 0x5A).all()
        outs.append(y)
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))

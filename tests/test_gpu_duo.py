"""The tile kernel whose two wave groups take turns (gemm_duo.hpp), on every tile height that is built: numbers of 128-byte sub-blocks around its
loop of four and below it, one to six K slices, ragged rows and columns."""
import ctypes
import random

import pytest
import torch

from llm_kernels_amd import _lib
from llm_kernels_amd.fast_dequant import w4a16
from llm_kernels_amd.fast_dequant.simple_marlin.marlin import mul
from llm_kernels_amd.fast_dequant.simple_marlin.utils import QuantUtils
from llm_kernels_amd.moe.group_gemm_kernel import grouped_gemm_triton
from llm_kernels_amd.quantization import fp8_kernel, int8_kernel, w4a8_kernel
from helpers import announce, assert_close_scaled, default_dtype
from test_gpu_moe import GROUPED_DUO

FP8 = [(138, 11136, 128), (136, 11557, 256), (167, 11056, 384), (131, 10896, 640), (133, 11096, 768), (137, 11553, 896), (162, 11128, 1024), (131, 11616, 1152),
       (142, 11264, 1280), (140, 11184, 1408), (751, 216, 3072), (572, 229, 4224), (1777, 224, 4224), (194, 11816, 1024), (209, 11291, 1152), (198, 11448, 1280),
       (195, 11104, 1408), (2028, 392, 6144), (130, 21768, 1152), (153, 22459, 1280),
       (129, 22056, 1408), (129, 22198, 1536), (131, 22127, 1664), (129, 16472, 1920), (130, 16472, 3072), (1111, 4001, 4224)]
INT8 = [(133, 11136, 640), (138, 11373, 768), (141, 11744, 896), (135, 11040, 1152), (137, 11968, 1408), (2044, 456, 6144), (667, 216, 3072), (937, 381, 4224),
        (197, 11248, 3072), (198, 11051, 4224), (129, 22921, 768), (131, 22120, 1152), (147, 21854, 1280), (160, 23189, 1408), (145, 23239, 1536),
        (145, 8197, 7680), (1210, 4090, 4096)]
PER_TOKEN = [(524, 3632, 1536), (519, 3607, 1152), (526, 248, 3072), (1011, 375, 4224), (289, 8424, 3072), (291, 8344, 4224), (2042, 407, 6144), (386, 9363, 768),
             (452, 8391, 1152), (590, 6536, 1408)]
PER_TOKEN_LONG = [(705, 1112, 10240), (887, 1856, 10752), (1260, 1904, 13696), (1099, 1528, 10496)]       # K slices beyond 512 rows and K = 8192
W4A8 = [(538, 248, 1024), (543, 328, 1152), (581, 232, 1280), (530, 232, 1408), (545, 224, 1536), (676, 200, 1664), (541, 256, 4224), (576, 976, 4224), (194, 11280, 1024),
        (198, 11008, 1152), (221, 10912, 1280), (195, 11544, 1408), (203, 7088, 6144), (1375, 272, 6144), (1636, 552, 4224), (79, 28672, 4096),
        (68, 19016, 1024), (65, 13184, 1152), (71, 14352, 1280), (68, 16264, 1408), (593, 72, 3968), (824, 112, 2304), (792, 80, 2560)]
MARLIN = [(208, 8576, 768), (208, 8320, 640), (560, 2304, 4096), (576, 192, 1536), (528, 192, 1664), (544, 192, 2176), (800, 320, 4224), (528, 5440, 1024),
          (528, 5632, 896), (208, 6784, 4224), (1168, 576, 4224), (1424, 320, 4224), (448, 8832, 512), (400, 8576, 640), (160, 7424, 4224)]
W4 = [(1081, 224, 128), (1465, 208, 256), (1054, 224, 384), (566, 216, 1152), (537, 240, 1280), (659, 208, 2176), (850, 280, 4224), (1849, 1552, 384), (1080, 2704, 512),
      (865, 1104, 4224), (1029, 3664, 128), (1538, 2456, 256), (1160, 3208, 384), (300, 14336, 4096), (148, 6672, 4224), (1605, 2952, 128), (979, 4728, 256),
      (983, 4688, 384), (990, 4688, 512), (169, 6408, 6144), (1802, 1072, 128), (1803, 1064, 256), (66, 17144, 384), (65, 22424, 512), (1064, 2720, 128),
      (1155, 2464, 256), (65, 17696, 512), (684, 72, 640), (1842, 1544, 640), (1744, 1672, 768), (130, 22552, 128), (135, 22336, 256), (132, 22680, 384), (132, 22112, 512),
      (129, 16800, 640), (322, 11008, 256), (325, 10952, 384), (324, 11256, 512)]
# (M, N, K, group) beside groups of 128: half of one to a whole row, K slices that start inside a group, and tiles of 96 to 192 rows
W4_GROUPS = [(66, 8328, 1024, 64), (68, 80, 6144, 64), (620, 888, 1536, 256), (621, 64, 2048, 256), (535, 64, 1536, 256), (678, 1296, 2048, 1024), (965, 400, 4096, 1024),
             (621, 64, 2048, 1024), (69, 20440, 1024, 1024), (621, 64, 2048, 2048), (169, 6408, 6144, 64), (169, 6408, 6144, 1024), (300, 14336, 4096, 4096)]
# those of them that other kernels take, being faster: few short tiles (us, others | this kernel: w4a8 1718 x 160 x 1152 9.6 | 10.7, fp16 1240 x 72 x 640
# 7.6 | 8.6), and in one of the two activation types the tiles of 16-bit or 128-column kernels
ELSEWHERE = {"w4a8": [*W4A8[:6], (1636, 552, 4224)],
             "fp16": [*W4[:3], (1029, 3664, 128), (1538, 2456, 256), (65, 17696, 512), (684, 72, 640), (130, 22552, 128), (135, 22336, 256), (132, 22680, 384),
                      (132, 22112, 512), (322, 11008, 256), (325, 10952, 384), (324, 11256, 512)],
             "bf16": [*W4[:3], (1849, 1552, 384), (1029, 3664, 128), (1538, 2456, 256), (1605, 2952, 128), (979, 4728, 256), (983, 4688, 384), (990, 4688, 512),
                      (1064, 2720, 128), (1155, 2464, 256)]}


def shape(entry, *args):
    out = (ctypes.c_int32 * 2)()
    return (out[0], out[1]) if getattr(_lib.load(), entry)(*args, ctypes.cast(out, ctypes.c_void_p)) else None


def shape8(kind, per_token, M, N, K):
    return shape("llmk_gemm_8bit_duo_shape", kind, per_token, M, N, K, _lib.load().llmk_gemm_workspace_bytes(M, N, K))


def shape_w4a8(M, N, K):
    return shape("llmk_gemm_w4a8_duo_shape", M, N, K, 128, _lib.load().llmk_gemm_w4a8_workspace_bytes(M, N, K, 128))


def shape_w4a16(marlin, dtype, group, *case):
    scratch = _lib.load().llmk_gemm_w4a16_marlin_workspace_bytes(*case) if marlin else _lib.load().llmk_gemm_w4a16_nk_workspace_bytes(*case, group, dtype)
    return shape("llmk_gemm_w4a16_duo_shape", marlin, dtype, *case, group, scratch)


PLANS = (("fp8", FP8, 1, {96, 128, 160}, lambda *c: shape8(_lib.KIND_FP8, 0, *c)), ("int8", INT8, 1, {96, 128, 160}, lambda *c: shape8(_lib.KIND_I8, 0, *c)),
         ("per token", PER_TOKEN, 1, {96, 128, 160}, lambda *c: shape8(_lib.KIND_I8, 1, *c)), ("w4a8", W4A8, 1, {96, 128}, shape_w4a8),
         ("marlin", MARLIN, 2, {96, 128, 160}, lambda *c: shape_w4a16(1, _lib.F16, 128, *c)),
         ("fp16", W4, 2, {96, 128, 160, 192}, lambda *c: shape_w4a16(0, _lib.F16, 128, *c)), ("bf16", W4, 2, {96, 128, 160, 192}, lambda *c: shape_w4a16(0, _lib.BF16, 128, *c)))


def test_the_cases_reach_every_tile():
    """Every height, with one and with several slices, and every remainder of a slice's sub-blocks by the loop's four."""
    for kind, cases, size, heights, plan in PLANS:
        got = {c: plan(*c) for c in cases}
        assert {c for c in cases if not got[c]} == set(ELSEWHERE.get(kind, ())), (kind, got)
        got = {c: p for c, p in got.items() if p}
        assert {rows for rows, _ in got.values()} == heights and {z > 1 for _, z in got.values()} == {False, True}, (kind, got)
        assert {-(-c[2] * size // 128 // z) % 4 for c, (_, z) in got.items()} == {0, 1, 2, 3}, (kind, got)


def test_the_groups_reach_the_kernel():
    plans = {(*c, dt): shape_w4a16(0, dt, c[3], *c[:3]) for c in W4_GROUPS for dt in (_lib.F16, _lib.BF16)}
    assert None not in plans.values() and {p[0] for p in plans.values()} == {96, 160, 192}, plans
    inside = {g for (M, N, K, g, _), (_, z) in plans.items() if z > 1 and -(-(K // 64) // z) * 64 % g}
    assert inside == {256, 1024, 2048} and {g for (M, N, K, g, _), (_, z) in plans.items() if z == 1} == {64, 256, 1024, 4096}, plans


def test_calls_that_are_faster_elsewhere():
    """Shapes that were measured slower on this kernel, and neighbours that are faster on it: short K on one row tile of int8 weights from HBM, more than a round of
    workgroups up to 512 rows, 256-row tiles of 4-bit weights beyond a round, few short tiles of two passes."""
    plan = {kind: p for kind, _, _, _, p in PLANS}
    for kind, case, took in (("int8", (97, 20048, 1664), False), ("int8", (111, 18304, 1664), False), ("per token", (131, 19264, 1664), False), ("per token", (150, 17248, 1792), False),
                             ("fp8", (130, 16472, 3072), True), ("int8", (97, 20048, 3200), True), ("per token", (159, 17248, 3200), True),
                             ("per token", (500, 17848, 11904), False), ("fp8", (289, 23480, 2304), False), ("fp8", (129, 16472, 1920), True),
                             ("fp16", (976, 10616, 7168), False), ("fp16", (201, 23784, 9728), False), ("bf16", (1384, 7224, 9344), False), ("marlin", (432, 13056, 9472), False),
                             ("marlin", (1920, 4544, 3968), False), ("fp16", (300, 14336, 4096), True), ("bf16", (300, 14336, 4096), True),
                             ("w4a8", (1718, 160, 1152), False), ("w4a8", (3723, 112, 1664), False), ("w4a8", (1024, 4096, 4096), True),
                             ("fp16", (1240, 72, 640), False), ("fp16", (2007, 440, 2048), False), ("bf16", (1027, 208, 1024), False), ("fp16", (1086, 536, 6016), True)):
        assert (plan[kind](*case) is not None) == took, (kind, case)


def test_scratch_of_its_slices_is_reported_and_small():
    """What is reported holds the planes of the slices, and for the 8-bit products never more than the array that serves calls without scratch."""
    for _, cases, _, _, plan in PLANS[:3]:
        for M, N, K in cases:
            z = plan(M, N, K)[1]
            assert 4 * z * M * N * (z > 1) <= _lib.load().llmk_gemm_workspace_bytes(M, N, K) <= 32 << 20, (M, N, K)
    for M, N, K in set(W4A8) - set(ELSEWHERE["w4a8"]):
        z = shape_w4a8(M, N, K)[1]
        assert 4 * z * M * N * (z > 1) <= _lib.load().llmk_gemm_w4a8_workspace_bytes(M, N, K, 128)


def test_grouped_cases_reach_every_tile():
    """The heights of the grouped form; not where an expert's rows are two 64-row tiles that leave CUs free: those stream the weights on twice as many
    (8 experts of 592 x 6912, 684 rows 29.7 us from HBM, 37.0 on the tall tiles)."""
    rows = lambda E, M, N, K: _lib.load().llmk_grouped_gemm_duo_rows(E, M, N, K)
    for height, cases in GROUPED_DUO.items():
        assert {rows(E, n * E + max(0, 42 - n), N, K) for E, n, N, K in cases} == {height}, cases
        assert {K // 128 % 4 for _, _, _, K in cases} == {0, 1, 2, 3}, cases
    for E, M, N, K in ((8, 684, 592, 6912), (2, 167, 1448, 9856), (9, 809, 664, 5760), (7, 619, 1992, 7936), (3, 254, 992, 8576)):
        assert rows(E, M, N, K) == 0, (E, M, N, K)
    for E, M, N, K, height in ((8, 362, 4096, 14336, 64), (8, 512, 4096, 14336, 96), (8, 645, 4096, 14336, 128), (8, 860, 4096, 14336, 128), (3, 166, 304, 5760, 96)):
        assert rows(E, M, N, K) == height, (E, M, N, K)


def test_per_token_scratch():
    """What is reported for a per-token product beyond 512 rows is what its K slices take, without the 64 MiB of a split last round, and the plan it gives
    is the one that any amount gives."""
    lib, rng = _lib.load(), random.Random(3)
    slices = 0
    for M, N, K in PER_TOKEN_LONG + [(rng.randint(513, 4096), rng.randint(64, 28672), 128 * rng.randint(1, 112)) for _ in range(3000)]:
        got = lib.llmk_gemm_i8_rowcol_workspace_bytes(M, N, K)
        plan = shape("llmk_gemm_8bit_duo_shape", _lib.KIND_I8, 1, M, N, K, got)
        assert plan == shape("llmk_gemm_8bit_duo_shape", _lib.KIND_I8, 1, M, N, K, 1 << 40), (M, N, K)
        assert got == (4 * plan[1] * M * N if plan and plan[1] > 1 else 0) <= lib.llmk_gemm_workspace_bytes(M, N, K), (M, N, K)
        slices += got > 0 and K >= 8192
    assert slices > 20
    for M, N, K in ((16, 4096, 14336), (64, 4096, 4096), (300, 4096, 14336), (512, 1112, 10240)):
        assert 0 < lib.llmk_gemm_i8_rowcol_workspace_bytes(M, N, K) <= lib.llmk_gemm_workspace_bytes(M, N, K), (M, N, K)


def test_grouped_scratch():
    """Scales that have to be widened and, from 513 rows and K = 8192, a split last round: nothing else."""
    need = _lib.load().llmk_grouped_gemm_workspace_bytes
    for kind in (_lib.KIND_I8, _lib.KIND_FP8):
        assert need(kind, _lib.F32, 4000, 4096, 8064) == need(kind, _lib.F32, 512, 4096, 14336) == 0
        assert need(kind, _lib.F16, 4000, 4096, 4096) == need(kind, _lib.BF16, 4000, 4096, 4096) == 4000 * 32 * 4
        assert need(kind, _lib.F32, 513, 4096, 8192) == 64 << 20 and need(kind, _lib.F16, 640, 4096, 8192) == (64 << 20) + 640 * 64 * 4
    assert need(_lib.KIND_F16, 0, 4000, 4096, 14336) == need(_lib.KIND_BF16, 0, 4000, 4096, 14336) == 0


@pytest.mark.gpu
def test_public_functions_reserve_what_they_use(dev):
    """The scratch that is kept after a call: the planes of a per-token product's slices, nothing for a grouped one that needs none."""
    announce("scratch of the public functions")
    M, N, K = 887, 1856, 10752
    _lib.release_workspaces()
    int8_kernel.int8_gemm_per_token(torch.zeros(M, K, dtype=torch.int8, device=dev), torch.ones(M, device=dev), torch.zeros(N, K, dtype=torch.int8, device=dev),
                                    torch.ones(N, device=dev))
    rows, z = shape("llmk_gemm_8bit_duo_shape", _lib.KIND_I8, 1, M, N, K, 1 << 40)
    assert z > 1 and [4 * z * M * N <= t.numel() < 64 << 20 for t in _lib._ws.values()] == [True]
    _lib.release_workspaces()
    E, M, N, K = 4, 900, 512, 1024
    grouped_gemm_triton(torch.zeros(M, K, dtype=torch.int8, device=dev), torch.zeros(E, N, K, dtype=torch.int8, device=dev), torch.empty(M, N, dtype=torch.bfloat16, device=dev),
                        E, True, torch.tensor([0, 200, 450, 700, M], device=dev), torch.arange(E, device=dev), False, torch.ones(M, K // 128, device=dev),
                        torch.ones(E, N // 128, K // 128, device=dev), [128, 128])
    assert not _lib._ws


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
@pytest.mark.parametrize("M,N,K", PER_TOKEN + PER_TOKEN_LONG)
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
@pytest.mark.parametrize("M,N,K,scales", [(*c, (torch.float16, torch.bfloat16, torch.float32)[i % 3]) for i, c in enumerate(W4A8)])
def test_two_level_weights_exact(dev, M, N, K, scales):
    """Weights int8(int8(q - z4) * s4) of any scale and zero point, wrap included, under powers of two: exact in fp32.  Tables at any offset, and words
    that are not 16-byte aligned, which go another way with the reported scratch."""
    announce("duo w4a8", M, N, K, scales)
    gen = torch.Generator(device=dev).manual_seed(M + K)
    kb = K // 128
    a, q = _ints(gen, dev, -3, 3, M, K), _ints(gen, dev, 0, 15, N, K)
    near = _ints(gen, dev, 0, 7, N, kb) > 0                  # mostly small weights, so that the sums stay below 2^24
    s4, z4 = torch.where(near, _ints(gen, dev, -1, 2, N, kb), _ints(gen, dev, -128, 127, N, kb)), torch.where(near, _ints(gen, dev, 0, 15, N, kb), _ints(gen, dev, -128, 127, N, kb))
    wide = lambda t: t.repeat_interleave(128, 1)
    b = ((q - wide(z4)).to(torch.int8).int() * wide(s4).int()).to(torch.int8)
    a_s, b_s = (2.0 ** _ints(gen, dev, 0, 1, M, kb)).to(scales), (2.0 ** _ints(gen, dev, 0, 1, -(-N // 128), kb)).to(scales)
    ref = (a.double() * wide(a_s.double())) @ (b.double() * wide(b_s.double()).repeat_interleave(128, 0)[:N]).t()
    assert ref.abs().max() < 1 << 24
    packed = torch.zeros(N // 8, K, dtype=torch.int64, device=dev)
    for i in range(8):
        packed |= q[i::8].long() << (4 * i)
    packed = torch.where(packed >= 1 << 31, packed - (1 << 32), packed).int()
    a8, bytes4 = a.to(torch.int8), torch.empty(2, N * kb + 1, dtype=torch.int8, device=dev)
    bytes4[0, 1:], bytes4[1, 1:] = s4.to(torch.int8).flatten(), z4.to(torch.int8).flatten()
    scratch = _lib.load().llmk_gemm_w4a8_workspace_bytes(M, N, K, 128)
    ws = torch.empty(max(scratch, 16), dtype=torch.uint8, device=dev)
    odd = torch.empty(N // 8 * K + 1, dtype=torch.int32, device=dev)[1:].copy_(packed.flatten())
    for words in (packed, odd):
        for room in (scratch, 0):
            if room < N * K and (words is odd or not shape("llmk_gemm_w4a8_duo_shape", M, N, K, 128, room)):
                continue                                     # (the expanded copy of the weights needs its scratch)
            out = torch.full((M, N), float("nan"), device=dev)
            _lib.call("llmk_gemm_w4a8", _lib.ptr(a8), _lib.ptr(a_s), _lib.ptr(words), _lib.ptr(b_s), _lib.dt(scales), _lib.ptr(bytes4[0, 1:]), _lib.ptr(bytes4[1, 1:]),
                      _lib.ptr(out), _lib.F32, M, N, K, 128, _lib.ptr(ws) if room else None, room, _lib.stream(a8))
            assert torch.equal(out.double(), ref), (room, words is odd)


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


def _packed_rows(codes):
    """[N, K] codes -> [N, K/8] words, element i of a word in bits 4 i .. 4 i + 3."""
    words = torch.zeros(codes.shape[0], codes.shape[1] // 8, dtype=torch.int64, device=codes.device)
    for i in range(8):
        words |= codes[:, i::8].long() << (4 * i)
    return torch.where(words >= 1 << 31, words - (1 << 32), words).int()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,group", W4_GROUPS)
def test_row_packed_groups(dev, M, N, K, group, dtype):
    """Every group has a scale of its own: one element of a row gives a column of the rounded weights, to the bit, over all of K."""
    announce("duo w4 groups", dtype, M, N, K, group)
    gen = torch.Generator(device=dev).manual_seed(M + K + group)
    codes, scales = _ints(gen, dev, 0, 15, N, K), (torch.rand(N, K // group, device=dev, generator=gen, dtype=torch.float32) * 0.02 + 0.001).half()
    weights = ((codes.float() - 8) * scales.float().repeat_interleave(group, 1)).to(dtype)
    packed = _packed_rows(codes)
    k = (max(7, K // M | 1) * torch.arange(M, device=dev) + 3) % K
    x = torch.zeros(M, K, dtype=dtype, device=dev)
    x[torch.arange(M, device=dev), k] = 1
    assert torch.equal(w4a16.w4a16_gemm(x, packed, scales, group), weights[:, k].t())
    x = torch.randn(M, K, device=dev, generator=gen, dtype=torch.float32).to(dtype)
    assert_close_scaled(w4a16.w4a16_gemm(x, packed, scales, group), x.double() @ weights.double().t(), rtol=2 ** -8 if dtype == torch.bfloat16 else 2 ** -11, atol=2e-5)


NAN, INF = float("nan"), float("inf")


def _only_their_rows(call, clean, dirty, rows, ref):
    """Rows with values that are no numbers: what `ref` says is NaN or infinite is, and the other rows are what they are without them."""
    before, after = call(clean), call(dirty)
    others = torch.ones(before.shape[0], dtype=torch.bool, device=before.device)
    others[list(rows)] = False
    assert bool(before.isfinite().all()) and torch.equal(before[others], after[others])
    got, want = after[list(rows)].cpu().double(), ref.cpu()
    assert torch.equal(got.isnan(), want.isnan()) and not bool(want.isfinite().all(1).any())
    for inf in (INF, -INF):
        assert torch.equal(got == inf, want == inf)


@pytest.mark.gpu
@pytest.mark.parametrize("kind,M,N,K", [("fp8", 751, 216, 3072), ("fp8", 131, 11616, 1152), ("fp8", 198, 11448, 1280), ("fp8", 129, 16472, 1920), ("int8", 667, 216, 3072),
                                        ("int8", 137, 11968, 1408), ("int8", 197, 11248, 3072), ("int8", 147, 21854, 1280), ("w4a8", 541, 256, 4224), ("w4a8", 203, 7088, 6144)])
def test_scales_that_are_no_numbers(dev, kind, M, N, K):
    """NaN and infinities among the activation scales (and, for fp8, the activations), in the first and the last K step: in their rows and nowhere else."""
    announce("duo non-finite", kind, M, N, K)
    assert {k: p for k, _, _, _, p in PLANS}[kind](M, N, K)
    gen = torch.Generator(device=dev).manual_seed(M + K)
    kb = K // 128
    a, b = _ints(gen, dev, -3, 3, M, K), _ints(gen, dev, -3, 3, N, K)
    scales = torch.float32 if kind == "fp8" else torch.float16
    a_s, b_s = (2.0 ** _ints(gen, dev, 0, 3, M, kb)).to(scales), (2.0 ** _ints(gen, dev, 0, 3, -(-N // 128), kb)).to(scales)
    a8 = a.float().to(torch.float8_e4m3fn) if kind == "fp8" else a.to(torch.int8)
    bad_a, bad_s = a8.clone(), a_s.clone()
    rows = [0, 17, 64, M - 1]
    bad_s[0, 0], bad_s[17, kb - 1], bad_s[64, kb // 2], bad_s[M - 1, kb - 1] = INF, -INF, NAN, INF
    if kind == "fp8":
        rows.append(40)
        bad_a[40, K - 1] = NAN
    ref = sum((bad_a[rows, 128 * i:128 * i + 128].float().double() @ b[:, 128 * i:128 * i + 128].double().t()) *
              (bad_s[rows, i:i + 1].double() * b_s[:, i].double().repeat_interleave(128)[:N]) for i in range(kb))
    if kind == "w4a8":
        one = torch.ones(N, kb, dtype=torch.int8, device=dev)
        words = _packed_rows((b + 8).t().contiguous()).t().contiguous()
        call = lambda v: w4a8_kernel.w4a8_gemm(*v, words, b_s, one, 8 * one, 128, 8, "row")
    else:
        b8 = b.float().to(torch.float8_e4m3fn) if kind == "fp8" else b.to(torch.int8)
        call = lambda v: (fp8_kernel.fp8_gemm if kind == "fp8" else int8_kernel.int8_gemm)(*v, b8, b_s)
    with default_dtype(torch.float32):
        _only_their_rows(call, (a8, a_s), (bad_a, bad_s), rows, ref)


@pytest.mark.gpu
@pytest.mark.parametrize("kind,M,N,K", [("fp16", 659, 208, 2176), ("fp16", 865, 1104, 4224), ("fp16", 1605, 2952, 128), ("bf16", 659, 208, 2176), ("bf16", 300, 14336, 4096),
                                        ("bf16", 169, 6408, 6144), ("marlin", 576, 192, 1536), ("marlin", 528, 5632, 896), ("marlin", 400, 8576, 640)])
def test_activations_that_are_no_numbers(dev, kind, M, N, K):
    """The same for 16-bit activations: infinities times the weights' signs, times a zero weight NaN."""
    announce("duo non-finite", kind, M, N, K)
    assert {k: p for k, _, _, _, p in PLANS}[kind](M, N, K)
    gen = torch.Generator(device=dev).manual_seed(M + K)
    dtype = torch.bfloat16 if kind == "bf16" else torch.float16
    x = torch.randn(M, K, device=dev, generator=gen, dtype=torch.float32).to(dtype)
    bad, rows = x.clone(), [0, 17, 64, M - 1]
    bad[0, 0], bad[17, K - 1], bad[64, K // 2], bad[M - 1, K - 1] = INF, -INF, NAN, INF
    if kind == "marlin":
        _, q, s = QuantUtils.fake_quantize((torch.randn(K, N, device=dev, generator=gen, dtype=torch.float32) * 0.02).half(), 128)
        weights = ((q.double() - 8) * s.double().repeat_interleave(128, 0)).t()
        words, s = QuantUtils.pack(q, s, 128)

        def call(v):
            out = torch.empty(M, N, dtype=dtype, device=dev)
            mul(v, words, out, s, torch.zeros(max(16, N // 128 * 16), dtype=torch.int32, device=dev))
            return out
    else:
        codes, scales = _ints(gen, dev, 0, 15, N, K), (torch.rand(N, K // 128, device=dev, generator=gen, dtype=torch.float32) * 0.01 + 0.001).half()
        weights, words = (codes.double() - 8) * scales.double().repeat_interleave(128, 1), _packed_rows(codes)
        call = lambda v: w4a16.w4a16_gemm(v, words, scales, 128)
    _only_their_rows(call, x, bad, rows, bad[rows].cpu().double() @ weights.cpu().t())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,group", [(*c, (128, 64, 256)[i % 3] if c[2] % 256 == 0 else (128, 64)[i % 2]) for i, c in enumerate(MARLIN)])
def test_marlin_words(dev, M, N, K, group):
    """As for the row-packed layout."""
    announce("duo marlin", M, N, K, group)
    gen = torch.Generator(device=dev).manual_seed(M + K)
    ref, q, s = QuantUtils.fake_quantize((torch.randn(K, N, device=dev, generator=gen, dtype=torch.float32) * 0.02).half(), group)
    words, scales = QuantUtils.pack(q, s, group)
    weights = ((q.float() - 8) * s.float().repeat_interleave(group, 0)).half()
    assert torch.equal(weights, ref)
    out = torch.full((M, N), float("nan"), dtype=torch.float16, device=dev)
    workspace = torch.zeros(max(16, N // 128 * 16), dtype=torch.int32, device=dev)
    k = (7 * torch.arange(M, device=dev) + 3) % K
    x = torch.zeros(M, K, dtype=torch.float16, device=dev)
    x[torch.arange(M, device=dev), k] = 1
    mul(x, words, out, scales, workspace)
    assert torch.equal(out, weights[k])
    x = torch.randn(M, K, device=dev, generator=gen, dtype=torch.float32).half()
    mul(x, words, out, scales, workspace)
    assert_close_scaled(out, x.double() @ weights.double(), rtol=2 ** -11, atol=2e-5)

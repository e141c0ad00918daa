"""The shapes of the GPU tests of the kernels whose waves stream their own K share reach every tile that these kernels are built with."""
import ctypes

import torch

from llm_kernels_amd import _lib
from test_gpu_duo import shape8, shape_w4a16
from test_gpu_gemm import MID_128_COLUMNS, MID_BLOCKS, W4A8_ANY_WORDS, WAVE_8BIT, WAVE_W4A8
from test_gpu_w4a16 import WAVE_MARLIN, WAVE_NK, WITHOUT_SCRATCH

MUCH = 1 << 50


def shape(name, *args):
    """(waves, 16-row tiles, 16-column tiles, form) of a call, or None where it goes to another kernel."""
    out = (ctypes.c_int32 * 5)()
    if not getattr(_lib.load(), "llmk_gemm_%s_wave_shape" % name)(*args, ctypes.cast(out, ctypes.c_void_p)):
        return None
    return out[0], out[1], out[2], out[4]


def eight(form, *but):
    """Eight waves, 16 to 64 rows x 16, 32 or 64 columns."""
    return {(8, mt, nt, form) for mt in (1, 2, 3, 4) for nt in (1, 2, 4) if (mt, nt) not in but}


def four(form, *mt):
    return {(4, m, 4, form) for m in mt}


def test_8bit():
    built = eight(1, (3, 1), (4, 1)) | four(1, 2, 3, 4) | {(8, 1, 1, 2)}
    for kind, per_token in ((_lib.KIND_FP8, 0), (_lib.KIND_I8, 0), (_lib.KIND_I8, 1)):
        got = set()
        for M, N, K in WAVE_8BIT:
            got.add(shape("8bit", kind, per_token, M, N, K, _lib.load().llmk_gemm_workspace_bytes(M, N, K)))
        assert got - {None} == built, (kind, per_token, built - got)


def test_w4a8():
    built = eight(1) | four(1, 3, 4) | {(8, 1, 1, 2), (8, 1, 2, 2)}
    got = {shape("w4a8", M, N, K, 128, scratch) for M, N, K, _ in WAVE_W4A8 for scratch in (MUCH, 0)}
    assert got - {None} == built, built - got


def test_w4a16():
    got = {shape("w4a16", 1, _lib.F16, M, N, K, gs, scratch) for M, N, K, gs in WAVE_MARLIN for scratch in (MUCH, 0)}
    built = eight(1, (4, 1), (4, 2)) | four(1, 1, 2, 3)
    assert got - {None} == built, ("marlin", built - got)
    for dt, built in ((_lib.F16, eight(0, (1, 4), (4, 1)) | four(0, 1, 2, 3) | eight(1) | four(1, 1, 2, 3)),
                      (_lib.BF16, eight(0, (4, 1)) | four(0, 1, 2, 3) | eight(1, (1, 2), (1, 4)) | four(1, 2, 3))):
        got = {shape("w4a16", 0, dt, M, N, K, gs, MUCH) for M, N, K, gs in WAVE_NK}
        got |= {shape("w4a16", 0, dt, M, N, K, 128, 0) for M, N, K in WITHOUT_SCRATCH if dt == _lib.F16}
        assert got - {None} == built, (dt, built - got, got - built)


def test_8bit_second_stage():
    """Two stages where one workgroup a CU has nothing else to cover the latency of a wave's second K step, one from there on and for 9
    rows and more on weights of 16 MB."""
    for kind, per_token in ((_lib.KIND_FP8, 0), (_lib.KIND_I8, 0), (_lib.KIND_I8, 1)):
        stages = lambda M, N, K: shape("8bit", kind, per_token, M, N, K, 0)[::3]
        for M, N, K in ((1, 4096, 4096), (8, 4096, 4096), (2, 2408, 3072), (16, 4096, 1152), (1, 2616, 4096), (16, 4088, 4096)):
            assert stages(M, N, K) == (8, 2), (kind, per_token, M, N, K)
        for M, N, K in ((1, 4097, 4096), (1, 6144, 4096), (1, 4096, 1024), (9, 4096, 4096), (16, 4096, 4096)):
            assert stages(M, N, K) == (8, 1), (kind, per_token, M, N, K)


def test_8bit_columns_of_a_decode_tile():
    """Weight-bound calls of 9 to 16 rows: 32 columns from 20480 columns on, with K of 4096 or more from 13 rows."""
    for kind, per_token in ((_lib.KIND_FP8, 0), (_lib.KIND_I8, 0), (_lib.KIND_I8, 1)):
        columns = lambda M, N, K: 16 * shape("8bit", kind, per_token, M, N, K, 0)[2]
        for M, N, K in ((9, 28672, 4096), (12, 57344, 4096), (16, 18000, 4096), (9, 18000, 4096), (14, 20000, 4096)):
            assert columns(M, N, K) == 16, (kind, per_token, M, N, K)
        for M, N, K in ((16, 28672, 4096), (13, 24576, 4096), (16, 128256, 4096), (10, 24000, 2304)):
            assert columns(M, N, K) == 32, (kind, per_token, M, N, K)


def test_8bit_beyond_64_rows():
    """Large weights from HBM: the tile kernels, which were 1.15 to 1.24 times as fast there, also for 65 to 128 rows and for per-token
    scales; small ones stay with the waves."""
    much = lambda kind, per_token, M, N, K: shape("8bit", kind, per_token, M, N, K, _lib.load().llmk_gemm_workspace_bytes(M, N, K))
    assert much(_lib.KIND_I8, 0, 90, 14336, 4096) is None
    assert much(_lib.KIND_I8, 1, 81, 21672, 3584) is None and much(_lib.KIND_I8, 1, 427, 5424, 14208) is None
    assert much(_lib.KIND_I8, 1, 300, 4096, 14336) is None and much(_lib.KIND_I8, 0, 128, 4096, 14336) is None
    assert much(_lib.KIND_I8, 1, 400, 1030, 9088) and much(_lib.KIND_I8, 0, 205, 1296, 8960)
    assert much(_lib.KIND_I8, 1, 337, 3592, 4608) and much(_lib.KIND_FP8, 0, 200, 1032, 7168) and much(_lib.KIND_I8, 0, 128, 2048, 4096)


def test_w4a8_reports_the_two_passes():
    """Where the operator has always had scratch for an expanded copy, words that are not 16-byte aligned rely on it."""
    for M, N, K in W4A8_ANY_WORDS:
        assert shape("w4a8", M, N, K, 128, MUCH) and _lib.load().llmk_gemm_w4a8_workspace_bytes(M, N, K, 128) >= N * K


def test_offsets_and_grids_of_very_wide_weights():
    """Marlin strips and groups beyond 32-bit offsets, and grids of 2^32 threads or more, are not taken."""
    marlin = lambda N, K, gs: shape("w4a16", 1, _lib.F16, 16, N, K, gs, MUCH)
    assert marlin((1 << 26) - 64, 128, 128) and not marlin(1 << 26, 128, 128)
    assert marlin(1 << 24, 16384 - 128, 128) and not marlin(1 << 24, 16384, 128) and marlin(1 << 24, 16384, 256)
    for N in (1 << 27, (1 << 27) + 1, 1 << 29, (1 << 31) - 1):
        for M in (1, 16, 64, 512):
            calls = [(N, shape("8bit", kind, per_token, M, N, 128, MUCH)) for kind, per_token in ((_lib.KIND_FP8, 0), (_lib.KIND_I8, 0), (_lib.KIND_I8, 1))]
            calls += [(N // 8 * 8, shape("w4a8", M, N // 8 * 8, 128, 128, MUCH)), (N // 2, shape("w4a16", 0, _lib.F16, M, N // 2, 128, 128, MUCH))]
            for n, got in calls:
                assert got is None or -(-n // (16 * got[2])) * -(-M // (16 * got[1])) * got[0] * 64 < 1 << 32, (M, n, got)


def test_the_mid_size_cases_stay_with_the_tile_kernels():
    """Neither the wave kernels nor the one of two wave groups takes the shapes that the tests of the mid-size kernels are for."""
    def others(kind, M, N, K):
        lib = _lib.load()
        if kind in ("fp16", "bf16"):
            dt = _lib.F16 if kind == "fp16" else _lib.BF16
            return shape("w4a16", 0, dt, M, N, K, 128, lib.llmk_gemm_w4a16_nk_workspace_bytes(M, N, K, 128, dt)) or shape_w4a16(0, dt, 128, M, N, K)
        k8 = (_lib.KIND_FP8, 0) if kind == "fp8" else (_lib.KIND_I8, int(kind == "per token"))
        return shape("8bit", *k8, M, N, K, lib.llmk_gemm_workspace_bytes(M, N, K)) or shape8(*k8, M, N, K)
    for kinds, cases in MID_BLOCKS.items():
        assert {(kind, c): others(kind, *c) for kind in kinds for c in cases if others(kind, *c)} == {}
    assert {c: others("fp8", *c) for c in MID_128_COLUMNS if others("fp8", *c)} == {}

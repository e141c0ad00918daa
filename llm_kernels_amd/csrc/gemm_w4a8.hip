// W4A8 GEMM: int8 activations x row-packed uint4 weights with two-level scales.
#include <algorithm>
#include "gemm_duo.hpp"
#include "gemm_wave.hpp"
#include "gemm_wide.hpp"

using namespace llmk;

namespace {

// 16-bit block scales that the same launch widens to fp32 for the int8 GEMM behind it (blocks past the expansion's):
// saves that GEMM a launch of its own for the activation scales
struct W4A8Widen {
    const void* a_s; const void* b_s;
    float* a_s32; float* b_s32;
    int64_t n_a, n_b;
    int s_dtype;
    unsigned first_block;       // 0: nothing to widen
};

// packed [N/8, K] int32 -> b8 [N, K] int8 with b8 = int8(int8(q - z4) * s4) (two's-complement wrap)
__global__ void w4a8_expand_kernel(const int32_t* __restrict__ packed, const int8_t* __restrict__ s4,
                                   const int8_t* __restrict__ z4, int8_t* __restrict__ out,
                                   int64_t N, int64_t K, int group, W4A8Widen wd) {
    if (wd.first_block && blockIdx.x >= wd.first_block) {
        const int64_t i = (int64_t)(blockIdx.x - wd.first_block) * blockDim.x + threadIdx.x;
        if (i < wd.n_a) wd.a_s32[i] = ld_scale(wd.a_s, i, wd.s_dtype);
        else if (i < wd.n_a + wd.n_b) wd.b_s32[i - wd.n_a] = ld_scale(wd.b_s, i - wd.n_a, wd.s_dtype);
        return;
    }
    // one thread: 8 rows x 4 consecutive k
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t kq = K / 4;
    if (idx >= (N / 8) * kq) return;
    const int64_t pr = idx / kq, k = (idx - pr * kq) * 4;
    const v4i w = ((const Loose<v4i, 4>*)(packed + pr * K + k))->v;          // (a view of the words at any offset)
    const int64_t kg = K / group;
    const int64_t gi = k / group;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int64_t n = pr * 8 + i;
        const int z = z4[n * kg + gi], s = s4[n * kg + gi];
        unsigned o = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int q = (w[j] >> (4 * i)) & 0xf;
            const int d = (int)(int8_t)(q - z);
            o |= ((unsigned)((d * s) & 0xff)) << (8 * j);
        }
        *(unsigned*)(out + n * K + k) = o;
    }
}


}  // namespace

// Which path a shape takes (pointer alignment aside) and the scratch that path uses.
namespace {
struct W4A8Plan {
    bool wave;            // wave kernel, else the kernel of two wave groups (duo.mi), else expansion to int8 and the int8 GEMM
    WavePlan shape;
    int64_t bytes;        // scratch the chosen path uses
    DuoPlan duo;
};
// scratch layout of the two-pass path: int8 copy of W | fp32 activation scales | fp32 weight scales | the int8 GEMM's own
inline int64_t w4a8_two_pass_scales_off(int64_t N, int64_t K) { return (N * K + 255) & ~(int64_t)255; }
inline int64_t w4a8_a_s32_bytes(int64_t M, int64_t K) { return (M * (K / 128) * 4 + 255) & ~(int64_t)255; }
inline int64_t w4a8_widened_bytes(int64_t M, int64_t N, int64_t K) {
    return w4a8_a_s32_bytes(M, K) + ((((N + 127) / 128) * (K / 128) * 4 + 255) & ~(int64_t)255);
}

// Up to 128 rows the wave kernel beats both what it replaced and the two passes (1.45 times over 180 shapes of 1 to 520 rows).
// From there to 512 rows it is taken 12 % below the estimate of the two passes: the expansion, the rounds of the int8 tiles, two
// launches (a fit of 12 % rms to 25 shapes).  (us, wave | two passes: 512 x 4096 x 4096 25.4 | 31.9, 384 x 4096 x 4096 22 | 30, but 245 x 28672 x 4096 78.9 | 70.4; every row
// tile unpacks the weights again, so large N K goes the other way.)
// From 65 rows on the kernel of two wave groups, which expands the words itself, is taken 8 % below the estimate of either: the two passes are the
// expansion, and the int8 tiles or that kernel on int8 weights, whichever is estimated faster (a fit of 7 % rms to 165 shapes).  Over 300
// random shapes of 64 to 4096 rows this was 1.05 times as fast as without; of 1070 more 5 were 5 to 10 % slower.  Others | this one, us: 1024 x 4096 x 4096
// 36.7 | 30.8, 425 x 6144 x 4096 32.5 | 25.3, 184 x 14272 x 1664 19.2 | 14.5, but 2373 x 6144 x 4096 79 | 107 and 91 x 5936 x 1024 7.1 | 9.5.
// The two passes of few tiles have an estimate of their own (7 % rms to 110 shapes of K below 3072): with the other one 48 of 161 shapes went to this kernel
// and were 3 to 10 % slower (1718 x 160 x 1152 9.6 | 10.7, 3723 x 112 x 1664 11.6 | 13.0).
W4A8Plan w4a8_plan(int64_t M, int64_t N, int64_t K, int group_int4, int64_t scratch) {
    W4A8Plan pl{false, {}, 0, {0, 1, 0.0}};
    if (M <= 0 || N <= 0 || K <= 0) return pl;
    DirectArgs q{};
    if (group_int4 == 128 && M <= 512 && N <= 0x7fffffff && K <= (1 << 25) && w4a8_wave_plan(M, N, K, scratch, pl.shape)) {
        q.M = (int)M; q.N = (int)N; q.K = (int)K; q.E = 1;
        pl.wave = M <= 128;
        if (!pl.wave) {
            const double two = 10.0 + (double)N * K * 0.41e-6 + 0.72 * dma_tile_estimate<K_I8_BLOCK, false>(q).cost * K / 4096.0;
            pl.wave = 1.12 * pl.shape.cost < two;
        }
    }
    const int64_t slices = pl.wave && pl.shape.z > 1 ? (int64_t)pl.shape.z * M * N * 4 : 0;
    const int64_t two_pass = w4a8_two_pass_scales_off(N, K) + w4a8_widened_bytes(M, N, K) + llmk_gemm_workspace_bytes(M, N, K);
    // Words that do not start on 16 bytes go through the two passes.  Callers who pass what is reported may have such words with any
    // shape but those of few rows or few tiles, whose scratch stays small: 64 rows, 128 with K up to 32768, 256 on one 64-column
    // workgroup a CU with K up to 16384.
    const bool small = M <= 64 || ((M <= 128 || (M <= 256 && mid_plan(M, N, K).tiles <= LLMK_CUS && K <= 16384)) && dma_eligible(q));
    // (from 17 rows on at least what the int8 GEMM of the shape can use, so that one buffer serves both)
    if (!pl.wave) pl.bytes = two_pass;
    else if (!small) pl.bytes = std::max(slices, two_pass);
    else pl.bytes = M <= 16 ? slices : std::max(slices, llmk_gemm_workspace_bytes(M, N, K));
    // (K from 1024 on: neither estimate was fitted to less)
    if (M > 64 && K >= 1024 && group_int4 == 128 && M <= 0x7fffffff && N <= 0x7fffffff && K <= 0x7fffffff) {
        q.M = (int)M; q.N = (int)N; q.K = (int)K; q.E = 1;
        pl.duo = duo_plan<K_W4A8>(q, scratch);
        if (pl.duo.mi) {
            double other = 1.05 * pl.shape.cost;
            if (!pl.wave) {
                const TileChoice c = dma_tile_estimate<K_I8_BLOCK, false>(q);
                const double tiles = (c.choice <= 2 ? 3.5 : 6.8) + (c.choice == 8 ? 1.03 : (c.choice == 2 ? 0.86 : 0.95)) * c.cost * (double)K / 4096.0;
                other = 4.3 + (double)N * K * 0.23e-6 + 1.03 * std::min(tiles, duo_plan<K_I8_BLOCK>(q, INT64_MAX).cost);
                // few short tiles: what the first pass takes is mostly its launch, and the second one's overlaps it
                if (c.choice == 1) other = std::min(other, 4.8 + (double)N * K * 0.12e-6 + 1.02 * c.cost * (double)K / 4096.0);
            }
            if (DU_MARGIN * pl.duo.cost >= other) pl.duo.mi = 0;
        }
        if (pl.duo.mi) {
            pl.wave = false;
            if (pl.duo.z > 1) pl.bytes = std::max(pl.bytes, (int64_t)pl.duo.z * M * N * 4);
        }
    }
    return pl;
}
}  // namespace

extern "C" int64_t llmk_gemm_w4a8_workspace_bytes(int64_t M, int64_t N, int64_t K, int group_int4) {
    return w4a8_plan(M, N, K, group_int4, INT64_MAX).bytes;
}

extern "C" int llmk_gemm_w4a8_wave_shape(int64_t M, int64_t N, int64_t K, int group_int4, int64_t scratch_bytes, int32_t* shape) {
    const W4A8Plan pl = w4a8_plan(M, N, K, group_int4, scratch_bytes);
    return pl.wave && shape ? wave_shape(pl.shape, wv_depth(pl.shape.mt, pl.shape.nt, ((K >> 7) + pl.shape.z - 1) / pl.shape.z), shape) : 0;
}

extern "C" int llmk_gemm_w4a8_duo_shape(int64_t M, int64_t N, int64_t K, int group_int4, int64_t scratch_bytes, int32_t* shape) {
    const W4A8Plan pl = w4a8_plan(M, N, K, group_int4, scratch_bytes);
    if (!pl.duo.mi || !shape) return 0;
    shape[0] = 32 * pl.duo.mi;
    shape[1] = pl.duo.z;
    return 1;
}

extern "C" int llmk_gemm_w4a8(const int8_t* a, const void* a_s, const int32_t* b_packed, const void* b_s, int s_dtype,
                              const int8_t* b_s4, const int8_t* b_z4, void* c, int c_dtype, int64_t M, int64_t N,
                              int64_t K, int group_int4, void* workspace, int64_t workspace_bytes, void* stream) {
    if (M < 0 || N < 0 || K < 0) LLMK_FAIL(LLMK_ERR_SHAPE, "gemm_w4a8: negative dimension");
    if (K % 128 || N % 8) LLMK_FAIL(LLMK_ERR_SHAPE, "gemm_w4a8: need K %% 128 == 0 and N %% 8 == 0 (K=%lld N=%lld)", (long long)K, (long long)N);
    if (group_int4 < 4 || group_int4 % 4 || K % group_int4) LLMK_FAIL(LLMK_ERR_SHAPE, "gemm_w4a8: group_int4=%d must divide K and be a multiple of 4", group_int4);
    if (M == 0 || N == 0) return LLMK_OK;
    if (!a || !a_s || !b_packed || !b_s || !b_s4 || !b_z4 || !c) LLMK_FAIL(LLMK_ERR_ARG, "gemm_w4a8: null pointer");
    const int64_t scratch = workspace && !((uintptr_t)workspace & 15) ? workspace_bytes : 0;
    const W4A8Plan pl = w4a8_plan(M, N, K, group_int4, scratch);
    if ((pl.wave || pl.duo.mi) && !(((uintptr_t)a | (uintptr_t)b_packed) & 15)) {
        if (s_dtype != LLMK_F32 && s_dtype != LLMK_F16 && s_dtype != LLMK_BF16) LLMK_FAIL(LLMK_ERR_DTYPE, "gemm_w4a8: s_dtype %d", s_dtype);
        if (c_dtype != LLMK_F32 && c_dtype != LLMK_F16 && c_dtype != LLMK_BF16) LLMK_FAIL(LLMK_ERR_DTYPE, "gemm_w4a8: c_dtype %d", c_dtype);
        DirectArgs p{};
        p.a = (const uint8_t*)a; p.b = (const uint8_t*)b_packed; p.c = c; p.a_s = a_s; p.b_s = b_s;
        p.w4_s4 = b_s4; p.w4_z4 = b_z4;
        p.c_dtype = c_dtype; p.s_dtype = s_dtype; p.M = (int)M; p.N = (int)N; p.K = (int)K; p.E = 1; p.group = 128;
        if (pl.duo.mi)
            return s_dtype == LLMK_F32 ? launch_duo_plan<K_W4A8>(p, pl.duo, workspace, (hipStream_t)stream, "gemm_w4a8(duo)")
                                       : launch_duo_plan<K_W4A8, true>(p, pl.duo, workspace, (hipStream_t)stream, "gemm_w4a8(duo)");
        p.partial = (float*)workspace;
        return launch_w4a8_wave_plan(p, pl.shape, (hipStream_t)stream, "gemm_w4a8(wave)");
    }
    if (!workspace || workspace_bytes < N * K) LLMK_FAIL(LLMK_ERR_ARG, "gemm_w4a8: workspace of N*K=%lld bytes required", (long long)(N * K));
    // 16-bit block scales are widened by spare blocks of the expansion launch when the scratch has room for them
    W4A8Widen wd{};
    int64_t used = (N * K + 15) & ~(int64_t)15;
    const int64_t soff = w4a8_two_pass_scales_off(N, K);
    if ((s_dtype == LLMK_F16 || s_dtype == LLMK_BF16) && K > 0 && !((uintptr_t)workspace & 255) &&
        workspace_bytes >= soff + w4a8_widened_bytes(M, N, K)) {
        wd.a_s = a_s; wd.b_s = b_s; wd.s_dtype = s_dtype;
        wd.n_a = M * (K / 128); wd.n_b = ((N + 127) / 128) * (K / 128);
        wd.a_s32 = (float*)((uint8_t*)workspace + soff);
        wd.b_s32 = (float*)((uint8_t*)workspace + soff + w4a8_a_s32_bytes(M, K));
        used = soff + w4a8_widened_bytes(M, N, K);
    }
    if (K > 0) {
        const unsigned expand_blocks = (unsigned)cdiv64((N / 8) * (K / 4), 256);
        unsigned blocks = expand_blocks;
        if (wd.a_s32) {
            wd.first_block = expand_blocks;
            blocks += (unsigned)cdiv64(wd.n_a + wd.n_b, 256);
        }
        w4a8_expand_kernel<<<blocks, 256, 0, (hipStream_t)stream>>>(b_packed, b_s4, b_z4, (int8_t*)workspace, N, K, group_int4, wd);
        LLMK_CHECK_LAUNCH("gemm_w4a8(expand)");
    }
    // what is left of the workspace behind the expanded weights (16-byte aligned) serves the int8 GEMM
    void* rest = workspace_bytes > used ? (void*)((uint8_t*)workspace + used) : nullptr;
    const int64_t rest_bytes = rest ? workspace_bytes - used : 0;
    if (wd.a_s32)
        return llmk_gemm_i8_block(a, wd.a_s32, (const int8_t*)workspace, wd.b_s32, LLMK_F32, c, c_dtype, M, N, K, rest, rest_bytes, stream);
    return llmk_gemm_i8_block(a, a_s, (const int8_t*)workspace, b_s, s_dtype, c, c_dtype, M, N, K, rest, rest_bytes, stream);
}

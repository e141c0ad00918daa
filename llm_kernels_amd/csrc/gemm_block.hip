// Dense block-scaled fp8 / int8 GEMM entry points.
#include <algorithm>
#include <mutex>

#include "gemm_duo.hpp"
#include "gemm_wave.hpp"
#include "gemm_wide.hpp"

using namespace llmk;

namespace {

int check_common(const char* name, const void* a, const void* b, int64_t M, int64_t N, int64_t K, int c_dtype) {
    if (M < 0 || N < 0 || K < 0) LLMK_FAIL(LLMK_ERR_SHAPE, "%s: negative dimension", name);
    if (K % 128 != 0) LLMK_FAIL(LLMK_ERR_SHAPE, "%s: K=%lld must be a multiple of 128", name, (long long)K);
    if (M > 0x7fffffff || N > 0x7fffffff || K > 0x7fffffff) LLMK_FAIL(LLMK_ERR_SHAPE, "%s: dimension exceeds int32", name);
    if (c_dtype != LLMK_F32 && c_dtype != LLMK_F16 && c_dtype != LLMK_BF16) LLMK_FAIL(LLMK_ERR_DTYPE, "%s: c_dtype %d", name, c_dtype);
    if (M && N && K && (!a || !b)) LLMK_FAIL(LLMK_ERR_ARG, "%s: null operand", name);
    if ((((uintptr_t)a) | ((uintptr_t)b)) & 15) LLMK_FAIL(LLMK_ERR_ARG, "%s: operands must be 16-byte aligned", name);
    return LLMK_OK;
}

// Planes of fp32 sums that the reported scratch of decode-sized calls is sized for, one per 4096 elements of K.  The wave kernels
// slice K beyond 16384 only, into as many ranges as these planes hold at most; up to there nothing touches them, but the size is what
// callers have been told, and what llmk_gemm_fp8_block_static accepts a shape by.
inline int stream_k_ranges(int64_t M, int64_t N, int64_t K) {
    if (M > 64 || K <= 4096 || mid_m_prefers_tiles(M, N, K)) return 1;
    return (int)((K / 128 + 31) / 32);
}

// scratch of the kernels beside the one of two wave groups, without the (fixed-size) part for a split last round of 256-column tiles
int64_t tiles_core_bytes(int64_t M, int64_t N, int64_t K) {
    // large-M kernels stream fp32 activation scales; 16-bit scales are widened into the workspace first;
    // mid-size M with few tiles adds the fp32 split-K partials behind them
    if (K <= 0) return 0;
    if (M <= 64 && !mid_m_prefers_tiles(M, N, K) && !mid_wanted(M, N, K)) {
        const int nz = stream_k_ranges(M, N, K);
        return nz > 1 ? (int64_t)nz * M * N * 4 : 0;
    }
    const int64_t scales = (M * (K / 128) * 4 + 255) & ~(int64_t)255;
    int z = splitk_factor(M, N, K);
    if (M <= 512) z = std::max({z, mid_plan(M, N, K).z, midw_plan(M, N, K).z});      // the mid-size kernels' K slices
    return scales + (z > 1 ? (int64_t)z * M * N * 4 : 0);
}
// Is there scratch for a decode-sized call's K slices on the tile kernels?  (from 65 rows on nothing is chosen by it)
bool slices_fit(const DirectArgs& p, const void* workspace, int64_t workspace_bytes) {
    return p.M > 64 || (workspace && workspace_bytes >= tiles_core_bytes(p.M, p.N, p.K));
}

// What the tile kernels take for 17 to 512 rows, in us like the wave kernels' estimates (a fit of 5 to 15 % rms to 600 shapes): the
// mid-size kernels with 64 and 128 columns, the 128-column tile in K slices, or rounds of the tiles that dma_tile_estimate chooses.
// Up to 16 rows, and up to 64 on weights that no tile kernel fills the chip with or without scratch for their K slices, the wave
// kernels have no rival.
// hbm: the mean of weights in the cache and weights from HBM (nk: the weights' MB) where it is far from the former, which is what the estimate of
// the two-group kernel gives: 64-row tiles beyond 8 KB rows 1.07, K slices in more than a round 1.11 to 1.16, 128-row tiles 1.04 to 1.08,
// 128 x 256 tiles 0.88 times the other one (600 timings of 200 random shapes of 65 to 512 rows; 3 to 7 % rms so).
template <int KIND>
double tiles_estimate(const DirectArgs& p, bool scratch, bool hbm = false) {
    const int64_t M = p.M, N = p.N, K = p.K;
    const double k = (double)K / 4096.0, nk = (double)N * K * 1e-6, plane = 4e-6 * (double)M * N;
    if (M <= 16 || (M <= 64 && (!scratch || !(mid_m_prefers_tiles(M, N, K) || mid_wanted(M, N, K))))) return 1e30;
    if (mid_wanted(M, N, K)) {
        const MidPlan pl = mid_plan(M, N, K);
        if (hbm && K > 8192 && pl.z == 1) return 3.6 + 6.7 * k + 0.06 * nk;
        return (pl.mt == 2 ? 3.2 + 7.4 * k / pl.z : 4.0 + 7.2 * k / pl.z) + (pl.z > 1 ? 2.9 : 0.0);
    }
    if (KIND == K_FP8_BLOCK && midw_wanted(M, N, K)) {
        const MidPlan pl = midw_plan(M, N, K);
        return (pl.mt == 4 ? 3.6 + 11.9 * k / pl.z : 5.2 + 19.2 * k / pl.z) + (pl.z > 1 ? 3.5 : 0.0);
    }
    const int z = splitk_factor(M, N, K);
    // K slices of 64-row tiles, two launches: by whether they are one round of workgroups and whether every K step is scaled (a fit of 7 to 9 %
    // rms to 37 shapes of int8 and per token).  A cost that is only proportional to the slices' length, 19 % rms, chose the slower kernel for
    // 12 of them by 6 to 19 % with weights from HBM, this one for 2 by 7 % (us, wave | tiles: int8 128 x 4096 x 14336 29.9 | 26.3, per token
    // 300 x 4096 x 14336 48.1 | 42.5, but 400 x 1030 x 9088 14.1 | 18.5).
    if (z > 1) {
        const bool one = ((M + 63) / 64) * ((N + 127) / 128) * z <= LLMK_CUS;
        if (hbm && !one) return (KIND == K_I8_ROWCOL ? 8.2 + 13.2 * k / z : 1.8 + 22.7 * k / z) + 0.59 * z * plane + 0.076 * nk;
        if (KIND == K_I8_ROWCOL) return one ? 7.0 + 13.5 * k / z : 10.0 + 16.5 * k / z;
        return 8.0 + (one ? 15.0 : 24.0) * k / z;
    }
    const TileChoice c = dma_tile_estimate<KIND, false>(p);
    const double e = c.cost * k * (KIND == K_I8_BLOCK ? 1.12 : 1.0);
    if (hbm && c.choice == 2) return 5.0 + (KIND == K_I8_BLOCK ? 0.77 : 0.74) * e;
    if (hbm && c.choice == 9 && KIND != K_I8_BLOCK) return 7.0 + 0.69 * e;
    return c.choice == 1 ? 3.4 + 0.87 * e : (c.choice == 2 ? 5.0 + 0.7 * e : (c.choice == 8 ? 9.0 + 0.85 * e : 7.5 + 0.8 * e));
}
// The wave kernel for this call (gemm_wave.hpp), or nw = 0: up to 512 rows, where it is estimated 8 % below the tile kernels, or 16 %.  The
// estimates are fitted to weights in the cache; from HBM the tile kernels, with more loads in flight a CU, lose less.  So 16 % for
// block-scaled operands beyond 128 rows, and from 65 rows for weights of 24 MB or more.  Measured on 237 random shapes of 65 to
// 512 rows, N 1024 to 28672, K 1024 to 14336, weights from HBM, both kernels timed; speed against the tile kernels alone with margins of
// 8 | 16 | 20 %: fp8 129 to 512 rows 1.015 | 1.019 | 1.005, int8 65 to 128 1.023 | 1.039 | 1.039, 129 to 512 1.022 | 1.028 | 1.028.  What
// 8 % lost on large weights, us, wave | tiles: int8 90 x 14336 x 4096 24.3 | 21.1, 74 x 21400 x 12160 86.1 | 75.2, per token 81 x 21672 x 3584
// 27.8 | 22.4, 427 x 5424 x 14208 77.1 | 62.8 (and gained: 280 x 4992 x 8960 9 %, on small ones int8 84 x 3952 x 1280 5.7 | 6.5).  What the
// wave kernel gains: int8 29 x 4096 x 4096 7.2 | 8.7, fp8 64 x 4096 x 4096 8.8 | 10.8, per token 337 x 3592 x 4608 17.9 | 21.0, 359 x
// 2112 x 10112 21.8 | 29.4; from 513 rows on it is 0.8 times as fast.
template <int KIND>
WavePlan wave_choice(const DirectArgs& p, int64_t scratch, bool tiles_scratch) {
    WavePlan w{0, 0, 0, 0, 0.0};
    if (p.M > 512 || !w8_wave_plan<KIND>(p.M, p.N, p.K, scratch, w)) w.nw = 0;
    const bool cold = (KIND != K_I8_ROWCOL && p.M > 128) || (p.M > 64 && (int64_t)p.N * p.K >= (24 << 20));
    const double margin = cold ? 1.16 : 1.08;
    if (w.nw && p.M > 16 && margin * w.cost >= tiles_estimate<KIND>(p, tiles_scratch)) w.nw = 0;
    return w;
}
template <int KIND>
WavePlan wave_choice(const DirectArgs& p, const void* workspace, int64_t workspace_bytes) {
    return wave_choice<KIND>(p, workspace && !((uintptr_t)workspace & 15) ? workspace_bytes : 0,
                             slices_fit(p, workspace, workspace_bytes));
}
// What the tile kernels take beyond 512 rows, in us: rounds of the tiles that dma_tile_estimate chooses (a fit of 3 to 5 % rms for the 128-column
// ones, 7 to 10 % for the 256-column ones, to 80 to 140 shapes a kind).  int8: with a widening pass in front of the 256-column tiles, which fp16 scales
// need in long launches only.  80 random shapes with those, both kernels timed: what is chosen takes 1.011 (from HBM 1.005) of the faster one's time, all of it in
// calls that the kernel of two wave groups would have done 3 to 8 % faster (2777 x 6144 x 4096 112 | 104.5); none that it gets is slower there.
template <int KIND>
double large_estimate(const DirectArgs& p, bool tail) {
    const TileChoice c = dma_tile_estimate<KIND, false>(p, tail);
    const double e = c.cost * (double)p.K / 4096.0;
    struct { double a, b; } f[5] = {{2.6, 0.83}, {3.0, 0.80}, {6.0, 0.80}, {5.2, 0.82}, {4.6, 0.80}};
    if (KIND == K_I8_BLOCK) { f[0] = {2.9, 0.97}; f[1] = {4.0, 0.86}; f[2] = {6.0, 0.95}; f[3] = {8.2, 1.03}; f[4] = {6.1, 0.94}; }
    if (KIND == K_I8_ROWCOL) { f[0] = {3.3, 0.80}; f[1] = {5.9, 0.64}; f[2] = {6.0, 0.78}; f[3] = {10.2, 0.74}; f[4] = {6.2, 0.73}; }
    const auto& s = f[c.choice == 1 ? 0 : (c.choice == 2 ? 1 : (c.choice == 4 ? 2 : c.choice - 5))];
    return s.a + s.b * e;
}
// The kernel of two wave groups (gemm_duo.hpp) for this call, or mi = 0: 8 % below the estimate of what the call gets otherwise (w: the wave
// kernel, if it does).  Over 300 random shapes of 64 to 4096 rows a kind this was 1.04 (fp8, int8, per token) times as fast as without,
// 0.5 to 1 % behind the faster one of each shape; of 4110 more, cached weights and weights from HBM, 5 were 5 to 8 % slower.  Others | this one, us: fp8 1024 x 4096 x 4096 25.5 | 20.7, int8 28.8 |
// 25.6, per token 23.9 | 20.3; the gain is largest where 96, 128 or 160 rows leave fewer rows of the last tiles empty than 64, 128 and
// 256 do, and where few tiles can be split along K beyond 512 rows.  Up to 512 rows the others are estimated with weights from HBM in the mean (450
// shapes 1.007 fp8, 1.002 int8, 1.005 per token times as fast as with their cached times, us, cached | HBM: fp8 129 x 4096 x 14336 22.8 | 33.6 -> 20.7 |
// 23.9, int8 110 x 15992 x 12032 48.5 | 66.3 -> 40.6 | 49.0, per token 452 x 3176 x 10112 31.1 | 37.5 -> 24.7 | 30.3).
// Two kinds of calls up to 512 rows are left to the others whatever the estimates say, which have no term for weights from HBM there: int8 and per-token
// products of short K on one row tile (66 shapes 0.98 times as fast here, us, others | this one, from HBM: int8 97 x 20048 x 1664 14.1 | 15.9, per token
// 131 x 19264 x 1664 15.1 | 17.6; fp8 gains there) and fp8 and per-token ones of more than a round of workgroups (18 shapes 0.98: per token 500 x
// 17848 x 11904 131 | 176, fp8 289 x 23480 x 2304 33.1 | 41.1; int8 gains).
template <int KIND>
DuoPlan duo_choice(const DirectArgs& p, const WavePlan& w, int64_t scratch, bool tiles_scratch, bool tail) {
    DuoPlan d = duo_plan<KIND>(p, scratch);
    if (!d.mi) return d;
    if (KIND != K_FP8_BLOCK && p.K < 2304 && p.M <= (KIND == K_I8_ROWCOL ? 160 : 128)) d.mi = 0;
    if (KIND != K_I8_BLOCK && p.M <= 512 && d.mi && duo_beyond_a_round(p, d)) d.mi = 0;
    const double other = p.M <= 512 ? (w.nw ? 1.05 * w.cost : tiles_estimate<KIND>(p, tiles_scratch, true)) : large_estimate<KIND>(p, tail);
    if (DU_MARGIN * d.cost >= other) d.mi = 0;
    return d;
}
template <int KIND>
DuoPlan duo_choice(const DirectArgs& p, const WavePlan& w, void* workspace, int64_t workspace_bytes) {
    return duo_choice<KIND>(p, w, workspace && !((uintptr_t)workspace & 15) ? workspace_bytes : 0,
                            slices_fit(p, workspace, workspace_bytes), wide_tail_ok<KIND>(p, workspace, workspace_bytes));
}
template <int KIND>
int launch_block(const DirectArgs& p, void* workspace, int64_t workspace_bytes, hipStream_t stream, const char* name) {
    const WavePlan w = wave_choice<KIND>(p, workspace, workspace_bytes);
    if (p.M > 64) {
        const DuoPlan d = duo_choice<KIND>(p, w, workspace, workspace_bytes);
        if (d.mi) {
            if constexpr (KIND == K_I8_BLOCK) if (p.s_dtype != LLMK_F32) return launch_duo_plan<KIND, true>(p, d, workspace, stream, name);
            return launch_duo_plan<KIND>(p, d, workspace, stream, name);
        }
    }
    if (w.nw) return launch_w8_wave_plan<KIND>(p, w, workspace, stream, name);
    if (p.K == 0) return launch_empty_sums<false>(p, stream, name);
    return launch_big<KIND, false>(p, workspace, workspace_bytes, stream, name);
}

}  // namespace

// planes of the kernel of two wave groups, where a kind takes it in K slices
template <int KIND>
static int64_t duo_bytes(int64_t M, int64_t N, int64_t K) {
    if (M <= 64 || N <= 0 || K < 12 * 128 || M > 0x7fffffff || N > 0x7fffffff || K > 0x7fffffff) return 0;
    DirectArgs p{};
    p.M = (int)M; p.N = (int)N; p.K = (int)K; p.E = 1; p.s_dtype = LLMK_F32;
    const WavePlan w = wave_choice<KIND>(p, INT64_MAX, true);
    const DuoPlan d = duo_choice<KIND>(p, w, INT64_MAX, true, KIND != K_I8_ROWCOL && M > 512 && K >= W_TAIL_MIN_KT * 128);
    return d.mi && d.z > 1 ? (int64_t)d.z * M * N * 4 : 0;
}
// (the plans of the three kinds take 0.2 us)
static int64_t workspace_core_bytes(int64_t M, int64_t N, int64_t K) {
    return std::max({tiles_core_bytes(M, N, K), duo_bytes<K_FP8_BLOCK>(M, N, K), duo_bytes<K_I8_BLOCK>(M, N, K), duo_bytes<K_I8_ROWCOL>(M, N, K)});
}
static int64_t tail_bytes(int64_t M, int64_t K) { return K >= W_TAIL_MIN_KT * 128 && M > 512 ? w_tail_bytes() : 0; }

extern "C" int64_t llmk_gemm_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    // more than 512 rows and at least W_TAIL_MIN_KT K steps of 128 bytes (shorter tiles are never split): room for
    // the partial sums of a split last round of 256-column tiles behind the rest
    return workspace_core_bytes(M, N, K) + tail_bytes(M, K);
}

// Per-token products slice K up to 512 rows, and beyond on the kernel of two wave groups only; they widen no scales there and split no last round.
extern "C" int64_t llmk_gemm_i8_rowcol_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    return std::max(M <= 512 ? tiles_core_bytes(M, N, K) : 0, duo_bytes<K_I8_ROWCOL>(M, N, K));
}

// Grouped products slice no K: fp32 activation scales where the caller's are 16-bit, and the split last round.
extern "C" int64_t llmk_grouped_gemm_workspace_bytes(int kind, int s_dtype, int64_t M, int64_t N, int64_t K) {
    if ((kind != LLMK_KIND_I8 && kind != LLMK_KIND_FP8) || M <= 0 || N <= 0 || K <= 0) return 0;
    return (s_dtype == LLMK_F32 ? 0 : (M * (K / 128) * 4 + 255) & ~(int64_t)255) + tail_bytes(M, K);
}

extern "C" int llmk_gemm_8bit_wave_shape(int kind, int per_token, int64_t M, int64_t N, int64_t K, int64_t scratch_bytes, int32_t* shape) {
    if (!shape || M <= 0 || N <= 0 || K <= 0 || K % 128 || M > 0x7fffffff || N > 0x7fffffff || K > 0x7fffffff) return 0;
    DirectArgs p{};
    p.M = (int)M; p.N = (int)N; p.K = (int)K; p.E = 1;
    const bool full = M > 64 || (scratch_bytes > 0 && scratch_bytes >= tiles_core_bytes(M, N, K));
    const WavePlan w = kind == LLMK_KIND_FP8 ? wave_choice<K_FP8_BLOCK>(p, scratch_bytes, full)
                                             : (per_token ? wave_choice<K_I8_ROWCOL>(p, scratch_bytes, full) : wave_choice<K_I8_BLOCK>(p, scratch_bytes, full));
    int32_t duo[2];
    if (!w.nw || llmk_gemm_8bit_duo_shape(kind, per_token, M, N, K, scratch_bytes, duo)) return 0;
    return wave_shape(w, w8_depth(w, M, N, K), shape);
}

extern "C" int llmk_gemm_8bit_duo_shape(int kind, int per_token, int64_t M, int64_t N, int64_t K, int64_t scratch_bytes, int32_t* shape) {
    if (!shape || M <= 64 || N <= 0 || K <= 0 || K % 128 || M > 0x7fffffff || N > 0x7fffffff || K > 0x7fffffff) return 0;
    DirectArgs p{};
    p.M = (int)M; p.N = (int)N; p.K = (int)K; p.E = 1; p.s_dtype = LLMK_F32;
    const bool tail = M > 512 && K >= W_TAIL_MIN_KT * 128 && scratch_bytes >= w_tail_bytes();
    auto plan = [&](auto kind_c) {
        constexpr int KIND = decltype(kind_c)::value;
        return duo_choice<KIND>(p, wave_choice<KIND>(p, scratch_bytes, true), scratch_bytes, true, KIND != K_I8_ROWCOL && tail);
    };
    const DuoPlan d = kind == LLMK_KIND_FP8 ? plan(std::integral_constant<int, K_FP8_BLOCK>{})
                                            : (per_token ? plan(std::integral_constant<int, K_I8_ROWCOL>{}) : plan(std::integral_constant<int, K_I8_BLOCK>{}));
    if (!d.mi) return 0;
    shape[0] = 32 * d.mi;
    shape[1] = d.z;
    return 1;
}

extern "C" int llmk_gemm_fp8_block(const void* a, const float* a_s, const void* b, const float* b_s, void* c,
                                   int c_dtype, int64_t M, int64_t N, int64_t K, void* workspace,
                                   int64_t workspace_bytes, void* stream) {
    int rc = check_common("gemm_fp8_block", a, b, M, N, K, c_dtype);
    if (rc) return rc;
    if (M == 0 || N == 0) return LLMK_OK;
    if (!c || (K && (!a_s || !b_s))) LLMK_FAIL(LLMK_ERR_ARG, "gemm_fp8_block: null pointer");
    DirectArgs p{};
    p.a = (const uint8_t*)a; p.b = (const uint8_t*)b; p.c = c; p.a_s = a_s; p.b_s = b_s;
    p.c_dtype = c_dtype; p.s_dtype = LLMK_F32; p.M = (int)M; p.N = (int)N; p.K = (int)K; p.E = 1;
    return launch_block<K_FP8_BLOCK>(p, workspace, workspace_bytes, (hipStream_t)stream, "gemm_fp8_block");
}

// The tile kernels of llmk_gemm_fp8_block for the benchmark's calibration, also where that call takes the kernel of two wave groups: workgroup 0 of
// the 256-column tile kernel reports the ticks of the shader clock and of the 100 MHz clock it lived (clocks[0], clocks[1]); shapes that run on
// other kernels leave clocks untouched.
extern "C" int llmk_calib_gemm_fp8_clock(const void* a, const float* a_s, const void* b, const float* b_s, void* c,
                                         int c_dtype, int64_t M, int64_t N, int64_t K, void* workspace,
                                         int64_t workspace_bytes, long long* clocks, void* stream) {
    int rc = check_common("calib_gemm_fp8_clock", a, b, M, N, K, c_dtype);
    if (rc) return rc;
    if (M <= 64 || N == 0 || !c || !a_s || !b_s || !clocks) LLMK_FAIL(LLMK_ERR_ARG, "calib_gemm_fp8_clock: needs M > 512 and every pointer");
    DirectArgs p{};
    p.a = (const uint8_t*)a; p.b = (const uint8_t*)b; p.c = c; p.a_s = a_s; p.b_s = b_s; p.clocks = clocks;
    p.c_dtype = c_dtype; p.s_dtype = LLMK_F32; p.M = (int)M; p.N = (int)N; p.K = (int)K; p.E = 1;
    return launch_big<K_FP8_BLOCK, false>(p, workspace, workspace_bytes, (hipStream_t)stream, "calib_gemm_fp8_clock");
}

extern "C" int llmk_gemm_i8_block(const int8_t* a, const void* a_s, const int8_t* b, const void* b_s, int s_dtype,
                                  void* c, int c_dtype, int64_t M, int64_t N, int64_t K, void* workspace,
                                  int64_t workspace_bytes, void* stream) {
    int rc = check_common("gemm_i8_block", a, b, M, N, K, c_dtype);
    if (rc) return rc;
    if (s_dtype != LLMK_F32 && s_dtype != LLMK_F16 && s_dtype != LLMK_BF16) LLMK_FAIL(LLMK_ERR_DTYPE, "gemm_i8_block: s_dtype %d", s_dtype);
    if (M == 0 || N == 0) return LLMK_OK;
    if (!c || (K && (!a_s || !b_s))) LLMK_FAIL(LLMK_ERR_ARG, "gemm_i8_block: null pointer");
    DirectArgs p{};
    p.a = (const uint8_t*)a; p.b = (const uint8_t*)b; p.c = c; p.a_s = a_s; p.b_s = b_s;
    p.c_dtype = c_dtype; p.s_dtype = s_dtype; p.M = (int)M; p.N = (int)N; p.K = (int)K; p.E = 1;
    return launch_block<K_I8_BLOCK>(p, workspace, workspace_bytes, (hipStream_t)stream, "gemm_i8_block");
}

extern "C" int llmk_gemm_i8_rowcol(const int8_t* a, const float* a_s, const int8_t* b, const float* b_s, void* c,
                                   int c_dtype, int32_t* c_i32, int64_t M, int64_t N, int64_t K, void* workspace,
                                   int64_t workspace_bytes, void* stream) {
    int rc = check_common("gemm_i8_rowcol", a, b, M, N, K, c_dtype);
    if (rc) return rc;
    if (M == 0 || N == 0) return LLMK_OK;
    if (!c && !c_i32) LLMK_FAIL(LLMK_ERR_ARG, "gemm_i8_rowcol: no output buffer");
    if (c && (!a_s || !b_s)) LLMK_FAIL(LLMK_ERR_ARG, "gemm_i8_rowcol: scales required for the scaled output");
    DirectArgs p{};
    p.a = (const uint8_t*)a; p.b = (const uint8_t*)b; p.c = c; p.c_i32 = c_i32; p.a_s = a_s; p.b_s = b_s;
    p.c_dtype = c_dtype; p.s_dtype = LLMK_F32; p.M = (int)M; p.N = (int)N; p.K = (int)K; p.E = 1;
    const WavePlan wave = wave_choice<K_I8_ROWCOL>(p, workspace, workspace_bytes);
    if (M > 64) {
        const DuoPlan d = duo_choice<K_I8_ROWCOL>(p, wave, workspace, workspace_bytes);
        if (d.mi) return launch_duo_plan<K_I8_ROWCOL>(p, d, workspace, (hipStream_t)stream, "gemm_i8_rowcol(duo)");
    }
    if (wave.nw) return launch_w8_wave_plan<K_I8_ROWCOL>(p, wave, workspace, (hipStream_t)stream, "gemm_i8_rowcol(wave)");
    // large M: the tile kernels accumulate int32 over the whole K range inside the MFMA and scale in the epilogue
    if ((M > 64 || ((mid_wanted(M, N, K) || mid_m_prefers_tiles(M, N, K)) && slices_fit(p, workspace, workspace_bytes))) &&
        dma_eligible(p)) {
        // few tiles and a long K: K slices over the CUs, int32 partial sums in the workspace, one pass that adds
        // them as integers and scales (same bits as the unsplit kernel)
        if (mid_wanted(M, N, K)) {
            MidPlan pl = mid_plan(M, N, K);
            if (pl.z > 1 && !(workspace && workspace_bytes >= (int64_t)pl.z * M * N * 4 && !((uintptr_t)workspace & 15))) pl.z = 1;
            if (mid_eligible<K_I8_ROWCOL>(p)) {
                if (pl.z > 1) { p.partial = (float*)workspace; p.ksplit = pl.z; }
                return pl.mt == 4 ? launch_mid<K_I8_ROWCOL, 4>(p, (hipStream_t)stream, "gemm_i8_rowcol(mid)")
                                  : launch_mid<K_I8_ROWCOL, 2>(p, (hipStream_t)stream, "gemm_i8_rowcol(mid)");
            }
        }
        const int z = splitk_factor(M, N, K);
        if (z > 1 && workspace && workspace_bytes >= (int64_t)z * M * N * 4 && !((uintptr_t)workspace & 15)) {
            p.partial = (float*)workspace;
            p.ksplit = z;
        }
        return launch_dma<K_I8_ROWCOL, false>(p, (hipStream_t)stream, "gemm_i8_rowcol(tiled)");
    }
    return launch_direct<K_I8_ROWCOL, false>(p, (int)M, (hipStream_t)stream, "gemm_i8_rowcol");
}

// ------------------------------------------------------------------ llmk_gemm_fp8_block without a scratch argument
// For callers that cannot allocate device memory (HIP graph capture, serving loops, harnesses that forbid
// hipMalloc): the fp32 partial sums of the split-K kernels live in a file-scope device array instead
// of a caller-provided buffer.  Every GPU the library runs on holds its own copy of the array until the
// process ends; its address on a device is looked up once, with that device current, and only that address
// (never the array's name, which is a host-side stand-in) is handed to kernels.
namespace {

static __device__ __align__(256) unsigned char scratch[LLMK_STATIC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};

int static_scratch(void** out, const char* name) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) LLMK_FAIL(LLMK_ERR_LAUNCH, "%s: hipGetDevice: %s", name, hipGetErrorString(e));
    if (dev < 0 || dev >= kMaxDevices) LLMK_FAIL(LLMK_ERR_ARG, "%s: device ordinal %d out of range", name, dev);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr)
            LLMK_FAIL(LLMK_ERR_LAUNCH, "%s: hipGetSymbolAddress(scratch) on device %d: %s", name, dev, hipGetErrorString(e));
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return LLMK_OK;
}

}  // namespace

extern "C" int llmk_gemm_fp8_block_static(const void* a, const float* a_s, const void* b, const float* b_s, void* c,
                                          int c_dtype, int64_t M, int64_t N, int64_t K, void* stream) {
    int rc = check_common("gemm_fp8_block_static", a, b, M, N, K, c_dtype);
    if (rc) return rc;
    // (the built-in array serves the scratch a shape cannot do without efficiently; the optional partial sums of a
    // split last round of tiles, 64 MiB, are left out: large shapes run unsplit here)
    const int64_t need = workspace_core_bytes(M, N, K);
    if (need > (int64_t)LLMK_STATIC_SCRATCH_BYTES)
        LLMK_FAIL(LLMK_ERR_SHAPE, "gemm_fp8_block_static: M=%lld N=%lld K=%lld needs %lld bytes of scratch, the built-in "
                  "buffer holds %lld; use llmk_gemm_fp8_block with a caller-provided workspace",
                  (long long)M, (long long)N, (long long)K, (long long)need, (long long)LLMK_STATIC_SCRATCH_BYTES);
    void* ws = nullptr;
    if (need > 0) {
        rc = static_scratch(&ws, "gemm_fp8_block_static");
        if (rc) return rc;
    }
    // Every plane of partial sums is written in full by the first kernel before the summing kernel reads it,
    // so nothing in the array has to start at zero; what a previous (possibly larger) call left is never read.
    return llmk_gemm_fp8_block(a, a_s, b, b_s, c, c_dtype, M, N, K, ws, need > 0 ? need : 0, stream);
}

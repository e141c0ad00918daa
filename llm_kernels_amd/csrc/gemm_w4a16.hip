// W4A16 GEMM kernels: fp16 (row-packed layout: also bf16) activations x 4-bit weights dequantised in registers.
//
// nibble -> fp16 without integer->float converts: (q | 0x6400) is the fp16 number 1024 + q,
// ((q << 4) | 0x6400) is 1024 + 16 q; one packed subtract / fma gives q - 8 exactly.
#include <algorithm>
#include "gemm_duo.hpp"
#include "gemm_wave.hpp"
#include "gemm_wide.hpp"
#include "stream_ring.hpp"

namespace {

__device__ __forceinline__ v2h as_h2(unsigned u) { v2h r; __builtin_memcpy(&r, &u, 4); return r; }
__device__ __forceinline__ unsigned as_u32(v2h h) { unsigned r; __builtin_memcpy(&r, &h, 4); return r; }

// nibbles at bits [3:0] and [19:16] of w -> (q_lo - 8, q_hi - 8)
__device__ __forceinline__ v2h deq_lo(unsigned w) {
    const v2h k1032 = {(_Float16)1032.f, (_Float16)1032.f};
    return as_h2((w & 0x000f000fu) | 0x64006400u) - k1032;
}
// nibbles at bits [7:4] and [23:20]
__device__ __forceinline__ v2h deq_hi(unsigned w) {
    const v2h k16 = {(_Float16)0.0625f, (_Float16)0.0625f};
    const v2h k72 = {(_Float16)72.f, (_Float16)72.f};
    return as_h2((w & 0x00f000f0u) | 0x64006400u) * k16 - k72;
}

__device__ __forceinline__ v8h make8(v2h a, v2h b, v2h c, v2h d) {
    v8h r;
    r[0] = a[0]; r[1] = a[1]; r[2] = b[0]; r[3] = b[1];
    r[4] = c[0]; r[5] = c[1]; r[6] = d[0]; r[7] = d[1];
    return r;
}

// Tree reduction of per-wave accumulators through LDS; the total ends in wave 0.
template <int NW, int NACC>
__device__ __forceinline__ void reduce_waves(float (&acc)[NACC], float* buf, int wave, int lane) {
#pragma unroll
    for (int half = NW / 2; half >= 1; half >>= 1) {
        if (wave >= half && wave < 2 * half) {
            float* dst = buf + (size_t)(wave - half) * NACC * 64;
#pragma unroll
            for (int i = 0; i < NACC; ++i) dst[i * 64 + lane] = acc[i];
        }
        __syncthreads();
        if (wave < half) {
            const float* src = buf + (size_t)wave * NACC * 64;
#pragma unroll
            for (int i = 0; i < NACC; ++i) acc[i] += src[i * 64 + lane];
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------------------------------
// simple-Marlin layout.  B viewed as 16-byte units: unit ((strip * N/64) + chunk) * 32 + 4c + q
// holds, for mma lane (c = column within 8, q = k pair), word j = 16-column sub-tile j:
//   bits  3:0 (k0, c)   7:4 (k0+8, c)   11:8 (k0, c+8)   15:12 (k0+8, c+8)      k0 = 2q
//   bits 19:16 (k0+1,c) 23:20 (k0+9,c)  27:24 (k0+1,c+8) 31:28 (k0+9,c+8)
// Scales are stored per 64-column chunk as [c][2j + b] (column 16j + 8b + c).
//
// gfx950 mapping: a wave owns two chunks (128 columns).  Lane l: r = l & 15 -> c = r & 7,
// chunk half h = r >> 3; g = l >> 4 plays the role of the mma k-pair q.  One MFMA 16x16x32
// step consumes two 16-K strips; MFMA (j, b) produces columns {64(2cp+h) + 16j + 8b + c}.
// A fragment order per lane: k in {2g, 2g+1, 2g+8, 2g+9} of strip 0, then of strip 1.
// A_LDS: the activations of the workgroup's K range are staged once in LDS, already in fragment order (one
// 16-byte read per lane and step), instead of four 4-byte global loads per lane and step.
template <int MT, int NW, bool TO_WS, bool A_LDS = false>
__global__ __launch_bounds__(NW * 64) void w4a16_marlin_kernel(
    const _Float16* __restrict__ A, const v4i* __restrict__ B, const _Float16* __restrict__ S,
    _Float16* __restrict__ C, float* __restrict__ ws, int M, int N, int K, int groupsize, int steps_per_z) {
    extern __shared__ float red[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane & 15, g = lane >> 4, c = r & 7, h = r >> 3;
    const int nchunks = N >> 6;
    const int strips = K >> 4;
    const int total_steps = (strips + 1) >> 1;
    const int chunk_raw = 2 * blockIdx.x + h;
    const bool chunk_ok = chunk_raw < nchunks;
    const int chunk = chunk_ok ? chunk_raw : nchunks - 1;
    const int m0 = blockIdx.y * 16 * MT;
    const int ks_begin = blockIdx.z * steps_per_z;
    const int ks_end = min(total_steps, ks_begin + steps_per_z);

    const _Float16* arow[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) arow[mt] = A + (int64_t)min(m0 + 16 * mt + r, M - 1) * K + 2 * g;

    float acc[MT * 32];
#pragma unroll
    for (int i = 0; i < MT * 32; ++i) acc[i] = 0.f;

    // LDS image of A for steps [ks_begin, ks_end): row-major over the tile rows, per step 64 bytes = four lane
    // groups x {strip 0: k 2g, 2g+1 | 2g+8, 2g+9; strip 1: the same}; rows padded by 16 bytes (bank spread).
    const int nst = max(ks_end - ks_begin, 0);
    const int rstride = nst * 64 + 16;
    uint8_t* alds = (uint8_t*)red;
    if constexpr (A_LDS) {
        const int chunks = 16 * MT * nst * 4;                // 16-byte pieces: (row, step, strip parity, k half)
        for (int idx = threadIdx.x; idx < chunks; idx += NW * 64) {
            const int row = idx / (nst * 4), rem = idx - row * (nst * 4), ks = rem >> 2, ch = rem & 3;
            const int strip = 2 * (ks_begin + ks) + (ch >> 1);
            v4i v = {0, 0, 0, 0};
            if (strip < strips) v = *(const v4i*)(A + (int64_t)min(m0 + row, M - 1) * K + strip * 16 + (ch & 1) * 8);
            uint8_t* dst = alds + row * rstride + ks * 64 + ch * 4;
#pragma unroll
            for (int q = 0; q < 4; ++q) *(int*)(dst + q * 16) = v[q];
        }
        __syncthreads();
    }

    // Batches of U steps: every load of a batch (weights, scales, activations) is issued before the first
    // one is used, with clamped indices and no branch in between, so that a batch costs one memory round
    // trip.  Steps past the end of the range multiply by a zero activation fragment.
    constexpr int U = MT == 4 ? 1 : 2;
    const v4i* bptr = B + (int64_t)chunk * 32 + 4 * c + g;
    const int64_t strip_stride = (int64_t)nchunks * 32;
    const _Float16* sptr = S + 64 * chunk + 8 * c;
    for (int ks0 = ks_begin + wave; ks0 < ks_end; ks0 += U * NW) {
        v4i w0[U], w1[U], x[U][MT];
        v8h s0[U], s1[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int ks = min(ks0 + u * NW, ks_end - 1);
            const int st0 = 2 * ks, st1 = min(2 * ks + 1, strips - 1);
            w0[u] = bptr[st0 * strip_stride];
            w1[u] = bptr[st1 * strip_stride];
            s0[u] = *(const v8h*)(sptr + (int64_t)((16 * st0) / groupsize) * N);
            s1[u] = *(const v8h*)(sptr + (int64_t)((16 * st1) / groupsize) * N);
            const int o1 = 2 * ks + 1 < strips ? 8 : 0;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                if constexpr (A_LDS) {
                    x[u][mt] = *(const v4i*)(alds + (16 * mt + r) * rstride + (ks - ks_begin) * 64 + g * 16);
                } else {
                    const unsigned* ap = (const unsigned*)(arow[mt] + 32 * ks);
                    x[u][mt] = (v4i){(int)ap[0], (int)ap[4], (int)ap[o1], (int)ap[o1 + 4]};
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);       // keep every load above ahead of the first use below
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int ks = ks0 + u * NW;
            const bool valid = ks < ks_end, valid1 = valid && 2 * ks + 1 < strips;
            v8h a[MT];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                a[mt] = make8(as_h2(valid ? (unsigned)x[u][mt][0] : 0u), as_h2(valid ? (unsigned)x[u][mt][1] : 0u),
                              as_h2(valid1 ? (unsigned)x[u][mt][2] : 0u), as_h2(valid1 ? (unsigned)x[u][mt][3] : 0u));
#pragma unroll
            for (int j = 0; j < 4; ++j) {
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    const int t = 2 * j + b;
                    const unsigned u0 = ((unsigned)w0[u][j]) >> (8 * b), u1 = ((unsigned)w1[u][j]) >> (8 * b);
                    const v2h sc0 = {s0[u][t], s0[u][t]}, sc1 = {s1[u][t], s1[u][t]};
                    const v8h bf = make8(deq_lo(u0) * sc0, deq_hi(u0) * sc0, deq_lo(u1) * sc1, deq_hi(u1) * sc1);
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) {
                        v4f d = {acc[(mt * 8 + t) * 4 + 0], acc[(mt * 8 + t) * 4 + 1], acc[(mt * 8 + t) * 4 + 2], acc[(mt * 8 + t) * 4 + 3]};
                        d = mfma_f16_16x16x32(a[mt], bf, d);
                        acc[(mt * 8 + t) * 4 + 0] = d[0]; acc[(mt * 8 + t) * 4 + 1] = d[1];
                        acc[(mt * 8 + t) * 4 + 2] = d[2]; acc[(mt * 8 + t) * 4 + 3] = d[3];
                    }
                }
            }
        }
    }

    // one-barrier reduction over the waves: slot e of lane l of wave w sits at red[(w * NE + e) * 64 + l]
    constexpr int NE = MT * 32;
    if constexpr (A_LDS) __syncthreads();                    // the reduction buffer reuses the activation image
#pragma unroll
    for (int e = 0; e < NE; ++e) red[(wave * NE + e) * 64 + lane] = acc[e];
    __syncthreads();
    for (int e = wave; e < NE; e += NW) {
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) v += red[(w * NE + e) * 64 + lane];
        const int mt = e >> 5, t = (e >> 2) & 7, i = e & 3;
        const int m = m0 + 16 * mt + 4 * g + i;
        const int n = 64 * chunk + 16 * (t >> 1) + 8 * (t & 1) + c;
        if (chunk_ok && m < M) {
            if constexpr (TO_WS) ws[((int64_t)blockIdx.z * M + m) * N + n] = v;
            else C[(int64_t)m * N + n] = (_Float16)v;
        }
    }
}

// four outputs per thread (MN is a multiple of 64): all Z partial vectors are requested before the first add
__global__ void splitk_reduce_f16_kernel(const float* __restrict__ ws, _Float16* __restrict__ C, int64_t MN, int Z) {
    const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (i >= MN) return;
    v4f s = {0.f, 0.f, 0.f, 0.f};
    int z = 0;
    for (; z + 8 <= Z; z += 8) {
        v4f t[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) t[j] = *(const v4f*)(ws + (int64_t)(z + j) * MN + i);
#pragma unroll
        for (int j = 0; j < 8; ++j) s += t[j];
    }
    for (; z < Z; ++z) s += *(const v4f*)(ws + (int64_t)z * MN + i);
    const v2h lo = {(_Float16)s[0], (_Float16)s[1]}, hi = {(_Float16)s[2], (_Float16)s[3]};
    unsigned u0, u1;
    __builtin_memcpy(&u0, &lo, 4);
    __builtin_memcpy(&u1, &hi, 4);
    *(uint2*)(C + i) = make_uint2(u0, u1);
}

// ------------------------------------------------------------------------------------------
// Marlin words -> dequantised fp16 W^T [N][K] (K contiguous), the operand layout of the tiled GEMM.
// One workgroup converts 8 strips (128 K) of one 64-column chunk: every thread expands one 16-byte unit
// (32 values, scaled in fp16 exactly as the fused kernels do), the tile is transposed through LDS and
// written as 256-byte row segments.
__global__ __launch_bounds__(256) void marlin_dequant_kernel(const v4i* __restrict__ B, const _Float16* __restrict__ S,
                                                             _Float16* __restrict__ Wt, int N, int K, int groupsize) {
    __shared__ __attribute__((aligned(16))) _Float16 tile[64][136];
    const int tid = threadIdx.x, sl = tid >> 5, ml = tid & 31, c = ml >> 2, q = ml & 3;
    const int nchunks = N >> 6, strips = K >> 4;
    const int chunk = blockIdx.x, strip = blockIdx.y * 8 + sl;
    if (strip < strips) {
        const v4i w = B[((int64_t)strip * nchunks + chunk) * 32 + ml];
        const v8h sc = *(const v8h*)(S + (int64_t)((16 * strip) / groupsize) * N + 64 * chunk + 8 * c);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const unsigned u = ((unsigned)w[j]) >> (8 * b);
                const v2h s2 = {sc[2 * j + b], sc[2 * j + b]};
                const int n = 16 * j + 8 * b + c, k = 16 * sl + 2 * q;
                *(v2h*)&tile[n][k] = deq_lo(u) * s2;
                *(v2h*)&tile[n][k + 8] = deq_hi(u) * s2;
            }
    }
    __syncthreads();
    // eight lanes write one 128-byte line of a row per instruction
    const int seg = tid & 7;
    const int k0 = blockIdx.y * 128;
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
        const int row = pass * 32 + (tid >> 3);
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            const int kl = x * 64 + seg * 8;
            if (k0 + kl < K)
                *(v8h*)(Wt + (int64_t)(64 * chunk + row) * K + k0 + kl) = *(const v8h*)&tile[row][kl];
        }
    }
}

// ------------------------------------------------------------------------------------------
// [N, K/8] layout (pack_weights_over_cols: nibble i of word w of row n is k = 8w + i) with
// scales [N, K/g].  Lane (r = column, g) loads one 16-byte unit = 32 consecutive k of its row per
// 128-K step; word j feeds MFMA j, whose fragment order is k offsets [0,4,1,5,2,6,3,7] -- the A
// fragment is permuted to the same order with v_perm_b32.
template <int MT, int NW>
__global__ __launch_bounds__(NW * 64) void w4a16_nk_kernel(
    const _Float16* __restrict__ A, const int32_t* __restrict__ B, const _Float16* __restrict__ S,
    _Float16* __restrict__ C, int M, int N, int K, int groupsize) {
    extern __shared__ float red[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * 16, m0 = blockIdx.y * 16 * MT;
    const int nrow = min(n0 + r, N - 1);
    const int steps = K >> 7;
    const int ngroups = K / groupsize;
    const int32_t* brow = B + (int64_t)nrow * (K >> 3) + 4 * g;
    const _Float16* srow = S + (int64_t)nrow * ngroups;
    const _Float16* arow[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) arow[mt] = A + (int64_t)min(m0 + 16 * mt + r, M - 1) * K + 32 * g;

    float acc[MT * 4];
#pragma unroll
    for (int i = 0; i < MT * 4; ++i) acc[i] = 0.f;

#pragma unroll 2
    for (int ks = wave; ks < steps; ks += NW) {
        const v4i w = *(const v4i*)(brow + ks * 16);
        const int kbase = ks * 128 + 32 * g;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const _Float16 sv = srow[(kbase + 8 * j) / groupsize];
            const v2h sc = {sv, sv};
            const unsigned u = (unsigned)w[j], u8 = u >> 8;
            const v8h bf = make8(deq_lo(u) * sc, deq_hi(u) * sc, deq_lo(u8) * sc, deq_hi(u8) * sc);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const v4i x = *(const v4i*)(arow[mt] + ks * 128 + 8 * j);
                v4i y;
                y[0] = (int)__builtin_amdgcn_perm((unsigned)x[2], (unsigned)x[0], 0x05040100u);  // k0,k4
                y[1] = (int)__builtin_amdgcn_perm((unsigned)x[2], (unsigned)x[0], 0x07060302u);  // k1,k5
                y[2] = (int)__builtin_amdgcn_perm((unsigned)x[3], (unsigned)x[1], 0x05040100u);  // k2,k6
                y[3] = (int)__builtin_amdgcn_perm((unsigned)x[3], (unsigned)x[1], 0x07060302u);  // k3,k7
                v8h a;
                __builtin_memcpy(&a, &y, 16);
                v4f d = {acc[mt * 4 + 0], acc[mt * 4 + 1], acc[mt * 4 + 2], acc[mt * 4 + 3]};
                d = mfma_f16_16x16x32(a, bf, d);
                acc[mt * 4 + 0] = d[0]; acc[mt * 4 + 1] = d[1]; acc[mt * 4 + 2] = d[2]; acc[mt * 4 + 3] = d[3];
            }
        }
    }
    reduce_waves<NW, MT * 4>(acc, red, wave, lane);
    if (wave != 0) return;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int m = m0 + 16 * mt + 4 * g + i, n = n0 + r;
            if (m < M && n < N) C[(int64_t)m * N + n] = (_Float16)acc[mt * 4 + i];
        }
}

// [N, K/8] words -> dequantised fp16 W [N][K] (the operand layout of the tiled GEMM): one thread expands one
// word (8 consecutive k of a row) and stores 16 bytes.
__global__ void nk_dequant_kernel(const int32_t* __restrict__ B, const _Float16* __restrict__ S, _Float16* __restrict__ W,
                                  int64_t N, int64_t K, int groupsize) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t kw = K >> 3;
    if (idx >= N * kw) return;
    const int64_t n = idx / kw, k = (idx - n * kw) * 8;
    const unsigned w = (unsigned)B[idx], w8 = w >> 8;
    const _Float16 sv = S[n * (K / groupsize) + k / groupsize];
    const v2h sc = {sv, sv};
    const unsigned p04 = as_u32(deq_lo(w) * sc), p15 = as_u32(deq_hi(w) * sc), p26 = as_u32(deq_lo(w8) * sc), p37 = as_u32(deq_hi(w8) * sc);
    v4i o;
    o[0] = (int)__builtin_amdgcn_perm(p15, p04, 0x05040100u);
    o[1] = (int)__builtin_amdgcn_perm(p37, p26, 0x05040100u);
    o[2] = (int)__builtin_amdgcn_perm(p15, p04, 0x07060302u);
    o[3] = (int)__builtin_amdgcn_perm(p37, p26, 0x07060302u);
    *(v4i*)(W + n * K + k) = o;
}

// The same for bf16 operands: (q - 8) * s formed in fp32 and rounded once to bf16, natural k order.
__global__ void nk_dequant_bf16_kernel(const int32_t* __restrict__ B, const _Float16* __restrict__ S,
                                       unsigned short* __restrict__ W, int64_t N, int64_t K, int groupsize) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t kw = K >> 3;
    if (idx >= N * kw) return;
    const int64_t n = idx / kw, k = (idx - n * kw) * 8;
    const unsigned w = (unsigned)B[idx];
    const float sc = (float)S[n * (K / groupsize) + k / groupsize];
    v4i o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float lo = (float)((int)((w >> (8 * i)) & 15u) - 8) * sc, hi = (float)((int)((w >> (8 * i + 4)) & 15u) - 8) * sc;
        o[i] = (int)pack_bf16x2(lo, hi);
    }
    *(v4i*)(W + n * K + k) = o;
}

// Weight-streaming variant of the [N, K/8] kernel for groupsize % 128 == 0 (every 128-K step lies in one
// scale group): persistent workgroups of 8 waves walk 16-column tiles; the waves split K by interleaved
// 128-K steps in batches of U, all loads of a batch issued before its first use and the weights of the next
// two tiles requested ahead.  When a wave's K share fits one batch (RESIDENT) its activation fragments are
// loaded and permuted once and stay in registers for every tile.  The group scale multiplies the fp32
// partial of the step (one FMA per output) instead of the eight fp16 weights.
template <int MT, int NT, bool RESIDENT, bool VS = false>
__global__ __launch_bounds__(512) void w4a16_nk_stream_kernel(
    const _Float16* __restrict__ A, const int32_t* __restrict__ B, const _Float16* __restrict__ S,
    _Float16* __restrict__ C, int M, int N, int Kfull, int groupsize, int Kc, float* __restrict__ partial) {
    constexpr int NW = 8;
    constexpr int U = MT == 1 ? 4 : (MT == 2 ? 2 : 1);
    extern __shared__ float red[];                       // [2][NW][NT][MT][64][4]
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, g = lane >> 4;
    // K range [k0, k0 + K) of this workgroup (gridDim.z ranges of Kc cover rows that are Kfull long; with more
    // than one range the outputs are fp32 partial sums for a summing pass)
    const int k0 = (int)blockIdx.z * Kc, K = min(Kc, Kfull - k0);
    const int steps = K >> 7, ngroups = Kfull / groupsize, kwords = Kfull >> 3;
    const int m0 = blockIdx.y * 16 * MT;
    const int ntiles = (N + 16 * NT - 1) / (16 * NT);    // a tile is NT adjacent 16-column blocks

    const _Float16* arow[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) arow[mt] = A + (int64_t)min(m0 + 16 * mt + r, M - 1) * Kfull + k0 + 32 * g;

    struct BBatch {
        v4i w[NT][U];
        unsigned short s[NT][U];
        uint2 sv[NT];          // VS: the four scales of the batch as loaded (unpacked when the batch is multiplied:
                               // any arithmetic on a value still in flight would wait for it right away)
    };
    struct ABatch {
        v4i a[U][MT][4];
    };
    // step u of the batch that starts at ks0 (= first step of the batch + wave).  VS: every wave takes U
    // consecutive steps and, with 128-wide groups, fetches their four scales with one load.
    auto step_of = [&](int ks0, int u) { return VS ? (ks0 - wave) + wave * U + u : ks0 + u * NW; };
    auto clamp_step = [&](int ks) { return min(ks, steps - 1); };
    // Addresses are a wave-uniform base (tile, K step: scalar registers) plus one 32-bit offset per lane, so that
    // a load needs no 64-bit per-lane address arithmetic and no address registers that could collide with
    // the destinations of loads still in flight.  Rows past N in the last tile repeat the last row.
    auto load_b = [&](BBatch& t, int tile, int ks0) __attribute__((always_inline)) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const int rowbase = (tile * NT + nt) * 16;
            const uint32_t lo = (uint32_t)min(r, N - 1 - rowbase) * (uint32_t)(kwords * 4) + 16u * (uint32_t)g;
            const char* tb = (const char*)B + ((int64_t)rowbase * kwords + (k0 >> 3)) * 4;
#pragma unroll
            for (int u = 0; u < U; ++u) t.w[nt][u] = *(const v4i*)(tb + (int64_t)clamp_step(step_of(ks0, u)) * 64 + lo);
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const int rowbase = (tile * NT + nt) * 16;
            const uint32_t lo = (uint32_t)min(r, N - 1 - rowbase) * (uint32_t)(ngroups * 2);
            const char* sb = (const char*)S + (int64_t)rowbase * ngroups * 2;
            if constexpr (VS) {
                static_assert(U == 4, "four scales per load");
                t.sv[nt] = *(const uint2*)(sb + (int64_t)((k0 >> 7) + min(step_of(ks0, 0), steps - U)) * 2 + lo);
            } else {
#pragma unroll
                for (int u = 0; u < U; ++u)
                    t.s[nt][u] = *(const unsigned short*)(sb + (int64_t)((k0 + clamp_step(step_of(ks0, u)) * 128) / groupsize) * 2 + lo);
            }
        }
    };
    auto load_a = [&](ABatch& t, int ks0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int j = 0; j < 4; ++j) t.a[u][mt][j] = *(const v4i*)(arow[mt] + clamp_step(step_of(ks0, u)) * 128 + 8 * j);
    };
    // k order of a dequantised word is [0,4,1,5,2,6,3,7]: bring the activation fragment into the same order
    auto perm_a = [&](ABatch& t) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const v4i x = t.a[u][mt][j];
                    v4i y;
                    y[0] = (int)__builtin_amdgcn_perm((unsigned)x[2], (unsigned)x[0], 0x05040100u);
                    y[1] = (int)__builtin_amdgcn_perm((unsigned)x[2], (unsigned)x[0], 0x07060302u);
                    y[2] = (int)__builtin_amdgcn_perm((unsigned)x[3], (unsigned)x[1], 0x05040100u);
                    y[3] = (int)__builtin_amdgcn_perm((unsigned)x[3], (unsigned)x[1], 0x07060302u);
                    t.a[u][mt][j] = y;
                }
    };
    auto mul = [&](const ABatch& ta, const BBatch& tb, int ks0, v4f (&acc)[NT][MT]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool valid = step_of(ks0, u) < steps;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                unsigned short sraw;
                if constexpr (VS) sraw = (unsigned short)((u < 2 ? tb.sv[nt].x : tb.sv[nt].y) >> (16 * (u & 1)));
                else sraw = tb.s[nt][u];
                const float sc = valid ? f16_to_f32(sraw) : 0.f;
                v4f t[MT];
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) t[mt] = (v4f){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const unsigned w = (unsigned)tb.w[nt][u][j], w8 = w >> 8;
                    const v8h bf = make8(deq_lo(w), deq_hi(w), deq_lo(w8), deq_hi(w8));
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) {
                        v8h a;
                        __builtin_memcpy(&a, &ta.a[u][mt][j], 16);
                        t[mt] = mfma_f16_16x16x32(a, bf, t[mt]);
                    }
                }
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) acc[nt][mt] += t[mt] * sc;
            }
        }
    };

    int tile = blockIdx.x;
    const int stride = gridDim.x;
    ABatch acur, anxt;
    BBatch bcur, bnxt, bnx2;
    // Every load of the ring is issued unconditionally (a tile index past the end is clamped to the last tile,
    // whose lines are then in cache): with loads under a condition the compiler cannot tell how many are in
    // flight and waits for all of them, the one just requested included, before it touches any.
    if (tile < ntiles) {
        // activations first (mostly L2 hits): they are permuted while the weights are still on their way
        load_a(acur, wave);
        load_b(bcur, tile, wave);
        if (RESIDENT) load_b(bnxt, min(tile + stride, ntiles - 1), wave);
        __builtin_amdgcn_sched_barrier(0);
        if (RESIDENT) perm_a(acur);
    }
    constexpr int NB = NT * MT;                          // 16x16 blocks per tile
    int parity = 0;
    v4f acc[NT][MT];
    auto clear_acc = [&]() {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = (v4f){0.f, 0.f, 0.f, 0.f};
    };
    // cross-wave reduction of the K split, two alternating buffers: one barrier per tile
    auto finish = [&](int tl) __attribute__((always_inline)) {
        float* rbuf = red + parity * NW * NB * 256;
        parity ^= 1;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) *(v4f*)(rbuf + ((wave * NB + nt * MT + mt) * 64 + lane) * 4) = acc[nt][mt];
        __syncthreads();
        for (int o = threadIdx.x; o < NB * 256; o += NW * 64) {
            const int blk = o >> 8, nt = blk / MT, mt = blk - nt * MT, row16 = (o & 255) >> 4, col = o & 15;
            const int src = (blk * 64 + (row16 >> 2) * 16 + col) * 4 + (row16 & 3);
            const int m = m0 + 16 * mt + row16, n = (tl * NT + nt) * 16 + col;
            if (m >= M || n >= N) continue;
            float v = 0.f;
#pragma unroll
            for (int w = 0; w < NW; ++w) v += rbuf[w * NB * 256 + src];
            if (partial) partial[((int64_t)blockIdx.z * M + m) * N + n] = v;
            else C[(int64_t)m * N + n] = (_Float16)v;
        }
        clear_acc();
    };
    clear_acc();
    // The batches form a ring that is never copied (a register copy of a batch whose loads are in flight
    // would wait for them).
    if constexpr (RESIDENT) {
        auto one = [&](BBatch& cur, BBatch& fill) __attribute__((always_inline)) {
            load_b(fill, min(tile + 2 * stride, ntiles - 1), wave);
            mul(acur, cur, wave, acc);
            finish(tile);
            tile += stride;
        };
        while (tile < ntiles) {
            one(bcur, bnx2);
            if (tile >= ntiles) break;
            one(bnxt, bcur);
            if (tile >= ntiles) break;
            one(bnx2, bnxt);
        }
    } else {
        int ks0 = wave;
        auto one = [&](ABatch& ca, BBatch& cb, ABatch& fa, BBatch& fb) __attribute__((always_inline)) {
            const int nk = ks0 + NW * U;
            const bool more = step_of(nk, 0) < steps;
            const int nt = more ? tile : tile + stride;
            const bool any = nt < ntiles;
            const int fk = more ? nk : wave;
            if (any) { load_b(fb, nt, fk); load_a(fa, fk); }
            perm_a(ca);                                  // permuted when it becomes current, not while in flight
            mul(ca, cb, ks0, acc);
            if (!more) finish(tile);
            tile = nt;
            ks0 = more ? nk : wave;
        };
        while (tile < ntiles) {
            one(acur, bcur, anxt, bnxt);
            if (tile >= ntiles) break;
            one(anxt, bnxt, acur, bcur);
        }
    }
}

// Ring variant of the weight-streaming kernel for 128-wide groups, at most 16 rows per workgroup and a K range
// of 4 to 32 steps: wave w owns U = ceil(steps / 8) consecutive 128-K steps from U w of every
// 16-column tile, its activation fragments stay in registers, and the packed words and group scales of the
// next DEPTH - 1 tiles are in flight in a ring of registers filled by hand-issued loads (see stream_ring.hpp:
// one s_waitcnt per tile that leaves exactly the younger tiles outstanding).
// Every wave loads U steps, so that one wait count serves all: where fewer are left in the range the share is moved
// back to its last U steps (the repeated ones hit L2) and the steps that another wave owns count as zero activations
// and zero scales.  (Ranges that are no multiple of
// 512 went through a bf16 copy of W, or the stream kernel for fp16; us per call, cold weights: bf16 3 x 4672 x 9088
// 70.6 -> 14.8, 16 x 14336 x 2176 32.7 -> 11.7, 60 x 24000 x 3968 90.0 -> 36.7; fp16 15.1 -> 15.3, 13.2 -> 12.4, 50.2 -> 41.1.)
// BF: bf16 activations and outputs.  A nibble becomes the bf16 number 128 + q by OR-ing it into 0x4300 (exact:
// seven mantissa bits, q < 16), and the missing "- 136" of every product is the accumulator the MFMA chain of a
// step starts from: -136 * sum_k a[m][k] over the step, computed once per wave with the same MFMA and a weight
// fragment of constant 136 (the same for every tile).
// (U = 4 for every K before; us per call: 16 x 28672 x 1024 13.6 -> 6.9, fp16 60 x 28672 x 1024 43.2 -> 15.6, 16 x 25600 x 1408
// 13.9 -> 9.4, 16 x 4096 x 1024 5.2 -> 3.3, 60 x 15368 x 3072 25.0 -> 20.4, 3 x 4672 x 9088 in three ranges 14.9 -> 12.8.)
// FULL: every range is 8 U steps, so no share is moved back and nothing counts as zero.  The general form's selects cost such
// a range up to 1.7 % (us, cold weights, before it | with it | FULL: bf16 16 x 6144 x 4096 7.73 | 7.86 | 7.72, 48 x 4096 x 4096
// 10.57 | 10.70 | 10.55, 16 x 4096 x 4096 5.92 | 5.95 | 5.94; fp16 7.82 | 7.86 | 7.76).  Taken for U = 4, the range of 4096
// elements: with U = 2 it measured slower (bf16 16 x 4096 x 2048 4.15 -> 4.37).
template <int DEPTH, int U, bool FULL, bool BF>
__global__ __launch_bounds__(512) void w4a16_nk_ring_kernel(
    const unsigned short* __restrict__ A, const int32_t* __restrict__ B, const _Float16* __restrict__ S,
    unsigned short* __restrict__ C, int M, int N, int Kfull, int Kc, float* __restrict__ partial) {
    using namespace llmk;
    constexpr int NW = 8, LPT = U + 1;                   // loads per tile and lane: U word vectors + the scales
    extern __shared__ float red[];                       // [2][NW][64][4]
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int k0 = (int)blockIdx.z * Kc, K = min(Kc, Kfull - k0);
    const int steps = K >> 7, ngroups = Kfull >> 7, kwords = Kfull >> 3;
    const int m0 = blockIdx.y * 16;
    const int ntiles = (N + 15) >> 4;
    const int s0 = FULL ? U * wave : min(U * wave, steps - U);           // first step this wave loads
    const int u0 = FULL ? 0 : min(U * wave - s0, U);     // steps s0 .. s0 + u0 - 1 belong to other waves

    // ---- activations, requested first: row i of the wave's K slice (512 elements = 1 KiB) is one fully
    // coalesced load.  (Fetching the MFMA fragments straight from global memory costs 2 us per launch: every
    // 16-lane group of such a load touches 16 different cache lines, 16 bytes of each.)  They pass through a
    // wave-private LDS area once and stay in registers as fragments for every tile.
    v4i a[4 * U];
    {
        // load 4 u + q: rows 4 q .. 4 q + 3 of the 256-byte slab of step u (a 16-lane group reads 256 contiguous bytes)
        const RingBase ab = ring_base((const char*)A + ((int64_t)k0 + s0 * 128) * 2);
        const uint32_t rowb = (uint32_t)(Kfull * 2), lrow = (uint32_t)(lane >> 4), lcol = 16u * (uint32_t)(lane & 15);
#define LLMK_LDA(u, q) a[4 * u + q] = ring_load_b128<u * 256>((uint32_t)min(m0 + 4 * q + (int)lrow, M - 1) * rowb + lcol, ab)
        LLMK_LDA(0, 0); LLMK_LDA(0, 1); LLMK_LDA(0, 2); LLMK_LDA(0, 3);
        if constexpr (U > 1) { LLMK_LDA(1, 0); LLMK_LDA(1, 1); LLMK_LDA(1, 2); LLMK_LDA(1, 3); }
        if constexpr (U > 2) { LLMK_LDA(2, 0); LLMK_LDA(2, 1); LLMK_LDA(2, 2); LLMK_LDA(2, 3); }
        if constexpr (U > 3) { LLMK_LDA(3, 0); LLMK_LDA(3, 1); LLMK_LDA(3, 2); LLMK_LDA(3, 3); }
#undef LLMK_LDA
    }
    // ---- ring of weight tiles
    v4i w[DEPTH][U];
    v2i sv[DEPTH];
    const char* bb = (const char*)B + ((int64_t)(k0 >> 3) + s0 * 16) * 4;
    const int sq = U == 4 ? s0 : min(s0, steps - 4);                   // the scales of four steps are loaded, this wave's among them
    const char* sb = (const char*)S + ((int64_t)(k0 >> 7) + sq) * 2;
    auto issue = [&](v4i (&tw)[U], v2i& ts, int tile) __attribute__((always_inline)) {
        const int rowbase = tile * 16;
        const uint32_t row = (uint32_t)min(r, N - 1 - rowbase);             // rows past N repeat the last row
        const uint32_t vo = row * (uint32_t)(kwords * 4) + 16u * (uint32_t)g;
        const RingBase tb = ring_base(bb + (int64_t)rowbase * kwords * 4);
        tw[0] = ring_load_b128<0>(vo, tb);
        if constexpr (U > 1) tw[1] = ring_load_b128<64>(vo, tb);
        if constexpr (U > 2) tw[2] = ring_load_b128<128>(vo, tb);
        if constexpr (U > 3) tw[3] = ring_load_b128<192>(vo, tb);
        ts = ring_load_b64<0>(row * (uint32_t)(ngroups * 2), ring_base(sb + (int64_t)rowbase * ngroups * 2));
    };
    int tile = blockIdx.x;
    const int stride = gridDim.x, last = ntiles - 1;
#pragma unroll
    for (int d = 0; d < DEPTH - 1; ++d) issue(w[d], sv[d], min(tile + d * stride, last));
    // the activations were requested before (DEPTH - 1) * LPT ring loads
#pragma unroll
    for (int i = 0; i < 4 * U; ++i) ring_wait<(DEPTH - 1) * LPT>(a[i]);
    {
        // one slab (16 rows x 256 bytes) at a time through the wave's LDS area; rows of 256 + 16 bytes, so that
        // the 16 rows of a fragment read fall into 16 different bank groups
        constexpr int AROW = 256 + 16;
        uint8_t* stage = (uint8_t*)red + 2 * NW * 256 * sizeof(float) + wave * (16 * AROW);
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int q = 0; q < 4; ++q) *(v4i*)(stage + (4 * q + (lane >> 4)) * AROW + 16 * (lane & 15)) = a[4 * u + q];
            // fragment (u, j) of lane (r, g): elements 128 u + 32 g + 8 j .. + 7 of row r.  The k order of a
            // dequantised word is [0,4,1,5,2,6,3,7]: bring the activation fragment into the same order.
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const v4i x = *(const v4i*)(stage + r * AROW + 64 * g + 16 * j);
                v4i y;
                y[0] = (int)__builtin_amdgcn_perm((unsigned)x[2], (unsigned)x[0], 0x05040100u);
                y[1] = (int)__builtin_amdgcn_perm((unsigned)x[2], (unsigned)x[0], 0x07060302u);
                y[2] = (int)__builtin_amdgcn_perm((unsigned)x[3], (unsigned)x[1], 0x05040100u);
                y[3] = (int)__builtin_amdgcn_perm((unsigned)x[3], (unsigned)x[1], 0x07060302u);
                a[4 * u + j] = y;
            }
        }
        if (!FULL && u0 > 0) {
#pragma unroll
            for (int i = 0; i < 4 * U; ++i)
                if (i < 4 * u0) a[i] = (v4i){0, 0, 0, 0};
        }
    }

    // bf16: the bias of step u, -136 * sum_k a[row][k] in every column of the MFMA result
    v4f bias[U];
#pragma unroll
    for (int u = 0; u < U; ++u) bias[u] = (v4f){0.f, 0.f, 0.f, 0.f};
    if constexpr (BF) {
        const v4i c136 = {(int)0xc308c308u, (int)0xc308c308u, (int)0xc308c308u, (int)0xc308c308u};   // bf16 -136
        v8bf neg136;
        __builtin_memcpy(&neg136, &c136, 16);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                v8bf af;
                __builtin_memcpy(&af, &a[4 * u + j], 16);
                bias[u] = mfma_bf16_16x16x32(af, neg136, bias[u]);
            }
    }

    int parity = 0;
    auto tile_done = [&](const v4i (&tw)[U], const v2i& ts, int tl) __attribute__((always_inline)) {
        v4f acc = {0.f, 0.f, 0.f, 0.f};
        uint64_t sc4 = 0;
        if constexpr (U < 4) sc4 = ((uint64_t)(uint32_t)ts[1] << 32 | (uint32_t)ts[0]) >> (16 * (s0 - sq));
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const unsigned sraw = (U < 4 ? (unsigned)(sc4 >> (16 * u)) : (unsigned)(u < 2 ? ts[0] : ts[1]) >> (16 * (u & 1))) & 0xffffu;
            const float sc = !FULL && u < u0 ? 0.f : f16_to_f32((unsigned short)sraw);
            v4f t = bias[u];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const unsigned x = (unsigned)tw[u][j];
                if constexpr (BF) {
                    // element pairs (k0,k4) (k1,k5) (k2,k6) (k3,k7) of the word, as for fp16
                    v4i bw;
                    bw[0] = (int)((x & 0x000f000fu) | 0x43004300u);
                    bw[1] = (int)(((x >> 4) & 0x000f000fu) | 0x43004300u);
                    bw[2] = (int)(((x >> 8) & 0x000f000fu) | 0x43004300u);
                    bw[3] = (int)(((x >> 12) & 0x000f000fu) | 0x43004300u);
                    v8bf bf, af;
                    __builtin_memcpy(&bf, &bw, 16);
                    __builtin_memcpy(&af, &a[4 * u + j], 16);
                    t = mfma_bf16_16x16x32(af, bf, t);
                } else {
                    const unsigned x8 = x >> 8;
                    const v8h bf = make8(deq_lo(x), deq_hi(x), deq_lo(x8), deq_hi(x8));
                    v8h af;
                    __builtin_memcpy(&af, &a[4 * u + j], 16);
                    t = mfma_f16_16x16x32(af, bf, t);
                }
            }
            acc += t * sc;
        }
        // cross-wave reduction of the K split, two alternating buffers: one barrier per tile
        float* rbuf = red + parity * NW * 256;
        parity ^= 1;
        *(v4f*)(rbuf + (wave * 64 + lane) * 4) = acc;
        __syncthreads();
        const int o = threadIdx.x;
        if (o < 256) {
            const int row16 = o >> 4, col = o & 15;
            const int src = ((row16 >> 2) * 16 + col) * 4 + (row16 & 3);
            const int m = m0 + row16, n = tl * 16 + col;
            float v = 0.f;
#pragma unroll
            for (int ww = 0; ww < NW; ++ww) v += rbuf[ww * 256 + src];
            if (m < M && n < N) {
                if (partial) partial[((int64_t)blockIdx.z * M + m) * N + n] = v;
                else C[(int64_t)m * N + n] = BF ? f32_to_bf16(v) : f32_to_f16(v);
            }
        }
    };
    // (the loop is left behind a full wait: no path of the flow graph may lead from a request back to the loop
    // head without passing a wait that covers it, and the clamped requests of the last tiles are drained)
    // Whole rounds of DEPTH tiles run in a loop whose body has no branch (every request and every wait is
    // executed on every path, so what the static check of the assembly sees is what runs); the last
    // my_tiles % DEPTH tiles, all requested by then, follow as straight-line code.  Requests past the last tile
    // of the workgroup are clamped to the last tile of the matrix (cache hits) and never consumed.
    const int my_tiles = (ntiles - (int)blockIdx.x + stride - 1) / stride;
    auto landed = [&](auto nc, v4i (&tw)[U], v2i& ts) __attribute__((always_inline)) {
        if constexpr (U == 4) {
            ring_wait<decltype(nc)::value>(tw[0], tw[1], tw[2], tw[3], ts);
        } else {
#pragma unroll
            for (int u = 0; u < U; ++u) ring_wait<decltype(nc)::value>(tw[u]);
            ring_wait<decltype(nc)::value>(ts);
        }
    };
    auto slot = [&](auto dc) __attribute__((always_inline)) {
        constexpr int d = decltype(dc)::value, NEXT = DEPTH - 1;
        issue(w[(d + NEXT) % DEPTH], sv[(d + NEXT) % DEPTH], min(tile + NEXT * stride, last));
        landed(std::integral_constant<int, (DEPTH - 1) * LPT>{}, w[d], sv[d]);
        tile_done(w[d], sv[d], tile);
        tile += stride;
    };
    auto tail = [&](auto dc) __attribute__((always_inline)) {
        constexpr int d = decltype(dc)::value;
        landed(std::integral_constant<int, (DEPTH - 2 - d) * LPT>{}, w[d], sv[d]);
        tile_done(w[d], sv[d], tile);
        tile += stride;
    };
    static_assert(DEPTH >= 2 && DEPTH <= 4, "ring slots are spelled out below");
    for (int rd = my_tiles / DEPTH; rd > 0; --rd) {
        slot(std::integral_constant<int, 0>{});
        if constexpr (DEPTH > 1) slot(std::integral_constant<int, 1>{});
        if constexpr (DEPTH > 2) slot(std::integral_constant<int, 2>{});
        if constexpr (DEPTH > 3) slot(std::integral_constant<int, 3>{});
    }
    const int rem = my_tiles % DEPTH;
    if constexpr (DEPTH > 1) { if (rem > 0) tail(std::integral_constant<int, 0>{}); }
    if constexpr (DEPTH > 2) { if (rem > 1) tail(std::integral_constant<int, 1>{}); }
    if constexpr (DEPTH > 3) { if (rem > 2) tail(std::integral_constant<int, 2>{}); }
    ring_drain<0>();
}

// The ring kernel takes 128-wide groups, K ranges of 4 to 32 steps (the last one takes what is left) and operands below
// 4 GiB (32-bit lane offsets); nz = number of K ranges.  The four group scales of a share are one 8-byte load at a
// multiple of two bytes: scale rows of any length (K / 128 not a multiple of four) are read as they lie.
bool nk_ring_ok(int64_t M, int64_t N, int64_t K, int groupsize, int nz) {
    const int64_t steps_all = K >> 7, steps = (steps_all + nz - 1) / nz, last = steps_all - (nz - 1) * steps;
    return groupsize == 128 && steps <= 32 && last >= 4 && N * (K / 2) < (1ll << 32) && M * K * 2 < (1ll << 32);
}

// fp16 or bf16 (bf) activations / outputs; partial: fp32 planes for nz > 1 (a summing pass follows)
int launch_nk_ring(const void* A, const int32_t* B, const _Float16* S, void* C, int M, int N, int K, int nz, float* partial,
                   bool bf, hipStream_t st) {
    const int steps_all = K >> 7, steps = (steps_all + nz - 1) / nz, Kc = steps * 128;
    const int ntiles = (N + 15) / 16, mtiles = (M + 15) / 16, rows = mtiles * nz;
    // One workgroup per CU and row tile, ring depth = tiles per workgroup (two to four).  Two workgroups per CU
    // with rings of two measured slower (20.4 vs 18.2 us at N = 28672): every workgroup reads all the activations
    // of its row tile, and that traffic doubles.
    const int cus = std::max(1, llmk_device_cus() > 0 ? llmk_device_cus() : LLMK_CUS);
    const int wg = min(ntiles, max(1, cus / min(rows, cus)));
    const int per_wg = (ntiles + wg - 1) / wg;
    dim3 rgrid((unsigned)((ntiles + per_wg - 1) / per_wg), (unsigned)mtiles, (unsigned)nz);
    // reduction buffers + the wave-private staging area of the activations
    const size_t rsmem = 2 * 8 * 256 * sizeof(float) + 8 * 16 * (256 + 16);
    const unsigned short* a16 = (const unsigned short*)A;
    unsigned short* c16 = (unsigned short*)C;
    float* part = nz > 1 ? partial : nullptr;
    auto ring = [&](auto uc) {
        constexpr int U = decltype(uc)::value;
        auto run = [&](auto kern) { kern<<<rgrid, 512, rsmem, st>>>(a16, B, S, c16, M, N, K, Kc, part); };
        auto form = [&](auto full) {
            constexpr bool FULL = decltype(full)::value;
            if (per_wg >= 4) bf ? run(w4a16_nk_ring_kernel<4, U, FULL, true>) : run(w4a16_nk_ring_kernel<4, U, FULL, false>);
            else if (per_wg == 3) bf ? run(w4a16_nk_ring_kernel<3, U, FULL, true>) : run(w4a16_nk_ring_kernel<3, U, FULL, false>);
            else bf ? run(w4a16_nk_ring_kernel<2, U, FULL, true>) : run(w4a16_nk_ring_kernel<2, U, FULL, false>);
        };
        if constexpr (U == 4) {
            if (steps == 8 * U && steps_all == nz * steps) return form(std::true_type{});
        }
        form(std::false_type{});
    };
    if (steps <= 8) ring(std::integral_constant<int, 1>{});
    else if (steps <= 16) ring(std::integral_constant<int, 2>{});
    else if (steps <= 24) ring(std::integral_constant<int, 3>{});
    else ring(std::integral_constant<int, 4>{});
    LLMK_CHECK_LAUNCH("gemm_w4a16_nk(ring)");
    if (nz > 1) {
        const int64_t mn = (int64_t)M * N;
        if (bf) llmk::splitk_sum_kernel<LLMK_BF16><<<(unsigned)cdiv64(cdiv64(mn, 4), 256), 256, 0, st>>>(partial, C, mn, nz);
        else splitk_reduce_f16_kernel<<<(unsigned)cdiv64(mn, 4 * 256), 256, 0, st>>>(partial, (_Float16*)C, mn, nz);
        LLMK_CHECK_LAUNCH("gemm_w4a16_nk(reduce)");
    }
    return LLMK_OK;
}

template <int MT, int NT>
int launch_nk_stream(const _Float16* A, const int32_t* B, const _Float16* S, _Float16* C, int M, int N, int K, int groupsize,
                     int nz, float* partial, hipStream_t st) {
    if constexpr (MT == 1 && NT == 1) {
        if (nk_ring_ok(M, N, K, groupsize, nz)) return launch_nk_ring(A, B, S, C, M, N, K, nz, partial, false, st);
    }
    constexpr int U = MT == 1 ? 4 : (MT == 2 ? 2 : 1);
    // nz K ranges, equally long up to one step
    const int steps_all = K >> 7, steps = (steps_all + nz - 1) / nz, Kc = steps * 128;
    const int ntiles = (N + 16 * NT - 1) / (16 * NT), mtiles = (M + 16 * MT - 1) / (16 * MT);
    const bool resident = steps <= 8 * U;
    const size_t smem = (size_t)2 * 8 * NT * MT * 256 * sizeof(float);
    static std::atomic<int> slots_cache[2];
    int slots[2] = {slots_cache[0].load(std::memory_order_relaxed), slots_cache[1].load(std::memory_order_relaxed)};
    if (slots[resident] == 0) {
        int dev = 0, cus = 0, per_cu = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
        if (e == hipSuccess)
            e = resident ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, w4a16_nk_stream_kernel<MT, NT, true>, 512, smem)
                         : hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, w4a16_nk_stream_kernel<MT, NT, false>, 512, smem);
        if (e != hipSuccess) LLMK_FAIL(LLMK_ERR_LAUNCH, "gemm_w4a16_nk: occupancy query failed: %s", hipGetErrorString(e));
        slots[resident] = max(1, cus * max(1, per_cu));
        slots_cache[resident].store(slots[resident], std::memory_order_relaxed);
    }
    const int rows = mtiles * nz;
    int gx = min(ntiles, max(1, slots[resident] / min(rows, slots[resident])));
    { const int per_wg = (ntiles + gx - 1) / gx; gx = (ntiles + per_wg - 1) / per_wg; }   // equal tile counts
    dim3 grid((unsigned)gx, (unsigned)mtiles, (unsigned)nz);
    float* part = nz > 1 ? partial : nullptr;
    bool launched = false;
    if constexpr (U == 4) {
        // consecutive steps per wave and one load for their four scales
        if (!launched && groupsize == 128 && steps_all % 4 == 0 && steps % 4 == 0 && !(((uintptr_t)S) & 7)) {
            if (resident) w4a16_nk_stream_kernel<MT, NT, true, true><<<grid, 512, smem, st>>>(A, B, S, C, M, N, K, groupsize, Kc, part);
            else w4a16_nk_stream_kernel<MT, NT, false, true><<<grid, 512, smem, st>>>(A, B, S, C, M, N, K, groupsize, Kc, part);
            launched = true;
        }
    }
    if (!launched) {
        if (resident) w4a16_nk_stream_kernel<MT, NT, true><<<grid, 512, smem, st>>>(A, B, S, C, M, N, K, groupsize, Kc, part);
        else w4a16_nk_stream_kernel<MT, NT, false><<<grid, 512, smem, st>>>(A, B, S, C, M, N, K, groupsize, Kc, part);
    }
    LLMK_CHECK_LAUNCH("gemm_w4a16_nk(stream)");
    if (nz > 1) {
        splitk_reduce_f16_kernel<<<(unsigned)cdiv64((int64_t)M * N, 4 * 256), 256, 0, st>>>(partial, C, (int64_t)M * N, nz);
        LLMK_CHECK_LAUNCH("gemm_w4a16_nk(reduce)");
    }
    return LLMK_OK;
}

// Rows for which the 128-column tile kernels expand the 4-bit weights themselves: 65 to 512 always (measured
// 1.3-2.8x faster than the separate expansion pass up to 256 rows, even to 1.4x at 512); 33 to 64 when the
// weight matrix is large, where the tile kernel with split-K beats the weight-streaming kernels (which read
// the activations once per 16 columns), provided the scratch for its partial sums is there.
// `wide`: the layout also has the expansion inside the 256-column tile kernel (row-packed layout only).  Up to 512
// rows the fused tile kernels win everywhere (1.3-2.8x).  Up to 1024 rows, where the separate pass is a good part of the
// call, by the estimates of the tile shapes (1.65 x for 16-bit operands) against that pass, N * 1.86e-3 us at K = 4096 (2.5
// bytes per weight at 5.5 TB/s), and the plain 16-bit GEMM: bf16 600 x 28672 x 4096 242 us in two passes, 192 fused, 1024 x
// 14336 x 4096 122 and 105.  Beyond, every row tile expands the weights again and the fused form needs two rounds of
// 256 x 256 tiles to win (fp16 4096 x 28672 x 4096: 741 vs 758 us, 2048 x 14336 x 4096: 198 vs 201; on one round 1300 x 6144
// x 4096: 119 vs 86), the dearer bf16 expansion at most 2048 rows as well (1500 x 28672 x 4096: 319 vs 344, 4096 rows: 775 vs 762).
bool w4_tiles_expand(int64_t M, int64_t N, int64_t K, int64_t scratch, bool wide = false, bool bf = false) {
    if (M > 512) {
        if (!wide) return false;
        if (M > 1024) return ((M + 255) / 256) * ((N + 255) / 256) >= 512 && (!bf || M <= 2048);
        llmk::DirectArgs p{};
        p.M = (int)M; p.N = (int)N; p.K = (int)K; p.E = 1;
        const double fused = bf ? llmk::dma_tile_estimate<llmk::K_W4NKB, false>(p).cost : llmk::dma_tile_estimate<llmk::K_W4NK, false>(p).cost;
        return 1.65 * fused < 1.65 * llmk::dma_tile_estimate<llmk::K_F16, false>(p).cost + (double)N * 1.86e-3;
    }
    if (M > 64) return true;
    if (M <= 32 || K % 64) return false;
    const int64_t nk = N * K;
    if (!(K > 4096 ? nk >= ((int64_t)32 << 20) : nk >= ((int64_t)96 << 20))) return false;
    const int z = llmk::splitk_factor_half(M, N, K);
    return z <= 1 || scratch >= (int64_t)z * M * N * 4;
}

// what of a caller's workspace the kernels can use
int64_t usable_scratch(const void* workspace, int64_t bytes) { return workspace && !((uintptr_t)workspace & 15) ? bytes : 0; }

// Mid-size M (and large M on many tiles): the tile kernels expand the row-packed words themselves, so every weight byte is
// read once; the separate expansion pass would write and re-read four times as much (bf16, 300 x 14336 x 4096: 26 us of
// pass and 51 us of GEMM, 58 us in one kernel).  Which of them a shape takes, and its K slices:
struct NkTiles {
    enum { MID, MIDW, BIG } form;
    int mt, z;
};
template <int KIND>
NkTiles nk_tiles(const llmk::DirectArgs& p) {
    const int64_t M = p.M, N = p.N, K = p.K;
    // few column tiles and short rows: the 64-column kernel with 512-byte K steps (128 x 4096 x 4096: 18.3 -> 14 us)
    if (2 * K <= 8192 && llmk::mid_wanted(M, N, 2 * K)) {       // (rows beyond 8 KB: measured only for the 8-bit kinds)
        const llmk::MidPlan pl = llmk::mid_plan(M, N, 2 * K);
        if (llmk::mid_eligible<KIND>(p)) return {NkTiles::MID, pl.mt, pl.z};
    }
    // wider weights on one round of 128-column tiles: the 128-column form of that kernel
    if (2 * K <= 8192 && llmk::midw_wanted(M, N, 2 * K) && (p.group & (p.group - 1)) == 0) {       // (longer rows: measured for fp8 only)
        const llmk::MidPlan pl = llmk::midw_plan(M, N, 2 * K);
        return {NkTiles::MIDW, pl.mt, pl.z};
    }
    return {NkTiles::BIG, 0, llmk::splitk_factor_half(M, N, K)};
}
template <int KIND>
int launch_nk_tiles(llmk::DirectArgs p, void* workspace, int64_t scratch, hipStream_t st) {
    const NkTiles t = nk_tiles<KIND>(p);
    if (t.form == NkTiles::BIG) return llmk::launch_big_half<KIND, false>(p, st, "gemm_w4a16_nk(fused tiles)", workspace, scratch);
    if (t.z > 1 && scratch >= (int64_t)t.z * p.M * p.N * 4) { p.partial = (float*)workspace; p.ksplit = t.z; }
    if (t.form == NkTiles::MID)
        return t.mt == 4 ? llmk::launch_mid<KIND, 4>(p, st, "gemm_w4a16_nk(mid)") : llmk::launch_mid<KIND, 2>(p, st, "gemm_w4a16_nk(mid)");
    return t.mt == 4 ? llmk::launch_mid<KIND, 4, false, true>(p, st, "gemm_w4a16_nk(mid, 128 columns)")
                     : llmk::launch_mid<KIND, 8, false, true>(p, st, "gemm_w4a16_nk(mid, 128 columns)");
}

// What the kernels next to the wave kernels (gemm_wave.hpp) take for 17 to 512 rows, in us like the estimates there.  Up to 64
// rows the ring kernel: its workgroups' tiles times the K steps of a wave, and the sums of its K ranges.  From there the tile
// kernels by their form: the mid-size ones with 64 and 128 columns, the 128-column tile in K slices, or rounds of the tiles that
// dma_tile_estimate chooses (at the rates of 4-bit weights).  A fit (3 to 10 % rms, 14 % for the K slices) to 350 shapes of M 17 to 520,
// N 1024 to 28672, K 1024 to 14336, as are the wave kernels' estimates; choosing by both was 1 to 2 % behind the faster one of
// each shape on average, and 1.16 (bf16 up to 64 rows) to 1.26 times faster than without the wave kernels.  Wave | other, us: bf16
// 48 x 4096 x 4096 10.8 | 12.3, 80 x 4096 x 4096 12.6 | 19.2, 160 x 4096 x 14336 44.6 | 75.0, 96 x 14336 x 4096 31.1 | 37.8, fp16
// 256 x 8192 x 8192 59.8 | 89.7, but 256 x 14336 x 4096 63.1 | 45.9 and bf16 24 x 4096 x 4096 9.6 | 9.2: every row tile unpacks the
// weights again, and short rows of few columns leave its waves too little to do.
template <int KIND>
double nk_other_estimate(const llmk::DirectArgs& p) {
    const int64_t M = p.M, N = p.N, K = p.K;
    const double k = (double)K / 4096.0;
    if (M <= 64) {
        const int64_t nz = (K / 128 + 31) / 32, rows = ((M + 15) / 16) * nz, tiles = (N + 15) / 16;
        const int64_t wg = std::max<int64_t>(1, LLMK_CUS / std::min<int64_t>(rows, LLMK_CUS)), per_wg = (tiles + wg - 1) / wg;
        const double u = (double)((((K / 128 + nz - 1) / nz) + 7) / 8);
        return 2.5 + 0.45 * u + (double)per_wg * (0.29 * u + 0.09) + (nz > 1 ? 2.9 : 0.0);
    }
    const NkTiles t = nk_tiles<KIND>(p);
    if (t.form == NkTiles::MID) return 4.3 + (t.mt == 2 ? 12.0 : 17.0) * k / t.z + (t.z > 1 ? 2.5 : 0.0);
    if (t.form == NkTiles::MIDW) return 4.4 + (t.mt == 4 ? 31.3 : 41.0) * k / t.z + (t.z > 1 ? 3.0 : 0.0);
    if (t.z > 1) return 7.5 + 54.0 * k / t.z;
    const llmk::TileChoice c = llmk::dma_tile_estimate<KIND, false>(p);
    const double e = c.cost * k;
    switch (c.choice) {
        case 1: return 2.0 + 2.3 * e;
        case 2: return 3.0 + 1.7 * e;
        case 4: return 7.0 + 1.4 * e;
        case 8: return 5.0 + 1.6 * e;
        default: return 3.0 + 1.7 * e;
    }
}
// What the weights of a call are, by its shape alone: (q - 8) * scale rounded to the activations' type, as in the tile kernels and in
// the 16-bit copy of W, or q - 8 exactly with the scale on fp32 sums, as in the streaming kernels.  The wave kernel has both and
// takes what those have that it stands in for: a row's result then does not hang on which kernel is faster, and a bf16 call
// that the ring kernel never took keeps its infinities (an infinite activation times -136, where the exact sums start, is a NaN).
bool nk_rounded_weights(int64_t M, int64_t N, int64_t K, int group, bool bf) {
    if (M > 64) return true;
    const int nz = (int)((K / 128 + 31) / 32);
    return bf ? !nk_ring_ok(M, N, K, group, nz) || (nz > 1 && (M * N) % 4) : w4_tiles_expand(M, N, K, INT64_MAX, true);
}
// The wave kernel for this call, or z = 0: taken 8 % below the others' estimate.
template <int KIND>
llmk::WavePlan nk_wave(const llmk::DirectArgs& p, int64_t scratch) {
    llmk::WavePlan w{0, 0, 0, 0, 0.0};
    const bool fits = nk_rounded_weights(p.M, p.N, p.K, p.group, KIND == llmk::K_W4NKB) ? llmk::w4a16_wave_plan<KIND, true>(p.M, p.N, p.K, p.group, scratch, w)
                                                                                       : llmk::w4a16_wave_plan<KIND, false>(p.M, p.N, p.K, p.group, scratch, w);
    if (!fits || 1.08 * w.cost >= nk_other_estimate<KIND>(p)) w.z = 0;
    return w;
}

// What a call beyond 512 rows gets without the kernel of two wave groups, in us: tiles that expand the words themselves (a fit of 2 to 6 % rms), or
// the 16-bit copy of W and the 16-bit tiles (9 %).
template <int KIND, int HALF_KIND>
double nk_large_estimate(const llmk::DirectArgs& p, bool copy) {
    const llmk::TileChoice c = copy ? llmk::dma_tile_estimate<HALF_KIND, false>(p) : llmk::dma_tile_estimate<KIND, false>(p);
    const double e = c.cost * (double)p.K / 4096.0, nk = (double)p.N * p.K * 1e-6;
    constexpr bool BF = KIND == llmk::K_W4NKB;
    // (few short tiles, where the passes are mostly their launches: 2 to 3 % rms to 176 shapes of up to 1024 columns.  With the estimate of the larger ones 58 of
    // them went to the kernel of two wave groups and were 3 to 14 % slower: fp16 1240 x 72 x 640 7.6 | 8.6, 2007 x 440 x 2048 16.2 | 18.7, bf16 1027 x 208 x 1024 9.7 | 10.9)
    if (copy && c.choice == 1) return 4.45 + 1.24 * e + 1.3 * std::min(nk, 4.0) + 0.5 * std::max(nk - 4.0, 0.0) + 0.54e-6 * (double)p.M * p.N;
    if (copy) return BF ? 6.3 + 1.37 * e + 0.44 * nk : 9.0 + 1.25 * e + 0.59 * nk;
    switch (c.choice) {
        case 1: return (BF ? 3.8 : 2.8) + (BF ? 2.08 : 2.19) * e;
        case 2: return 3.6 + (BF ? 1.59 : 1.55) * e;
        case 4: return 3.0 + (BF ? 1.38 : 1.45) * e;
        default: return 2.0 + (BF ? 1.55 : 1.58) * e;
    }
}

// The kernels of a call on the [N, K/8] layout, in the order in which they are preferred, and the scratch they use: what
// llmk_gemm_w4a16_nk runs with `scratch` bytes there, and what llmk_gemm_w4a16_nk_workspace_bytes reports for any amount.
struct NkPlan {
    enum { RING, TILES, COPY, RANGES, STREAM, NONE, WAVE, DUO } route;
    int nz;
    int64_t bytes;
    llmk::WavePlan wave;
    llmk::DuoPlan duo;
};
NkPlan nk_plan_others(int64_t M, int64_t N, int64_t K, int group, bool bf, int64_t scratch, bool c8) {
    const int nz = (int)((K / 128 + 31) / 32);               // K ranges of the streaming kernels
    const int64_t planes = nz > 1 ? (int64_t)nz * M * N * 4 : 0;
    const bool sums = nz == 1 || ((M * N) % 4 == 0 && scratch >= planes);
    llmk::DirectArgs p{};
    p.M = (int)M; p.N = (int)N; p.K = (int)K; p.E = 1; p.group = group;
    llmk::WavePlan w{};
    if (M > 16 && M <= 512) w = bf ? nk_wave<llmk::K_W4NKB>(p, scratch) : nk_wave<llmk::K_W4NK>(p, scratch);
    if (w.z > 0) return {NkPlan::WAVE, 1, w.z > 1 ? w.z * M * N * 4 : 0, w};
    if (bf && M <= 64 && c8 && sums && nk_ring_ok(M, N, K, group, nz)) return {NkPlan::RING, nz, planes, {}};
    if (llmk::dma_eligible(p, 2)) {
        if (w4_tiles_expand(M, N, K, scratch, true, bf) && group % 64 == 0) {
            int z = bf ? nk_tiles<llmk::K_W4NKB>(p).z : nk_tiles<llmk::K_W4NK>(p).z;
            if (M <= 64) z = max(z, llmk::splitk_factor_half(M, N, K));      // (w4_tiles_expand asks for these there)
            return {NkPlan::TILES, 1, z > 1 ? (int64_t)z * M * N * 4 : 0, {}};
        }
        // the 16-bit copy of W, and behind it whatever the 16-bit GEMM's K slices take
        if ((M > 64 || bf) && scratch >= N * K * 2) return {NkPlan::COPY, 1, ((N * K * 2 + 255) & ~(int64_t)255) + (M <= 512 ? 8 * M * N * 4 : 0), {}};
    }
    if (bf) return {NkPlan::NONE, 1, 0, {}};
    // K > 4096: ranges of at most 4096 (each with resident activations) and fp32 partial sums
    if (group % 128 == 0 && M <= 64 && nz > 1 && sums && c8 && ((K / 128 + nz - 1) / nz * 128) % group == 0) return {NkPlan::RANGES, nz, planes, {}};
    return {NkPlan::STREAM, 1, 0, {}};
}

// The same with the kernel of two wave groups (gemm_duo.hpp) from 65 to 2048 rows, 8 % below the estimate of the route above.  Over 300 random shapes of
// 64 to 4096 rows fp16 calls were 1.08 and bf16 calls 1.11 times as fast as without, 1 % behind the faster one of each shape.  (The line at 2048
// rows is no border of the kernel's: 190 of 500 random shapes from 2049 to 4096 would go here, and the 500 be 1.06, fp16, and 1.07 times as fast.)  Others | this
// one, us: bf16 300 x 14336 x 4096 54 | 45.5, 1024 x 4096 x 4096 48 | 40.7.
template <int KIND, int HALF_KIND>
NkPlan nk_plan_of(int64_t M, int64_t N, int64_t K, int group, int64_t scratch, bool c8) {
    constexpr bool BF = KIND == llmk::K_W4NKB;
    const NkPlan pl = nk_plan_others(M, N, K, group, BF, scratch, c8);
    if (M <= 64 || M > 2048) return pl;
    llmk::DirectArgs p{};
    p.M = (int)M; p.N = (int)N; p.K = (int)K; p.E = 1; p.group = group;
    const llmk::DuoPlan d = llmk::duo_plan<KIND>(p, scratch);
    if (!d.mi) return pl;
    double other = 1e30, margin = llmk::DU_MARGIN;           // (streaming kernels this far out: no scratch for a copy)
    const bool copy = pl.route == NkPlan::COPY, tiles = pl.route == NkPlan::TILES;
    if (pl.route == NkPlan::WAVE) other = 1.05 * pl.wave.cost;
    else if (tiles && M <= 512) other = nk_other_estimate<KIND>(p);
    else if (tiles || copy) other = nk_large_estimate<KIND, HALF_KIND>(p, copy);
    if ((tiles || copy) && llmk::duo_beyond_a_round(p, d)) {
        // (fp16 tiles that expand the words themselves: all of them; bf16 256 x 256 ones not, 25 shapes are 1.07 times as fast here)
        const int choice = copy ? llmk::dma_tile_estimate<HALF_KIND, false>(p).choice : llmk::dma_tile_estimate<KIND, false>(p).choice;
        if (copy ? choice == 8 : (!BF || choice == 4)) margin = llmk::DU_MARGIN_TALL;
    }
    if (margin * d.cost >= other) return pl;
    return {NkPlan::DUO, 1, d.z > 1 ? (int64_t)d.z * M * N * 4 : 0, {}, d};
}
NkPlan nk_plan(int64_t M, int64_t N, int64_t K, int group, bool bf, int64_t scratch, bool c8) {
    return bf ? nk_plan_of<llmk::K_W4NKB, llmk::K_BF16>(M, N, K, group, scratch, c8) : nk_plan_of<llmk::K_W4NK, llmk::K_F16>(M, N, K, group, scratch, c8);
}

// launch shape of the Marlin-layout kernel for a given problem
struct MarlinPlan {
    int mt, nw, mblocks, col_groups, z, steps_per_z;
};

MarlinPlan marlin_plan(int64_t M, int64_t N, int64_t K) {
    MarlinPlan pl{};
    pl.mt = 1;                                              // 16-row workgroups side by side (measured faster than taller ones)
    pl.nw = 8;                                              // nw * mt * 8 KiB of reduction LDS <= 64 KiB
    pl.mblocks = (int)cdiv64(M, 16 * pl.mt);
    pl.col_groups = (int)((N / 64 + 1) / 2);
    const int total_steps = (int)((K / 16 + 1) / 2);
    // split K over workgroups until the grid covers the chip; every slice keeps >= nw steps
    int z = 1;
    if (M <= 64)
        while ((int64_t)pl.col_groups * pl.mblocks * z < 256 && total_steps / (z * 2) >= pl.nw) z *= 2;
    pl.z = z;
    pl.steps_per_z = (total_steps + z - 1) / z;
    return pl;
}

// What the 128-column tile kernels that expand Marlin words take for 65 to 512 rows, in us (see below).
double marlin_tiles_estimate(int64_t M, int64_t N, int64_t K, int group) {
    llmk::DirectArgs p{};
    p.M = (int)M; p.N = (int)N; p.K = (int)K; p.E = 1; p.group = group;
    const double k = (double)K / 4096.0;
    const int64_t tiles = ((M + 63) / 64) * ((N + 127) / 128), z = std::min<int64_t>(llmk::splitk_factor_half(M, N, K), std::max<int64_t>(1, LLMK_CUS / tiles));
    if (z > 1) return 7.7 + 42.5 * k / z;
    const llmk::TileChoice c = llmk::dma_tile_estimate<llmk::K_W4MARLIN, false>(p);
    return c.choice == 1 ? 4.0 + 2.5 * c.cost * k : (c.choice == 2 ? 5.3 + 1.75 * c.cost * k : 5.0 + 1.58 * c.cost * k);
}
// The wave kernel for a call on Marlin words, or z = 0: always up to 64 rows, up to 512 where it is estimated 8 % below the
// 128-column tile kernels that expand the words in LDS (a fit of 3 to 7 % rms to 70 shapes: the scatter of the Marlin layout is most
// of their time).  Choosing so was 1 % behind the faster one of each shape and 1.47 times faster than without the wave kernel over
// 180 shapes of 16 to 528 rows.  Wave | other, us, cold weights: 16 x 4096 x 4096 9.9 | 10.6, 16 x 14336 x 4096 14.4 | 18.5, 32 x 28672
// x 4096 25.6 | 47.2, 64 x 14336 x 4096 20.1 | 47.0, 96 x 4096 x 14336 26.9 | 52.2, 256 x 4096 x 4096 19.0 | 35.9, 192 x 14336 x 4096
// 47.1 | 60.2, but 384 x 14336 x 4096 87.8 | 80.0.
llmk::WavePlan marlin_wave(int64_t M, int64_t N, int64_t K, int group, int64_t scratch) {
    llmk::WavePlan w{0, 0, 0, 0, 0.0};
    if (M > 512 || !llmk::w4a16_wave_plan<llmk::K_W4MARLIN, true>(M, N, K, group, scratch, w)) { w.z = 0; return w; }
    if (M > 64 && 1.08 * w.cost >= marlin_tiles_estimate(M, N, K, group)) w.z = 0;
    return w;
}
// The kernel of two wave groups (gemm_duo.hpp) for a call on Marlin words, or mi = 0: from 65 rows on, 8 % below the estimate of the wave kernel, the
// tiles above, or beyond 512 rows the 16-bit copy of W and the fp16 tiles (a fit of 10 % rms to 146 shapes).  Its threads scatter the words
// without bank conflicts.  Over 300 random shapes of 64 to 4096 rows 1.06 times as fast as without, 0.5 % behind the faster one of each
// shape; of 1070 more 3 were 5 to 8 % slower.  Others | this one, us: 1024 x 4096 x 4096 52.7 | 43.7, 432 x 6144 x 4096 42.0 | 36.6, 1072 x 3200 x 6400 76 | 61,
// 832 x 2560 x 2560 31.5 | 25.1, but 2384 x 6144 x 4096 106 | 134 and 416 x 1600 x 1664 9.0 | 16.7.
llmk::DuoPlan marlin_duo(int64_t M, int64_t N, int64_t K, int group, const llmk::WavePlan& wave, int64_t scratch) {
    if (M <= 64 || K % 64) return {0, 1, 0.0};
    llmk::DirectArgs p{};
    p.M = (int)M; p.N = (int)N; p.K = (int)K; p.E = 1; p.group = group;
    llmk::DuoPlan d = llmk::duo_plan<llmk::K_W4MARLIN>(p, scratch);
    if (!d.mi) return d;
    double other = wave.z > 0 ? 1.05 * wave.cost : marlin_tiles_estimate(M, N, K, group), margin = llmk::DU_MARGIN;
    const llmk::TileChoice c = M > 512 ? llmk::dma_tile_estimate<llmk::K_F16, false>(p) : llmk::dma_tile_estimate<llmk::K_W4MARLIN, false>(p);
    if (M > 512) other = 6.1 + 0.40e-6 * (double)N * K + 1.38 * c.cost * (double)K / 4096.0;
    if ((M > 512 || wave.z <= 0) && c.choice == (M > 512 ? 8 : 4) && llmk::duo_beyond_a_round(p, d)) margin = llmk::DU_MARGIN_TALL;
    if (margin * d.cost >= other) d.mi = 0;
    return d;
}

}  // namespace

extern "C" int64_t llmk_gemm_w4a16_marlin_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    if (M <= 0 || N <= 0 || K <= 0 || M > 0x7fffffff / 2 || N > 0x7fffffff / 2 || K > 0x7fffffff / 2) return 0;
    // the group size is not known here: what the wave kernel's slices take with groups of 128, and what the others take
    const llmk::WavePlan wave = marlin_wave(M, N, K, 128, INT64_MAX);
    const llmk::DuoPlan duo = marlin_duo(M, N, K, 128, wave, INT64_MAX);
    const int64_t slices = std::max(wave.z > 1 ? wave.z * M * N * 4 : 0, duo.mi && duo.z > 1 ? duo.z * M * N * 4 : 0);
    if (M > 64) {                                        // dequantised fp16 copy of W for the tiled GEMM (+ split-K partials)
        if (K % 64) return 0;
        const int z = llmk::splitk_factor_half(M, N, K);
        return std::max(slices, ((N * K * 2 + 255) & ~(int64_t)255) + (z > 1 ? (int64_t)z * M * N * 4 : 0));
    }
    const MarlinPlan pl = marlin_plan(M, N, K);
    const int64_t zt = M > 16 && K % 64 == 0 ? llmk::splitk_factor_half(M, N, K) : 1;   // tile kernels with split-K
    const int64_t z = pl.z > zt ? pl.z : zt;
    return std::max(slices, z > 1 ? z * M * N * 4 : 0);
}

extern "C" int llmk_gemm_w4a16_wave_shape(int marlin, int ac_dtype, int64_t M, int64_t N, int64_t K, int groupsize, int64_t scratch_bytes,
                                          int32_t* shape) {
    if (!shape || M <= 0 || N <= 0 || K <= 0 || K % 128 || M > 0x7fffffff / 2 || N > 0x7fffffff / 2 || K > 0x7fffffff / 2) return 0;
    if (groupsize == -1) groupsize = (int)K;
    if (groupsize < 8 || K % groupsize) return 0;
    if (marlin) {
        const llmk::WavePlan w = marlin_wave(M, N, K, groupsize, scratch_bytes);
        return w.z > 0 && !marlin_duo(M, N, K, groupsize, w, scratch_bytes).mi ? llmk::wave_shape(w, 1, shape) : 0;
    }
    const bool bf = ac_dtype == LLMK_BF16;
    const NkPlan pl = nk_plan(M, N, K, groupsize, bf, scratch_bytes, true);
    return pl.route == NkPlan::WAVE ? llmk::wave_shape(pl.wave, nk_rounded_weights(M, N, K, groupsize, bf), shape) : 0;
}

extern "C" int llmk_gemm_w4a16_duo_shape(int marlin, int ac_dtype, int64_t M, int64_t N, int64_t K, int groupsize, int64_t scratch_bytes, int32_t* shape) {
    if (!shape || M <= 0 || N <= 0 || K <= 0 || K % 64 || M > 0x7fffffff / 2 || N > 0x7fffffff / 2 || K > 0x7fffffff / 2) return 0;
    if (groupsize == -1) groupsize = (int)K;
    if (groupsize < 8 || groupsize % 8 || K % groupsize || (!marlin && K % 128)) return 0;
    llmk::DuoPlan d{0, 1, 0.0};
    if (marlin) {
        d = marlin_duo(M, N, K, groupsize, marlin_wave(M, N, K, groupsize, scratch_bytes), scratch_bytes);
    } else {
        const NkPlan pl = nk_plan(M, N, K, groupsize, ac_dtype == LLMK_BF16, scratch_bytes, true);
        if (pl.route == NkPlan::DUO) d = pl.duo;
    }
    if (!d.mi) return 0;
    shape[0] = 32 * d.mi;
    shape[1] = d.z;
    return 1;
}

extern "C" int llmk_gemm_w4a16_marlin(const void* a, const int32_t* b, void* c, const void* s, int64_t M, int64_t N,
                                      int64_t K, int groupsize, void* workspace, int64_t workspace_bytes,
                                      void* stream) {
    // the reference launcher returns -1 for any dimension not divisible by 16 (marlin_w4a16_gemm.cu:300-302)
    if (M % 16 || N % 16 || K % 16 || M < 0 || N < 0 || K < 0)
        LLMK_FAIL(LLMK_ERR_SHAPE, "gemm_w4a16_marlin: M, N, K must be multiples of 16 (M=%lld N=%lld K=%lld)", (long long)M, (long long)N, (long long)K);
    if (N % 64) LLMK_FAIL(LLMK_ERR_SHAPE, "gemm_w4a16_marlin: N=%lld must be a multiple of 64 (packed chunk width)", (long long)N);
    if (M == 0 || N == 0) return LLMK_OK;
    if (K == 0) LLMK_FAIL(LLMK_ERR_SHAPE, "gemm_w4a16_marlin: K == 0");
    if (groupsize == -1) groupsize = (int)K;
    if (groupsize < 16 || groupsize % 16 || K % groupsize)
        LLMK_FAIL(LLMK_ERR_SHAPE, "gemm_w4a16_marlin: groupsize=%d must be a multiple of 16 dividing K=%lld", groupsize, (long long)K);
    if (!a || !b || !c || !s) LLMK_FAIL(LLMK_ERR_ARG, "gemm_w4a16_marlin: null pointer");
    if (((uintptr_t)a | (uintptr_t)b | (uintptr_t)s) & 15) LLMK_FAIL(LLMK_ERR_ARG, "gemm_w4a16_marlin: operands must be 16-byte aligned");
    if (M > 0x7fffffff / 2 || N > 0x7fffffff / 2 || K > 0x7fffffff / 2) LLMK_FAIL(LLMK_ERR_SHAPE, "gemm_w4a16_marlin: dimension too large");

    hipStream_t st = (hipStream_t)stream;
    const llmk::WavePlan wave = marlin_wave(M, N, K, groupsize, usable_scratch(workspace, workspace_bytes));
    const llmk::DuoPlan duo = marlin_duo(M, N, K, groupsize, wave, usable_scratch(workspace, workspace_bytes));
    if (duo.mi) {
        llmk::DirectArgs p{};
        p.a = (const uint8_t*)a; p.b = (const uint8_t*)b; p.b_s = s; p.c = c; p.c_dtype = LLMK_F16;
        p.M = (int)M; p.N = (int)N; p.K = (int)K; p.E = 1; p.group = groupsize;
        return llmk::launch_duo_plan<llmk::K_W4MARLIN>(p, duo, workspace, st, "gemm_w4a16_marlin(duo)");
    }
    if (wave.z > 0) {
        llmk::DirectArgs p{};
        p.a = (const uint8_t*)a; p.b = (const uint8_t*)b; p.b_s = s; p.c = c; p.c_dtype = LLMK_F16;
        p.M = (int)M; p.N = (int)N; p.K = (int)K; p.E = 1; p.group = groupsize; p.partial = (float*)workspace;
        return llmk::launch_w4a16_wave_plan<llmk::K_W4MARLIN, true>(p, wave, st, "gemm_w4a16_marlin(wave)");
    }
    if (w4_tiles_expand(M, N, K, usable_scratch(workspace, workspace_bytes)) && K % 64 == 0 && groupsize % 64 == 0) {
        // mid-size M: the 128-column tile kernels expand the Marlin units themselves (see gemm_w4a16_nk)
        llmk::DirectArgs p{};
        p.a = (const uint8_t*)a; p.b = (const uint8_t*)b; p.b_s = s; p.c = c; p.c_dtype = LLMK_F16;
        p.M = (int)M; p.N = (int)N; p.K = (int)K; p.E = 1; p.group = groupsize;
        if (llmk::dma_eligible(p, 2))
            return llmk::launch_big_half<llmk::K_W4MARLIN, false>(p, st, "gemm_w4a16_marlin(fused tiles)", workspace, workspace_bytes);
    }
    if (M > 64 && K % 64 == 0 && workspace && workspace_bytes >= N * K * 2 && !((uintptr_t)workspace & 15)) {
        // compute-bound: expand W once to fp16 [N, K], then run the tiled MFMA GEMM on it
        llmk::DirectArgs p{};
        p.a = (const uint8_t*)a; p.b = (const uint8_t*)workspace; p.c = c; p.c_dtype = LLMK_F16;
        p.M = (int)M; p.N = (int)N; p.K = (int)K; p.E = 1;
        if (llmk::dma_eligible(p, 2)) {
            dim3 dgrid((unsigned)(N / 64), (unsigned)cdiv64(K, 128));
            marlin_dequant_kernel<<<dgrid, 256, 0, st>>>((const v4i*)b, (const _Float16*)s, (_Float16*)workspace, (int)N, (int)K, groupsize);
            LLMK_CHECK_LAUNCH("gemm_w4a16_marlin(dequant)");
            const int64_t used = (N * K * 2 + 255) & ~(int64_t)255;
            return llmk::launch_big_half<llmk::K_F16, false>(p, st, "gemm_w4a16_marlin(tiled)", (uint8_t*)workspace + used,
                                                             workspace_bytes > used ? workspace_bytes - used : 0);
        }
    }
    MarlinPlan pl = marlin_plan(M, N, K);
    if (pl.z > 1 && (!workspace || workspace_bytes < (int64_t)pl.z * M * N * 4 || (((uintptr_t)workspace) & 15) || (((uintptr_t)c) & 7))) {
        pl.z = 1;                                   // no scratch: every workgroup walks all of K
        pl.steps_per_z = (int)((K / 16 + 1) / 2);
    }
    const _Float16* A = (const _Float16*)a;
    const v4i* B = (const v4i*)b;
    const _Float16* S = (const _Float16*)s;
    _Float16* C = (_Float16*)c;
    float* ws = (float*)workspace;
    dim3 grid(pl.col_groups, pl.mblocks, pl.z), blk(pl.nw * 64);
    const size_t red_bytes = (size_t)pl.nw * pl.mt * 32 * 64 * sizeof(float);
    const size_t a_bytes = (size_t)16 * pl.mt * ((size_t)pl.steps_per_z * 64 + 16);     // activation image of one K range
    // staged while every workgroup fits on the chip at once; with several rounds of workgroups the unoverlapped
    // staging of each costs more than the global fragment loads (measured at N = 128256: 88 vs 84 us)
    const bool a_lds = a_bytes <= 144 * 1024 && (int64_t)pl.col_groups * pl.mblocks * pl.z <= 512;
    const size_t smem = a_lds && a_bytes > red_bytes ? a_bytes : red_bytes;
    if (smem > 64 * 1024) {
        static std::atomic<uint64_t> cfg_a{0}, cfg_b{0};
        if (int rc = llmk_reserve_lds((const void*)w4a16_marlin_kernel<1, 8, true, true>, 160 * 1024, cfg_a, "gemm_w4a16_marlin")) return rc;
        if (int rc = llmk_reserve_lds((const void*)w4a16_marlin_kernel<1, 8, false, true>, 160 * 1024, cfg_b, "gemm_w4a16_marlin")) return rc;
    }
#define LLMK_MARLIN_LAUNCH(MT, NW)                                                                              \
    do {                                                                                                        \
        if (pl.z > 1 && a_lds) w4a16_marlin_kernel<MT, NW, true, true><<<grid, blk, smem, st>>>(A, B, S, C, ws, (int)M, (int)N, (int)K, groupsize, pl.steps_per_z); \
        else if (pl.z > 1) w4a16_marlin_kernel<MT, NW, true><<<grid, blk, smem, st>>>(A, B, S, C, ws, (int)M, (int)N, (int)K, groupsize, pl.steps_per_z); \
        else if (a_lds) w4a16_marlin_kernel<MT, NW, false, true><<<grid, blk, smem, st>>>(A, B, S, C, nullptr, (int)M, (int)N, (int)K, groupsize, pl.steps_per_z); \
        else w4a16_marlin_kernel<MT, NW, false><<<grid, blk, smem, st>>>(A, B, S, C, nullptr, (int)M, (int)N, (int)K, groupsize, pl.steps_per_z); \
    } while (0)
    LLMK_MARLIN_LAUNCH(1, 8);
#undef LLMK_MARLIN_LAUNCH
    LLMK_CHECK_LAUNCH("gemm_w4a16_marlin");
    if (pl.z > 1) {
        splitk_reduce_f16_kernel<<<(unsigned)cdiv64(M * N, 4 * 256), 256, 0, st>>>((const float*)workspace, C, M * N, pl.z);
        LLMK_CHECK_LAUNCH("gemm_w4a16_marlin(reduce)");
    }
    return LLMK_OK;
}

extern "C" int64_t llmk_gemm_w4a16_nk_workspace_bytes(int64_t M, int64_t N, int64_t K, int groupsize, int ac_dtype) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 128 || M > 0x7fffffff / 2 || N > 0x7fffffff / 2 || K > 0x7fffffff / 2) return 0;
    if (groupsize == -1) groupsize = (int)K;
    if (groupsize < 8) return 0;
    return nk_plan(M, N, K, groupsize, ac_dtype == LLMK_BF16, INT64_MAX, true).bytes;
}

extern "C" int llmk_gemm_w4a16_nk(const void* a, const int32_t* b_packed, void* c, const void* s, int ac_dtype,
                                  int64_t M, int64_t N, int64_t K, int groupsize, void* workspace,
                                  int64_t workspace_bytes, void* stream) {
    if (ac_dtype != LLMK_F16 && ac_dtype != LLMK_BF16) LLMK_FAIL(LLMK_ERR_DTYPE, "gemm_w4a16_nk: activations / outputs must be fp16 or bf16 (dtype code %d)", ac_dtype);
    const bool bf = ac_dtype == LLMK_BF16;
    if (M < 0 || N < 0 || K < 0 || K % 128) LLMK_FAIL(LLMK_ERR_SHAPE, "gemm_w4a16_nk: K=%lld must be a multiple of 128", (long long)K);
    if (M == 0 || N == 0) return LLMK_OK;
    if (K == 0) LLMK_FAIL(LLMK_ERR_SHAPE, "gemm_w4a16_nk: K == 0");
    if (groupsize == -1) groupsize = (int)K;
    if (groupsize < 8 || groupsize % 8 || K % groupsize)
        LLMK_FAIL(LLMK_ERR_SHAPE, "gemm_w4a16_nk: groupsize=%d must be a multiple of 8 dividing K", groupsize);
    if (!a || !b_packed || !c || !s) LLMK_FAIL(LLMK_ERR_ARG, "gemm_w4a16_nk: null pointer");
    if (((uintptr_t)a | (uintptr_t)b_packed) & 15) LLMK_FAIL(LLMK_ERR_ARG, "gemm_w4a16_nk: operands must be 16-byte aligned");
    if (M > 0x7fffffff / 2 || N > 0x7fffffff / 2 || K > 0x7fffffff / 2) LLMK_FAIL(LLMK_ERR_SHAPE, "gemm_w4a16_nk: dimension too large");
    hipStream_t st = (hipStream_t)stream;
    const _Float16* A = (const _Float16*)a;
    const _Float16* S = (const _Float16*)s;
    _Float16* C = (_Float16*)c;
    const int64_t scratch = usable_scratch(workspace, workspace_bytes);
    const NkPlan pl = nk_plan(M, N, K, groupsize, bf, scratch, !((uintptr_t)c & 7));
    llmk::DirectArgs p{};
    p.a = (const uint8_t*)a; p.c = c; p.c_dtype = ac_dtype;
    p.M = (int)M; p.N = (int)N; p.K = (int)K; p.E = 1;
    switch (pl.route) {
        case NkPlan::WAVE:
            p.b = (const uint8_t*)b_packed; p.b_s = s; p.group = groupsize; p.partial = (float*)workspace;
            if (nk_rounded_weights(M, N, K, groupsize, bf))
                return bf ? llmk::launch_w4a16_wave_plan<llmk::K_W4NKB, true>(p, pl.wave, st, "gemm_w4a16_nk(wave)")
                          : llmk::launch_w4a16_wave_plan<llmk::K_W4NK, true>(p, pl.wave, st, "gemm_w4a16_nk(wave)");
            return bf ? llmk::launch_w4a16_wave_plan<llmk::K_W4NKB, false>(p, pl.wave, st, "gemm_w4a16_nk(wave)")
                      : llmk::launch_w4a16_wave_plan<llmk::K_W4NK, false>(p, pl.wave, st, "gemm_w4a16_nk(wave)");
        case NkPlan::DUO:
            p.b = (const uint8_t*)b_packed; p.b_s = s; p.group = groupsize;
            return bf ? llmk::launch_duo_plan<llmk::K_W4NKB>(p, pl.duo, workspace, st, "gemm_w4a16_nk(duo)")
                      : llmk::launch_duo_plan<llmk::K_W4NK>(p, pl.duo, workspace, st, "gemm_w4a16_nk(duo)");
        case NkPlan::RING:                               // bf16 decode; fp16 reaches that kernel through launch_nk_stream
            return launch_nk_ring(a, b_packed, S, c, (int)M, (int)N, (int)K, pl.nz, (float*)workspace, true, st);
        case NkPlan::TILES:
            p.b = (const uint8_t*)b_packed; p.b_s = s; p.group = groupsize;
            return bf ? launch_nk_tiles<llmk::K_W4NKB>(p, workspace, scratch, st) : launch_nk_tiles<llmk::K_W4NK>(p, workspace, scratch, st);
        case NkPlan::COPY: {
            // compute-bound: expand W once to fp16 / bf16 [N, K], then run the tiled MFMA GEMM on it
            p.b = (const uint8_t*)workspace;
            const unsigned blocks = (unsigned)cdiv64(N * (K / 8), 256);
            if (bf) nk_dequant_bf16_kernel<<<blocks, 256, 0, st>>>(b_packed, S, (unsigned short*)workspace, N, K, groupsize);
            else nk_dequant_kernel<<<blocks, 256, 0, st>>>(b_packed, S, (_Float16*)workspace, N, K, groupsize);
            LLMK_CHECK_LAUNCH("gemm_w4a16_nk(dequant)");
            const int64_t used = (N * K * 2 + 255) & ~(int64_t)255;
            void* rest = (uint8_t*)workspace + used;
            const int64_t rest_bytes = scratch > used ? scratch - used : 0;
            if (bf) return llmk::launch_big_half<llmk::K_BF16, false>(p, st, "gemm_w4a16_nk(tiled, bf16)", rest, rest_bytes);
            return llmk::launch_big_half<llmk::K_F16, false>(p, st, "gemm_w4a16_nk(tiled)", rest, rest_bytes);
        }
        case NkPlan::NONE:
            LLMK_FAIL(LLMK_ERR_ARG, "gemm_w4a16_nk: this bf16 call needs a 16-byte aligned workspace of N*K*2 = %lld bytes (bf16 copy of W)",
                      (long long)(N * K * 2));
        case NkPlan::RANGES:
            return launch_nk_stream<1, 1>(A, b_packed, S, C, (int)M, (int)N, (int)K, groupsize, pl.nz, (float*)workspace, st);
        case NkPlan::STREAM: break;
    }
    if (groupsize % 128 == 0 && M <= 64) {
        // one 16-column block per tile: two blocks per tile (NT = 2) measured slower at every shape tried.
        // While the activations of a 16-row workgroup stay resident (K <= 4096), such workgroups side by side
        // beat taller ones by up to 2x.
        if (M <= 16 || K <= 4096) return launch_nk_stream<1, 1>(A, b_packed, S, C, (int)M, (int)N, (int)K, groupsize, 1, nullptr, st);
        if (M <= 32) return launch_nk_stream<2, 1>(A, b_packed, S, C, (int)M, (int)N, (int)K, groupsize, 1, nullptr, st);
        return launch_nk_stream<4, 1>(A, b_packed, S, C, (int)M, (int)N, (int)K, groupsize, 1, nullptr, st);
    }
    const unsigned gx = (unsigned)cdiv64(N, 16);
    if (M <= 16) {
        constexpr int NW = 8;
        w4a16_nk_kernel<1, NW><<<dim3(gx, 1), NW * 64, (NW / 2) * 4 * 64 * sizeof(float), st>>>(A, b_packed, S, C, (int)M, (int)N, (int)K, groupsize);
    } else {
        constexpr int MT = 4, NW = 4;
        w4a16_nk_kernel<MT, NW><<<dim3(gx, (unsigned)cdiv64(M, 16 * MT)), NW * 64, (NW / 2) * MT * 4 * 64 * sizeof(float), st>>>(A, b_packed, S, C, (int)M, (int)N, (int)K, groupsize);
    }
    LLMK_CHECK_LAUNCH("gemm_w4a16_nk");
    return LLMK_OK;
}

// Helpers shared by the quantizer kernels: 8-element loads, the reference's rounding rules, e4m3 packing
// and group reductions over lanes.
#pragma once
#include "common.hpp"

namespace {

constexpr int EPL = 8;   // elements per lane in the 1 x block kernels

template <int DT>
__device__ __forceinline__ void load8(const void* p, int64_t i, float (&v)[EPL]) {
    if constexpr (DT == LLMK_F32) {
        const float4* q = (const float4*)((const float*)p + i);
        float4 a = q[0], b = q[1];
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    } else {
        uint4 u = *(const uint4*)((const unsigned short*)p + i);
        unsigned w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            unsigned short lo = (unsigned short)(w[j] & 0xffff), hi = (unsigned short)(w[j] >> 16);
            v[2 * j]     = (DT == LLMK_F16) ? f16_to_f32(lo) : bf16_to_f32(lo);
            v[2 * j + 1] = (DT == LLMK_F16) ? f16_to_f32(hi) : bf16_to_f32(hi);
        }
    }
}

// 8 consecutive elements in the storage type DT (16-byte aligned for the 16-bit types, 32-byte for fp32)
template <int DT>
__device__ __forceinline__ void store8(void* p, int64_t i, const float (&v)[EPL]) {
    if constexpr (DT == LLMK_F32) {
        float4* q = (float4*)((float*)p + i);
        q[0] = make_float4(v[0], v[1], v[2], v[3]);
        q[1] = make_float4(v[4], v[5], v[6], v[7]);
    } else {
        unsigned w[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            w[j] = DT == LLMK_F16 ? ((unsigned)f32_to_f16(v[2 * j]) | ((unsigned)f32_to_f16(v[2 * j + 1]) << 16))
                                  : ((unsigned)f32_to_bf16(v[2 * j]) | ((unsigned)f32_to_bf16(v[2 * j + 1]) << 16));
        *(uint4*)((unsigned short*)p + i) = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

__device__ __forceinline__ float round_mode(float v, int mode) {
    // half-away: roundf is exact; half-up: floor(v + 0.5f) with the fp32 add as the reference states it
    return mode == LLMK_ROUND_HALF_AWAY ? roundf(v) : floorf(v + 0.5f);
}

__device__ __forceinline__ unsigned pack_fp8x4(float a, float b, float c, float d) {
    // saturate finite values to +-448 (comparisons leave NaN untouched), then RNE hardware convert
    auto sat = [](float x) { return x > 448.f ? 448.f : (x < -448.f ? -448.f : x); };
    int w = __builtin_amdgcn_cvt_pk_fp8_f32(sat(a), sat(b), 0, false);
    w = __builtin_amdgcn_cvt_pk_fp8_f32(sat(c), sat(d), w, true);
    return (unsigned)w;
}

// the value of the lane that reduction step O of a group of lanes exchanges with: groups of up to 16 lanes are a DPP row,
// where the exchange is an operand modifier of the reducing instruction; a shuffle through LDS costs an address, a trip of
// about 60 cycles and a wait.  (Steps 4 and 8 mirror half a row and a row: the lanes of a group of 4, or 8, hold the same
// value by then.)
template <int O>
__device__ __forceinline__ int lane_step(int v) {
    if constexpr (O <= 8) {
        constexpr int CTRL = O == 1 ? 0xB1 : (O == 2 ? 0x4E : (O == 4 ? 0x141 : 0x140));
        return __builtin_amdgcn_mov_dpp(v, CTRL, 0xf, 0xf, true);
    } else {
        return __shfl_xor(v, O, 64);
    }
}
template <int LPG, int O = 1>
__device__ __forceinline__ int group_imax(int v) {
    if constexpr (O < LPG) return group_imax<LPG, 2 * O>(max(v, lane_step<O>(v)));
    else return v;
}
template <int LPG, int O = 1>
__device__ __forceinline__ int group_imin(int v) {
    if constexpr (O < LPG) return group_imin<LPG, 2 * O>(min(v, lane_step<O>(v)));
    else return v;
}
// maximum of non-negative values (and no NaN: what fmaxf made of absolute values) over the LPG lanes that share a group
// (LPG power of two <= 64).  Their bits order as integers, whose maximum needs no quieting of its operands.
template <int LPG>
__device__ __forceinline__ float group_max(float v) { return __int_as_float(group_imax<LPG>(__float_as_int(v))); }
// the same over the four lanes l, l + 16, l + 32, l + 48: rows of 16 lanes change places between two registers, without a trip through LDS
__device__ __forceinline__ float max_of_rows(float v) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    const int m = max((int)a[0], (int)a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap((unsigned)m, (unsigned)m, false, false);
    return __int_as_float(max((int)b[0], (int)b[1]));
}


// a / b from r = RN(1 / b): one product and the residual correction q - (q b - a) r, both in fma.  The
// residual is exact whenever q is within an ulp of the quotient, and the corrected value is then the rounded
// quotient (the final step of the usual fma division); in 80 M random trials over the quantisers' operand
// ranges it equalled the IEEE division every time.  Nothing may leave the normal range: callers check b
// and take the division otherwise.  A quantiser divides the 8 values of a lane by one scale, so the
// reciprocal is shared and a quotient costs three instructions instead of about ten.
// The residual is formed as its negative, q b - a, and subtracted: with a = -0 the sum q b - a is +0 and
// q - (+0) r keeps the -0 of the quotient, where q + (a - q b) r would return +0 (an e4m3 result keeps the sign
// of a zero: 0x80).
__device__ __forceinline__ float div_by(float a, float b, float r) {
    const float q = a * r;
    const float nrem = fmaf(q, b, -a);
    return fmaf(-nrem, r, q);
}
// scales whose reciprocal, products and residuals stay normal for every |a| <= 448 b that does not round to
// zero in the 8-bit result anyway
__device__ __forceinline__ bool div_by_ok(float b) { return b > 1e-30f && b < 1e30f; }

// The scale of a group whose absmax is m, and what dividing by it takes.
template <bool FP8>
struct QuantScale {
    float sc, r;
    bool fast;
    __device__ __forceinline__ explicit QuantScale(float m) {
        sc = m / (FP8 ? 448.f : 127.f);
        fast = div_by_ok(sc);
        r = fast ? 1.0f / sc : 0.f;
    }
};

// 8 values of such a group as 8 bytes: exactly the arithmetic of the 1 x 128 activation quantizers.
// BOUNDED: no value exceeds m (the quantizers of memory can meet signalling NaN, which hide others from the maximum).  With a scale in the fast range the
// quotients are then at most 448 (1 + 2^-23), which converts to 448 without a clamp.
template <bool FP8, bool BOUNDED = false>
__device__ __forceinline__ uint2 quant8_by(const float (&v)[EPL], const QuantScale<FP8>& s, int mode) {
    float q[EPL];
    if (s.fast) {
#pragma unroll
        for (int j = 0; j < EPL; ++j) q[j] = div_by(v[j], s.sc, s.r);
        if constexpr (FP8 && BOUNDED) {
            unsigned w[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) w[h] = (unsigned)__builtin_amdgcn_cvt_pk_fp8_f32(q[4 * h + 2], q[4 * h + 3], __builtin_amdgcn_cvt_pk_fp8_f32(q[4 * h], q[4 * h + 1], 0, false), true);
            return make_uint2(w[0], w[1]);
        }
    } else {
#pragma unroll
        for (int j = 0; j < EPL; ++j) q[j] = v[j] / s.sc;
    }
    if constexpr (FP8) {
        return make_uint2(pack_fp8x4(q[0], q[1], q[2], q[3]), pack_fp8x4(q[4], q[5], q[6], q[7]));
    } else {
        unsigned w[2] = {0, 0};
#pragma unroll
        for (int j = 0; j < EPL; ++j) w[j >> 2] |= ((unsigned)((int)round_mode(q[j], mode) & 0xff)) << (8 * (j & 3));
        return make_uint2(w[0], w[1]);
    }
}
// the same with the scale worked out here
template <bool FP8>
__device__ __forceinline__ uint2 quant8(const float (&v)[EPL], float m, int mode, float& sc) {
    const QuantScale<FP8> s(m);
    sc = s.sc;
    return quant8_by<FP8>(v, s, mode);
}

// stores what quant8 returned (the scale from the group's first lane; e4m3: fp32, or fp16 in the payload format)
template <bool FP8>
__device__ __forceinline__ void store_quant8(uint2 w, float sc, void* y, int64_t off, void* s, int64_t grp, bool first_lane,
                                             bool fp8_scale_f16 = false) {
    *(uint2*)((uint8_t*)y + off) = w;
    if (!first_lane) return;
    if (FP8 && !fp8_scale_f16) ((float*)s)[grp] = sc;
    else ((unsigned short*)s)[grp] = f32_to_f16(sc);
}

template <bool FP8>
__device__ __forceinline__ void quant_store8(const float (&v)[EPL], float m, void* y, int64_t off, void* s, int64_t grp,
                                             bool first_lane, int mode, bool fp8_scale_f16 = false) {
    float sc;
    const uint2 w = quant8<FP8>(v, m, mode, sc);
    store_quant8<FP8>(w, sc, y, off, s, grp, first_lane, fp8_scale_f16);
}

// round-trip through the storage type: the reference multiplies in the tensor dtype
// (fp16: the value is pinned first.  A product that is only converted to fp16 otherwise becomes
// v_fma_mixlo_f16(a, b, +0), and (-0) + (+0) = +0 loses the sign of a zero product, which the e4m3 quantiser
// behind the activation would store as 0x00 instead of 0x80.)
template <int DT> __device__ __forceinline__ float rnd(float v) {
    if constexpr (DT == LLMK_F16) return f16_to_f32(f32_to_f16(keep_f32(v)));
    else if constexpr (DT == LLMK_BF16) return bf16_to_f32(f32_to_bf16(v));
    else return v;
}

// 1 / (1 + e^-x).  For 16-bit tensors the result is rounded to 8 or 11 significant bits right after, so the
// hardware exp2 and reciprocal (1 ulp each in fp32) are used: large |x| gives exp2 -> inf or 0 and the
// quotient 0 or 1, as the exact expression does.  fp32 tensors keep the library routines.
template <int IDT>
__device__ __forceinline__ float sigmoid_f(float x) {
    if constexpr (IDT == LLMK_F32) return 1.0f / (1.0f + expf(-x));
    else return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * x));
}

// gated activation of one element with the reference's rounding points (activation in fp32, rounded to the
// tensor dtype, product in the tensor dtype, optional per-expert scale in the tensor dtype)
template <int IDT, int ACT>
__device__ __forceinline__ float gated_act(float gv, float up, bool has_scale, float scale) {
    if constexpr (ACT == 0) {
        gv = gv * sigmoid_f<IDT>(gv);
    } else {
        const float kAlpha = 0.7978845608028654f;
        const float u = kAlpha * (gv + 0.044715f * gv * gv * gv);
        const float th = 2.0f * sigmoid_f<IDT>(2.0f * u) - 1.0f;
        gv = 0.5f * gv * (1.0f + th);
    }
    gv = rnd<IDT>(gv);
    float r = rnd<IDT>(gv * up);
    if (has_scale) r = rnd<IDT>(r * scale);
    return r;
}
template <int IDT>
__device__ __forceinline__ float gated_act(float gv, float up, int act, bool has_scale, float scale) {
    return act == 0 ? gated_act<IDT, 0>(gv, up, has_scale, scale) : gated_act<IDT, 1>(gv, up, has_scale, scale);
}
// eight of them.  The branch stands around all eight: one around each made every element a chain of its own, two transcendental instructions long, which
// nothing ran beside.
template <int IDT>
__device__ __forceinline__ void gated_act8(const float (&gv)[EPL], const float (&up)[EPL], int act, bool has_scale, float scale, float (&y)[EPL]) {
    if (act == 0) {
#pragma unroll
        for (int q = 0; q < EPL; ++q) y[q] = gated_act<IDT, 0>(gv[q], up[q], has_scale, scale);
    } else {
#pragma unroll
        for (int q = 0; q < EPL; ++q) y[q] = gated_act<IDT, 1>(gv[q], up[q], has_scale, scale);
    }
}

}  // namespace

// Tile kernels for 4-bit weights on up to some hundred rows: every wave streams its own share of K through its own piece of
// LDS, and the waves of a workgroup meet only at the end of the tile.
//
// A workgroup owns 16 MT rows x 16 NT columns over its whole K range; wave w takes the w-th part of the 128-element K steps.
// Per step it moves the activation rows (128 bytes each), the packed words of its columns and the scale column into its own
// LDS stage by direct-to-LDS loads, reads them into registers as fragments, requests its next step into the stage that is
// free by then, and unpacks and multiplies from registers.  Nothing in the loop waits for another wave: one wave's loads and
// LDS reads run under another one's arithmetic.  The partial sums of the waves meet in LDS once.
//
// Why like this: the tile kernels this replaces expanded the words into int8 rows in LDS for the other waves to read, behind
// one barrier per step, and repeated that for every 32 or 64 rows; the decode kernel read every packed word eight times.
// Fragments must not come straight from global memory: a 64-lane load whose neighbouring lanes lie in different rows takes
// the address path 64 cycles, a coalesced one 17 (measured per 1 KB instruction and CU, from L2).
// What bounds it: vector-ALU work (unpacking: 5.5 instructions per four weights, scaling: 2 per output and step), 60 % of the
// cycles of 16 and of 64 rows alike, and at 16 rows on cold weights HBM; per tile 3 to 5 us for tables, first loads and
// reduction.  us per launch, cold weights, before | now: 16 x 4096 x 4096 9.2 | 6.5, 16 x 14336 x 4096 16.9 | 11.3, 32 x 28672
// x 4096 33.8 | 20.9, 48 x 14336 x 4096 22.8 | 14.1, 64 x 4096 x 14336 32.6 | 20.9, 105 x 4096 x 14336 50.1 | 26.8, 128 x 14336
// x 4096 38.8 | 26.1, 256 x 4096 x 4096 22.5 | 16.0, 512 x 4096 x 4096 31.9 | 25.4.
// Not kept: a second stage where the tile is large (16 x 14336 x 4096 11.3 -> 12.3).
#pragma once
#include "gemm_mid.hpp"
#include "stream_ring.hpp"

namespace llmk {

// one stage of a wave: 16 mt activation rows of 128 bytes, the packed words of 16 nt columns and a K step (64 bytes per
// column), the activation-scale column
constexpr int wv_stage(int mt, int nt) { return 16 * mt * 128 + nt * 1024 + 256; }
constexpr int wv_loads(int mt, int nt) { return 2 * mt + nt + 1; }
constexpr int wv_red(int nw, int mt, int nt) { return nw * 16 * mt * (16 * nt + 4) * 4; }
// scales and zero points of the tile's columns (one byte each) and the block scale, per K step of the workgroup
constexpr int wv_tab_row(int nt) { return 16 * nt + 4; }         // bytes; + 4: the steps of a column start in different banks
constexpr int wv_tab(int nt, int steps) { return steps * (2 * wv_tab_row(nt) + 4); }
constexpr int wv_lds(int nw, int mt, int nt, int d, int steps) {
    const int a = nw * d * wv_stage(mt, nt) + wv_tab(nt, steps), b = wv_red(nw, mt, nt);
    return a > b ? a : b;
}

// K steps of a workgroup: their block scales are loaded by one load of its 256 or 512 threads
constexpr int WV_MAX_STEPS = 256;
// stages of a wave: two for 16-row tiles of at most 32 columns, where every wave has at least two steps
constexpr int wv_depth(int mt, int nt, int64_t steps) { return mt == 1 && nt <= 2 && steps >= 16 ? 2 : 1; }

// two 16-bit integers in a register
typedef unsigned short wv_us2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ wv_us2 wv_as_us2(unsigned u) { return __builtin_bit_cast(wv_us2, u); }
__device__ __forceinline__ unsigned wv_bits(wv_us2 v) { return __builtin_bit_cast(unsigned, v); }

template <int N>
__device__ __forceinline__ void wv_wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

// int8 activations [M, K] with a scale per row and 128 elements, uint4 weights packed eight rows per word [N / 8, K] with an int8
// zero point and scale per row and 128 elements (groups) and a scale per 128 x 128 block: the int8 weight is
// int8(int8(q - z4) * s4) with two's-complement wrap.
// S32: fp32 scales, else 16-bit ones (fp16 or bf16 by p.s_dtype)
template <int NW, int MT, int NT, int D, bool S32>
__global__ __launch_bounds__((NW * 64)) void w4a8_wave_kernel(DirectArgs p) {
    constexpr int BM = 16 * MT, BN = 16 * NT, STAGE = wv_stage(MT, NT), LPS = wv_loads(MT, NT);
    constexpr int OFF_B = BM * 128, OFF_S = OFF_B + NT * 1024, TR = wv_tab_row(NT);
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int N = p.N, K = p.K, KT_all = K >> 7;
    int kt0 = 0, KT = KT_all;
    if (p.ksplit > 1) {
        const int per = (KT_all + p.ksplit - 1) / p.ksplit;
        kt0 = (int)blockIdx.z * per;
        KT = min(per, KT_all - kt0);
    }
    const int n0 = blockIdx.x * BN, m0 = blockIdx.y * BM, m_end = min(p.M, m0 + BM);
    if (n0 >= N) return;                                    // the grid is padded to a multiple of the XCDs
    const int s_lo = wave * KT / NW, n = (wave + 1) * KT / NW - s_lo;

    uint8_t* const mine = lds + wave * (D * STAGE);
    const uint32_t mine_addr = lds_base + (uint32_t)wave * (D * STAGE);
    uint8_t* const tab_s = lds + NW * D * STAGE;          // [K step][column]
    uint8_t* const tab_z = tab_s + KT * TR;
    float* const bsl = (float*)(tab_z + KT * TR);

    // ---- tables, requested first, by loads that share the hand-counted scheme: the wait for them leaves the first stages in
    // flight.  (Only K ranges of more than 8192 / NT elements of a column have a second round of them, by ordinary loads.)
    const bool s_f16 = p.s_dtype == LLMK_F16;
    auto scale_f32 = [&](unsigned raw) { return S32 ? __uint_as_float(raw) : (s_f16 ? f16_to_f32((unsigned short)raw) : bf16_to_f32((unsigned short)raw)); };
    constexpr uint32_t ssz = S32 ? 4u : 2u;
    const int8_t* const tab4 = p.w4_s4 + (int64_t)n0 * KT_all;
    const int8_t* const tabz = p.w4_z4 + (int64_t)n0 * KT_all;
    const int W = (KT + 3) >> 2;                             // dwords per column (the last one may reach past the range)
    const uint32_t tab_last = (uint32_t)min((int64_t)(N - n0) * KT_all - 4, (int64_t)0x7fffffff);
    auto tab_at = [&](int idx, int& col, int& w, int& shift) {
        col = idx / W;
        w = idx - col * W;
        const uint32_t want = (uint32_t)min(min(col, BN - 1), N - 1 - n0) * (uint32_t)KT_all + (uint32_t)(kt0 + 4 * w);
        const uint32_t at = min(want, tab_last);
        shift = (int)(want - at) * 8;
        return at;
    };
    auto tab_put = [&](int col, int w, int shift, unsigned s4, unsigned z4) {
        s4 = shift < 32 ? s4 >> shift : 0u;
        z4 = shift < 32 ? z4 >> shift : 0u;
#pragma unroll
        for (int b = 0; b < 4; ++b)
            if (4 * w + b < KT) {
                tab_s[(4 * w + b) * TR + col] = (uint8_t)(s4 >> (8 * b));
                tab_z[(4 * w + b) * TR + col] = (uint8_t)(z4 >> (8 * b));
            }
    };
    int t_col, t_w, t_shift, t_s, t_z, t_bs;
    {
        const uint32_t at = tab_at(tid, t_col, t_w, t_shift);
        t_s = ring_load_b32<0>(at, ring_base(tab4));
        t_z = ring_load_b32<0>(at, ring_base(tabz));
        const RingBase bsb = ring_base((const uint8_t*)p.b_s + ((int64_t)(n0 >> 7) * KT_all + kt0) * ssz);
        const uint32_t bat = (uint32_t)min(tid, KT - 1) * ssz;
        if constexpr (S32) t_bs = ring_load_b32<0>(bat, bsb);
        else t_bs = ring_load_u16<0>(bat, bsb);
    }

    // ---- source offsets of the loads of a stage
    uint32_t aoff[2 * MT], boff[NT];
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) {
        const int row = 8 * i + (lane >> 3);
        aoff[i] = (uint32_t)min(row, m_end - 1 - m0) * (uint32_t)K + (uint32_t)((lane & 7) ^ ((row >> 1) & 7)) * 16u;
    }
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        const int pr = 2 * i + (lane >> 5);
        boff[i] = (uint32_t)min(pr, ((N - n0) >> 3) - 1) * (uint32_t)(K * 4) + (uint32_t)((lane & 31) ^ pr) * 16u;
    }
    const uint32_t soff = (uint32_t)min(min(lane, BM - 1), m_end - 1 - m0) * (uint32_t)KT_all * ssz;
    const uint8_t* const ga = p.a + (int64_t)m0 * K;
    const uint8_t* const gb = p.b + (int64_t)(n0 >> 3) * K * 4;
    const uint8_t* const gs = (const uint8_t*)p.a_s + (int64_t)m0 * KT_all * ssz;
    auto issue = [&](int slot, int s) __attribute__((always_inline)) {
        const int kb = kt0 + min(s, KT - 1);
        const uint32_t st = mine_addr + (uint32_t)slot * STAGE;
#pragma unroll
        for (int i = 0; i < NT; ++i) dma16(st + OFF_B + i * 1024u, boff[i], gb + (int64_t)kb * 512);
#pragma unroll
        for (int i = 0; i < 2 * MT; ++i) dma16(st + i * 1024u, aoff[i], ga + (int64_t)kb * 128);
        if constexpr (S32) dma4(st + OFF_S, soff, gs + (int64_t)kb * 4);
        else dma2(st + OFF_S, soff, gs + (int64_t)kb * 2);
    };
#pragma unroll
    for (int d = 0; d < D; ++d) issue(d, s_lo + d);

    ring_wait<D * LPS>(t_s, t_z, t_bs);
    if (tid < BN * W) tab_put(t_col, t_w, t_shift, (unsigned)t_s, (unsigned)t_z);
    for (int idx = tid + (NW * 64); idx < BN * W; idx += (NW * 64)) {
        int col, w, shift;
        const uint32_t at = tab_at(idx, col, w, shift);
        unsigned vs, vz;
        __builtin_memcpy(&vs, tab4 + at, 4);
        __builtin_memcpy(&vz, tabz + at, 4);
        tab_put(col, w, shift, vs, vz);
    }
    if (tid < KT) bsl[tid] = scale_f32((unsigned)t_bs);
    __syncthreads();

    // acc[mt][j][i] = C[row 16 mt + r][column NT (4 g + i) + j] over this wave's K steps
    v4f acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};

    // lane (r, g) of the weight fragment j is column NT r + j: nibble (NT r + j) & 7 of packed row pr
    const int pr = (NT * r) >> 3, sub = NT == 4 ? (r & 1) : (NT == 2 ? (r & 3) : (r & 7));
    const unsigned sel = NT == 4 ? (sub ? 0x07060302u : 0x05040100u)
                                 : (0x0c000c00u | (unsigned)(NT == 2 ? sub : sub >> 1) | ((unsigned)(4 + (NT == 2 ? sub : sub >> 1)) << 16));
    const int swz = (r >> 1) & 7;
    const int lo = r * 128 + ((g ^ swz) * 16), hi = r * 128 + (((g + 4) ^ swz) * 16);

    v4i a_lo[MT], a_hi[MT];
    unsigned a_sc[MT];
    unsigned h[8][2];                                        // 16-bit nibble holders of words 4 q .. 4 q + 3 of the lane's eight quads
    auto fetch = [&](int slot) __attribute__((always_inline)) {
        const uint8_t* st = mine + slot * STAGE;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            a_lo[mt] = *(const v4i*)(st + mt * 2048 + lo);
            a_hi[mt] = *(const v4i*)(st + mt * 2048 + hi);
            a_sc[mt] = *(const unsigned*)(st + OFF_S + (16 * mt + r) * 4);
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int c = 16 * (q >> 2) + 4 * g + (q & 3);
            const v4i w = *(const v4i*)(st + OFF_B + pr * 512 + ((c ^ pr) * 16));
            h[q][0] = __builtin_amdgcn_perm((unsigned)w[1], (unsigned)w[0], sel);
            h[q][1] = __builtin_amdgcn_perm((unsigned)w[3], (unsigned)w[2], sel);
        }
    };
    // q * s + c in the high byte of a 16-bit lane, c = -z * s: the nibble stays where it is in the word (q << a) and the
    // scale is shifted by 8 - a instead; the low byte of the product is the int8 weight with its two's-complement wrap
    auto compute = [&](int s) __attribute__((always_inline)) {
        const float bs = bsl[s];
        float sa[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
            sa[mt] = scale_f32(a_sc[mt]) * bs;
        unsigned s4, z4;
        if constexpr (NT == 4) { s4 = *(const unsigned*)(tab_s + s * TR + 4 * r); z4 = *(const unsigned*)(tab_z + s * TR + 4 * r); }
        else if constexpr (NT == 2) { s4 = *(const unsigned short*)(tab_s + s * TR + 2 * r); z4 = *(const unsigned short*)(tab_z + s * TR + 2 * r); }
        else { s4 = tab_s[s * TR + r]; z4 = tab_z[s * TR + r]; }
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const unsigned sj = (s4 >> (8 * j)) & 0xffu, zj = (z4 >> (8 * j)) & 0xffu;
            const unsigned c8 = (0u - __umul24(zj, sj)) << 8;
            const unsigned cp = __builtin_amdgcn_perm(c8, c8, 0x01000100u);
            unsigned mask, sh;
            if constexpr (NT == 1) { mask = sub & 1 ? 0x00f000f0u : 0x000f000fu; sh = sub & 1 ? 4u : 8u; }
            else { mask = j == 3 ? 0u : 0x000f000fu << (4 * j); sh = j == 3 ? 8u : 8u - 4u * j; }
            const unsigned sx = sj << sh;
            const unsigned sp = __builtin_amdgcn_perm(sx, sx, 0x01000100u);
            v4i b[2];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                unsigned x0, x1;
                if (NT == 4 && j == 3) {
                    x0 = wv_bits(wv_as_us2(h[q][0]) >> (unsigned short)12);
                    x1 = wv_bits(wv_as_us2(h[q][1]) >> (unsigned short)12);
                } else {
                    x0 = h[q][0] & mask;
                    x1 = h[q][1] & mask;
                }
                const unsigned y0 = wv_bits(wv_as_us2(x0) * wv_as_us2(sp) + wv_as_us2(cp));
                const unsigned y1 = wv_bits(wv_as_us2(x1) * wv_as_us2(sp) + wv_as_us2(cp));
                b[q >> 2][q & 3] = (int)__builtin_amdgcn_perm(y1, y0, 0x07050301u);
            }
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                v4i t = {0, 0, 0, 0};
                t = mfma_i8_16x16x64(b[0], a_lo[mt], t);
                t = mfma_i8_16x16x64(b[1], a_hi[mt], t);
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[mt][j][i] = fmaf((float)t[i], sa[mt], acc[mt][j][i]);
            }
        }
    };

    int i = 0, slot = 0;
    for (; i + D < n; ++i) {
        wv_wait_loads<(D - 1) * LPS>();
        fetch(slot);
        __builtin_amdgcn_s_waitcnt(0xc07f);                  // lgkmcnt(0): the slot is free
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        issue(slot, s_lo + i + D);
        __builtin_amdgcn_sched_barrier(0);
        compute(s_lo + i);
        slot = slot + 1 == D ? 0 : slot + 1;
    }
    md_static_for<0, D>([&](auto dc) __attribute__((always_inline)) {
        constexpr int d = decltype(dc)::value;
        if (i < n) {
            wv_wait_loads<(D - 1 - d) * LPS>();
            fetch(slot);
            compute(s_lo + i);
            slot = slot + 1 == D ? 0 : slot + 1;
            ++i;
        }
    });
    wv_wait_loads<0>();
    __syncthreads();

    // ---- the eight partial sums of every output meet in LDS
    constexpr int RED_ROW = BN + 4;
    float* red = (float*)lds;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        float* dst = red + (wave * BM + 16 * mt + r) * RED_ROW + 4 * NT * g;
        if constexpr (NT == 4) {
#pragma unroll
            for (int e = 0; e < 4; ++e) *(v4f*)(dst + 4 * e) = (v4f){acc[mt][0][e], acc[mt][1][e], acc[mt][2][e], acc[mt][3][e]};
        } else if constexpr (NT == 2) {
#pragma unroll
            for (int e = 0; e < 4; e += 2) *(v4f*)(dst + 2 * e) = (v4f){acc[mt][0][e], acc[mt][1][e], acc[mt][0][e + 1], acc[mt][1][e + 1]};
        } else {
            *(v4f*)dst = acc[mt][0];
        }
    }
    __syncthreads();
    constexpr int RUNS = BN / 8, ROWS_PASS = (NW * 64) / RUNS;
    const bool split = p.ksplit > 1;
    void* cout = split ? (void*)(p.partial + (int64_t)blockIdx.z * p.M * N) : p.c;
    const int cdt = split ? LLMK_F32 : p.c_dtype;
    const int esz = cdt == LLMK_F32 ? 4 : 2;
    const bool vec_ok = ((((uintptr_t)cout) & 15) == 0) && (((int64_t)N * esz) % 16 == 0);
    const int ocol = 8 * (tid % RUNS), nn = n0 + ocol, nv = N - nn;
    if (nn >= N) return;
#pragma unroll
    for (int pass = 0; pass < (BM + ROWS_PASS - 1) / ROWS_PASS; ++pass) {
        const int orow = pass * ROWS_PASS + tid / RUNS, m = m0 + orow;
        if (orow >= BM || m >= m_end) continue;
        v4f sa = {0.f, 0.f, 0.f, 0.f}, sb = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const float* src = red + (w * BM + orow) * RED_ROW + ocol;
            sa += *(const v4f*)src;
            sb += *(const v4f*)(src + 4);
        }
        const int64_t off = (int64_t)m * N + nn;
        if (cdt == LLMK_BF16) store_run8<LLMK_BF16>(cout, off, sa, sb, nv, vec_ok);
        else if (cdt == LLMK_F16) store_run8<LLMK_F16>(cout, off, sa, sb, nv, vec_ok);
        else store_run8<LLMK_F32>(cout, off, sa, sb, nv, vec_ok);
    }
}

template <int NW, int MT, int NT, int D, bool S32>
int launch_w4a8_wave(const DirectArgs& p, int z, hipStream_t stream, const char* name) {
    static std::atomic<uint64_t> configured{0};
    auto kern = w4a8_wave_kernel<NW, MT, NT, D, S32>;
    const int KT_all = p.K >> 7, per = (KT_all + z - 1) / z;
    const int bytes = wv_lds(NW, MT, NT, D, per);
    if (bytes > D_LDS_MAX) LLMK_FAIL(LLMK_ERR_SHAPE, "%s: %d bytes of LDS needed", name, bytes);
    if (int rc = llmk_reserve_lds((const void*)kern, D_LDS_MAX, configured, name)) return rc;
    DirectArgs q = p;
    q.ksplit = z;
    const int zg = (KT_all + per - 1) / per;
    unsigned gx = (unsigned)((p.N + 16 * NT - 1) / (16 * NT)), gy = (unsigned)((p.M + 16 * MT - 1) / (16 * MT));
    if (gy > 1) gx = (gx + 7) & ~7u;
    kern<<<dim3(gx, gy, (unsigned)zg), (NW * 64), bytes, stream>>>(q);
    LLMK_CHECK_LAUNCH(name);
    if (z > 1) {
        const int64_t mn = (int64_t)p.M * p.N;
        const unsigned blocks = (unsigned)cdiv64(cdiv64(mn, 4), 256);
        if (p.c_dtype == LLMK_BF16) splitk_sum_kernel<LLMK_BF16><<<blocks, 256, 0, stream>>>(p.partial, p.c, mn, zg);
        else if (p.c_dtype == LLMK_F16) splitk_sum_kernel<LLMK_F16><<<blocks, 256, 0, stream>>>(p.partial, p.c, mn, zg);
        else splitk_sum_kernel<LLMK_F32><<<blocks, 256, 0, stream>>>(p.partial, p.c, mn, zg);
        LLMK_CHECK_LAUNCH(name);
    }
    return LLMK_OK;
}

// Launch shape: waves per workgroup, row and column tiles of a wave, K slices over workgroups, estimated microseconds.
struct WavePlan {
    int nw, mt, nt, z;
    double cost;
};

// us of a tile of eight waves per K step of each of them, [mt - 1][log2 nt] (a fit to launches of 8 to 14 steps a wave)
constexpr double WV_STEP_US[4][3] = {{0.68, 0.94, 1.38}, {1.04, 1.30, 1.68}, {1.43, 1.58, 1.90}, {1.75, 1.86, 2.30}};

// The cheapest shape that fits.  Eight waves: rounds of 256 workgroups, each a fixed part (tables, first loads, reduction) and
// its steps.  Four waves (48 and 64 rows, 64 columns): two workgroups share a CU and cover each other's fixed parts, so their
// rounds are counted in fractions; slower on a single round (64 x 14336 x 4096 18.2 against 17.0 us), faster from two on
// (64 x 28672 x 4096 27.6 against 30.2, 128 rows 46.8 against 54).  K slices cost a second launch and their fp32 sums.
inline bool w4a8_wave_plan(int64_t M, int64_t N, int64_t K, int64_t scratch, WavePlan& best) {
    const int64_t KT = K >> 7;
    bool found = false;
    for (int nw = 8; nw >= 4; nw -= 4)
        for (int mt = 1; mt <= 4; ++mt)
            for (int nt = 1; nt <= 4; nt *= 2) {
                if ((mt > 1 && M <= 16 * (mt - 1)) || (nw == 4 && (mt < 3 || nt < 4))) continue;
                const int64_t tiles = ((N + 16 * nt - 1) / (16 * nt)) * ((M + 16 * mt - 1) / (16 * mt));
                const int64_t zmin = (KT + WV_MAX_STEPS - 1) / WV_MAX_STEPS;
                for (int64_t z = zmin; z <= (zmin > 4 ? zmin : 4); z *= 2) {
                    const int64_t per = (KT + z - 1) / z;
                    if (z > 1 && ((z > zmin && (per < 8 || tiles * z > 320)) || scratch < z * M * N * 4)) continue;
                    if (wv_lds(nw, mt, nt, wv_depth(mt, nt, per), (int)per) > D_LDS_MAX) continue;
                    const int64_t steps = (per + nw - 1) / nw;
                    double cost;
                    if (nw == 8) cost = (double)((tiles * z + LLMK_CUS - 1) / LLMK_CUS) * ((nt < 4 ? 2.5 : 4.5) + steps * WV_STEP_US[mt - 1][nt >> 1]);
                    else cost = 6.0 + (tiles * z > LLMK_CUS ? (double)(tiles * z) / LLMK_CUS : 1.0) * steps * (mt == 4 ? 1.22 : 1.04);
                    if (z > 1) cost += 3.5 + (double)(z * M * N) * 8.0 / 5e6;
                    if (!found || cost < best.cost) best = WavePlan{nw, mt, nt, (int)z, cost};
                    found = true;
                }
            }
    return found;
}

inline int launch_w4a8_wave_plan(const DirectArgs& p, const WavePlan& w, hipStream_t stream, const char* name) {
    const int per = (int)(((p.K >> 7) + w.z - 1) / w.z);
    auto run = [&](auto nw, auto mt, auto nt, auto d) {
        constexpr int NW = decltype(nw)::value, MT = decltype(mt)::value, NT = decltype(nt)::value, D = decltype(d)::value;
        return p.s_dtype == LLMK_F32 ? launch_w4a8_wave<NW, MT, NT, D, true>(p, w.z, stream, name) : launch_w4a8_wave<NW, MT, NT, D, false>(p, w.z, stream, name);
    };
    const std::integral_constant<int, 1> i1;
    const std::integral_constant<int, 2> i2;
    const std::integral_constant<int, 3> i3;
    const std::integral_constant<int, 4> i4;
    const std::integral_constant<int, 8> i8;
    if (w.nw == 4) return w.mt == 4 ? run(i4, i4, i4, i1) : run(i4, i3, i4, i1);
    const bool deep = wv_depth(w.mt, w.nt, per) == 2;
    auto rows = [&](auto mt) {
        if (w.nt == 4) return run(i8, mt, i4, i1);
        if constexpr (decltype(mt)::value == 1) {
            if (deep) return w.nt == 2 ? run(i8, mt, i2, i2) : run(i8, mt, i1, i2);
        }
        return w.nt == 2 ? run(i8, mt, i2, i1) : run(i8, mt, i1, i1);
    };
    return w.mt == 1 ? rows(i1) : (w.mt == 2 ? rows(i2) : (w.mt == 3 ? rows(i3) : rows(i4)));
}

}  // namespace llmk

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

// Tile of a workgroup.  Ids go to the eight XCDs round robin; each XCD takes an eighth of the list of tiles, column by column with
// the row tiles of a column back to back, so that a column's weights are read through one L2.  (Columns dealt to the XCDs whole
// give some of them more tiles than they have CUs: 216 x 2304 x 1280 16.3 us for 252 tiles, 9.1 this way.)
struct WaveTile {
    int col, row;
};
__device__ __forceinline__ WaveTile wave_tile(int M, int bm, FastDiv by_rows) {
    const int lin = blockIdx.x, total = gridDim.x, rows = (M + bm - 1) / bm, x = lin & 7;
    const int idx = x * (total >> 3) + min(x, total & 7) + (lin >> 3);
    const int col = (int)by_rows((uint32_t)idx);
    return {col, idx - col * rows};
}

// The launch arguments in front of the first loads of an 8-bit kernel, asked for in one round trip: used here, they are all loaded before the first wait.
// Left to itself the compiler gave the register of an argument that no wave kernel uses (it came with its neighbours) to the next value, waited for all of
// them to do so, and only then asked for the division by the row tiles and the grid: a second trip, to HBM where the weights have displaced the arguments.
// us, weights from HBM, two trips | one: per token 5 x 4096 x 4096 5.80 | 5.54, 12 x 4096 x 4096 6.49 | 6.09, 46 x 1288 x 8320 7.92 | 7.55, 5 x 28672 x
// 4096 22.67 | 22.33; 60 shapes of 1 to 64 rows each, per token 1.03 times as fast, fp8 and int8 1.004.
__device__ __forceinline__ void wv_arguments(const DirectArgs& p) {
    asm volatile("" ::"s"(p.a), "s"(p.b), "s"(p.a_s), "s"(p.b_s), "s"(p.M), "s"(p.N), "s"(p.K), "s"(p.s_dtype), "s"(p.ksplit), "s"(p.by_rows.mul), "s"(p.by_rows.shift),
                 "s"((int)gridDim.x));
}

template <int N>
__device__ __forceinline__ void wv_wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

// The end of a tile, behind the barrier that follows the waves' writes: red [wave][row][column], rows of 16 NT + 4 floats, is
// summed over the waves in their order and stored (K slices: as fp32 sums).  A thread owns eight columns of a row.
// ROWCOL: int32 sums, scaled per row and column here.
template <int NW, int MT, int NT, bool ROWCOL = false>
__device__ __forceinline__ void wv_store(const DirectArgs& p, const float* red, int n0, int m0, int m_end) {
    constexpr int BM = 16 * MT, BN = 16 * NT, RED_ROW = BN + 4, RUNS = BN / 8, ROWS_PASS = (NW * 64) / RUNS;
    const int tid = threadIdx.x, N = p.N;
    const bool split = p.ksplit > 1;
    void* cout = split ? (void*)(p.partial + (int64_t)blockIdx.z * p.M * N) : p.c;
    const int cdt = split ? LLMK_F32 : p.c_dtype;
    const int ocol = 8 * (tid % RUNS), nn = n0 + ocol, nv = N - nn;
    if (nn >= N) return;
#pragma unroll
    for (int pass = 0; pass < (BM + ROWS_PASS - 1) / ROWS_PASS; ++pass) {
        const int orow = pass * ROWS_PASS + tid / RUNS, m = m0 + orow;
        if (orow >= BM || m >= m_end) continue;
        v4f sa = {0.f, 0.f, 0.f, 0.f}, sb = {0.f, 0.f, 0.f, 0.f};
        v4i ia = {0, 0, 0, 0}, ib = {0, 0, 0, 0};
        // four waves' reads on their way before their first sum: few threads have an output here, and each would wait for one read after the other
#pragma unroll
        for (int w0 = 0; w0 < NW; w0 += 4) {
            v4f part[4][2];
#pragma unroll
            for (int w = 0; w < 4; ++w)
#pragma unroll
                for (int h = 0; h < 2; ++h) part[w][h] = *(const v4f*)(red + ((w0 + w) * BM + orow) * RED_ROW + ocol + 4 * h);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                if constexpr (ROWCOL) {
                    ia += __builtin_bit_cast(v4i, part[w][0]);
                    ib += __builtin_bit_cast(v4i, part[w][1]);
                } else {
                    sa += part[w][0];
                    sb += part[w][1];
                }
            }
            // (the sums are made here: eight waves' reads at a time take more registers than the loop)
            if constexpr (ROWCOL) asm volatile("" : "+v"(ia), "+v"(ib) : : "memory");
            else asm volatile("" : "+v"(sa), "+v"(sb) : : "memory");
        }
        const int64_t off = (int64_t)m * N + nn;
        if constexpr (ROWCOL) {
            sa = __builtin_bit_cast(v4f, ia);
            sb = __builtin_bit_cast(v4f, ib);
            rowcol_epilogue8(p, sa, sb, m, off, nn, nv);
            if (!p.c) continue;
        }
        if (cdt == LLMK_BF16) store_run8<LLMK_BF16>(cout, off, sa, sb, nv);
        else if (cdt == LLMK_F16) store_run8<LLMK_F16>(cout, off, sa, sb, nv);
        else store_run8<LLMK_F32>(cout, off, sa, sb, nv);
    }
}

// Summing pass of a launch whose K range was sliced.
inline int wv_sum_slices(const DirectArgs& p, int z, hipStream_t stream, const char* name) {
    const int64_t mn = (int64_t)p.M * p.N;
    const unsigned blocks = (unsigned)cdiv64(cdiv64(mn, 4), 256);
    if (p.c_dtype == LLMK_BF16) splitk_sum_kernel<LLMK_BF16><<<blocks, 256, 0, stream>>>(p.partial, p.c, mn, z);
    else if (p.c_dtype == LLMK_F16) splitk_sum_kernel<LLMK_F16><<<blocks, 256, 0, stream>>>(p.partial, p.c, mn, z);
    else splitk_sum_kernel<LLMK_F32><<<blocks, 256, 0, stream>>>(p.partial, p.c, mn, z);
    LLMK_CHECK_LAUNCH(name);
    return LLMK_OK;
}

// int8 activations [M, K] with a scale per row and 128 elements, uint4 weights packed eight rows per word [N / 8, K] with an int8
// zero point and scale per row and 128 elements (groups) and a scale per 128 x 128 block: the int8 weight is
// int8(int8(q - z4) * s4) with two's-complement wrap.
// S32: fp32 scales, else 16-bit ones (fp16 or bf16 by p.s_dtype)
template <int NW, int MT, int NT, int D, bool S32>
__global__ __launch_bounds__(NW * 64) void w4a8_wave_kernel(DirectArgs p) {
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
    const WaveTile tile = wave_tile(p.M, BM, p.by_rows);
    const int n0 = tile.col * BN, m0 = tile.row * BM, m_end = min(p.M, m0 + BM);
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
    // dwords per column of a whole slice (the last ones may reach past the range)
    const int W = p.words;
    const uint32_t tab_last = (uint32_t)min((int64_t)(N - n0) * KT_all - 4, (int64_t)0x7fffffff);
    auto tab_at = [&](int idx, int& col, int& w, int& shift) {
        col = (int)p.by_words((uint32_t)idx);
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
    for (int idx = tid + NW * 64; idx < BN * W; idx += NW * 64) {
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
    wv_store<NW, MT, NT>(p, red, n0, m0, m_end);
}

template <int NW, int MT, int NT, int D, bool S32>
int launch_w4a8_wave(const DirectArgs& p, int z, hipStream_t stream, const char* name) {
    static std::atomic<uint64_t> configured{0};
    auto kern = w4a8_wave_kernel<NW, MT, NT, D, S32>;
    const int KT_all = p.K >> 7, per = (KT_all + z - 1) / z;
    const int bytes = wv_lds(NW, MT, NT, D, per);
    if (bytes > D_LDS_MAX) LLMK_FAIL(LLMK_ERR_SHAPE, "%s: %d bytes of LDS needed", name, bytes);
    if (bytes > 64 * 1024)       // (less needs no leave, and asking for it costs a decode call 0.1 us)
        if (int rc = llmk_reserve_lds((const void*)kern, D_LDS_MAX, configured, name)) return rc;
    DirectArgs q = p;
    q.ksplit = z;
    const int zg = (KT_all + per - 1) / per, rows = (p.M + 16 * MT - 1) / (16 * MT);
    const unsigned tiles = (unsigned)(((p.N + 16 * NT - 1) / (16 * NT)) * rows);
    q.by_rows = fast_div((uint32_t)rows);
    q.words = (per + 3) >> 2;
    q.by_words = fast_div((uint32_t)q.words);
    kern<<<dim3(tiles, 1, (unsigned)zg), NW * 64, bytes, stream>>>(q);
    LLMK_CHECK_LAUNCH(name);
    if (z > 1) return wv_sum_slices(p, zg, stream, name);
    return LLMK_OK;
}

// ------------------------------------------------------------------------------------------------------------
// fp16 / bf16 activations [M, K], 4-bit weights with fp16 group scales: row-packed [N, K / 8] (K_W4NK, K_W4NKB) or Marlin words
// (K_W4MARLIN).  K steps are 128 elements of weights and two halves of 64 elements (128 bytes) of activations.  16-row tiles: a wave has one stage
// for a whole step, words and both halves.  More rows: one stage of activation rows, half a step, requested a half ahead, and two of packed
// words (a second stage of activations has no room beside 64 rows).
// What bounds it: latency.  64 x 14336 x 4096, of 37600 cycles a wave lives: vector ALU 46 %, address path 52 %, LDS 30 %, MFMA 22 %;
// a half's activations are requested one half ahead, which two waves per SIMD do not cover.  The words of a chunk come from LDS
// with the order of the activations' dwords as the Marlin fragments want it; scattering them into rows was most of the tile kernel.
// us per launch, before | now, cold weights: Marlin 16 x 14336 x 4096 18.5 | 14.4, 64 x 14336 x 4096 47.0 | 20.1, 96 x 4096 x 14336
// 52.2 | 26.9, 256 x 4096 x 4096 35.9 | 19.0; [N, K / 8] bf16 48 x 22096 x 4352 42.4 | 32.4, 80 x 4096 x 4096 19.2 | 12.8, 160 x 4096 x
// 14336 75.0 | 44.6, fp16 128 x 8192 x 8192 51.5 | 33.6.
constexpr int wh_a(int mt) { return 16 * mt * 128; }
constexpr bool wh_marlin(int kind) { return kind == K_W4MARLIN; }
constexpr int wh_b(int kind, int nt) { return wh_marlin(kind) ? 4096 : nt * 1024; }     // Marlin: the whole 64-column chunk
// 16 rows: a whole K step; more: the activations of a half, and the words of two steps
constexpr int wh_stage(int kind, int mt, int nt) { return mt == 1 ? 2 * wh_a(1) + wh_b(kind, nt) : wh_a(mt) + 2 * wh_b(kind, nt); }
constexpr int wh_tab_cols(int kind, int nt) { return wh_marlin(kind) ? 64 : 16 * nt; }
constexpr int wh_tab_row(int kind, int nt) { return 2 * wh_tab_cols(kind, nt) + 8; }
constexpr int wh_lds(int kind, int nw, int mt, int nt, int groups) {
    const int a = nw * wh_stage(kind, mt, nt) + wh_tab_row(kind, nt) * groups, b = wv_red(nw, mt, nt);
    return a > b ? a : b;
}

// groups that `per` K steps touch, at most
constexpr int wh_groups(int K, int group, int per) {
    const int a = (per * 128 - 1) / group + 2, b = K / group;
    return a < b ? a : b;
}

// Scales of a row-packed tile are loaded four at a time (8 bytes) at the offset of the first one, but no further than the end of the
// table: a load there starts earlier and is shifted.  A last tile of fewer than four scales (one column and groups as long as K, say)
// has its loads start in front of its own first column: `back` bytes, for a table of at least four scales in all (w4a16_wave_plan).
struct WhTable {
    int64_t back, last;          // bytes in front of the tile's first scale; offset (from there) of the last load
};
__host__ __device__ constexpr WhTable wh_table(int64_t scales) {       // from the tile's first column to the end of the table
    const int64_t bytes = 2 * scales, back = bytes < 8 ? 8 - bytes : 0;
    return {back, bytes + back - 8};
}
constexpr bool wh_table_covers(int64_t scales) {
    const WhTable t = wh_table(scales);
    for (int64_t i = 0; i < scales; ++i) {
        const int64_t want = t.back + 2 * i, at = want < t.last ? want : t.last;
        if (at < 0 || at + 8 > t.back + 2 * scales || want - at > 6) return false;
    }
    return true;
}
static_assert(wh_table_covers(1) && wh_table_covers(2) && wh_table_covers(3) && wh_table_covers(4) && wh_table_covers(5) && wh_table_covers(63),
              "every load of scales ends inside the table and holds its scale");

// PRE: the weights are (q - 8) * scale rounded to the activations' type, as the tile kernels of larger M have them (and the
// reference's Marlin kernel: marlin_w4a16_gemm.cu:152-236), and sums run over all of K; otherwise they are q - 8 exactly and the scale
// multiplies the fp32 sums of a half step.  Marlin words always, row-packed ones where the caller's rule says so.  (us, weights from
// HBM, exact weights | rounded: Marlin 16 x 4096 x 4096 8.2 | 8.1, 64 x 14336 x 4096 18.4 | 18.0, 128 x 4096 x 4096 12.0 | 12.7, 16 x 4096 x
// 14336 13.8 | 14.5, fp16 160 x 4096 x 14336 40.1 | 40.1: the scale is one more packed product a word, or a product an output and half step.)
template <int KIND, int NW, int MT, int NT, bool PRE>
__global__ __launch_bounds__(NW * 64) void w4a16_wave_kernel(DirectArgs p) {
    static_assert(is_w4nk(KIND) || wh_marlin(KIND), "4-bit weights, 16-bit activations");
    static_assert(PRE || !wh_marlin(KIND), "Marlin words: scaled weights");
    constexpr bool MARLIN = wh_marlin(KIND), BF = (KIND == K_W4NKB);
    constexpr int BM = 16 * MT, BN = 16 * NT, STAGE = wh_stage(KIND, MT, NT), WB = wh_b(KIND, NT), NB = WB / 1024;
    // 16 rows: a step's words and activations are one request, and the wave waits once for them: us, halves | whole steps, weights in the cache (from
    // HBM): Marlin words 16 x 4096 x 4096 6.49 (7.22) | 6.30 (6.76), 16 x 14336 x 4096 10.4 (12.1) | 10.1 (11.7), 16 x 9984 x 1152 6.2 (6.7) | 5.8 (6.2); row-packed
    // ones, fp16 20 x 1416 x 11904 9.6 (12.7) | 8.7 (11.0), 44 x 2240 x 5248 7.7 (9.2) | 7.5 (8.6), bf16 29 x 4096 x 14336 15.8 (18.4) | 13.7 (15.9), 34 x 4208 x 4864
    // 9.7 (11.5) | 10.0 (11.3).  25 random shapes a type and width, 16, 32, 64 columns: bf16 1.11 (1.11), 1.12 (1.15), 0.98 (1.02) times as fast as in halves,
    // fp16 1.07 (1.10), 1.03 (1.07), 1.03 (1.03).  The larger stage (5 KB a wave for 4 at 16 columns) costs no residency: of 57000 calls that get 16-row tiles
    // of row-packed words all on eight waves are at most one workgroup a CU, those on four at most two.  Two stages of whole steps are
    // slower (Marlin 16 x 4096 x 4096 6.85: twice the loads are issued in front of the scale table), and so are whole steps of 32 rows from HBM (Marlin 32 x
    // 14336 x 4096 14.1 | 14.7).
    constexpr bool WHOLE = MT == 1;
    constexpr int OFF_B = (WHOLE ? 2 : 1) * wh_a(MT);
    constexpr int TR = wh_tab_row(KIND, NT), TC = wh_tab_cols(KIND, NT);
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int N = p.N, K = p.K, KT_all = K >> 7, G = (int)p.by_group((uint32_t)KT_all), nchunks = N >> 6;
    int kt0 = 0, KT = KT_all;
    if (p.ksplit > 1) {
        const int per = (KT_all + p.ksplit - 1) / p.ksplit;
        kt0 = (int)blockIdx.z * per;
        KT = min(per, KT_all - kt0);
    }
    // Marlin: the workgroups that share a chunk (64 columns) are neighbours in the list of tiles, so that one L2 serves them
    const WaveTile tile = wave_tile(p.M, BM, p.by_rows);
    const int n0 = tile.col * BN, m0 = tile.row * BM, m_end = min(p.M, m0 + BM);
    const int chunk = n0 >> 6, sub = MARLIN ? tile.col & (4 / NT - 1) : 0;
    const int s_lo = wave * KT / NW, n = (wave + 1) * KT / NW - s_lo;

    uint8_t* const mine = lds + wave * STAGE;
    const uint32_t mine_addr = lds_base + (uint32_t)wave * STAGE;
    uint8_t* const tab = lds + NW * STAGE;                   // [group][column] fp16

    // ---- group scales of the tile, requested first (four per load)
    const int g_lo = (int)p.by_group((uint32_t)kt0), GR = (int)p.by_group((uint32_t)(kt0 + KT - 1)) - g_lo + 1;
    const int W = p.words, tab_n = MARLIN ? GR * 16 : BN * W;
    const WhTable range = wh_table((int64_t)(N - n0) * G);
    const uint8_t* const tabp = (const uint8_t*)p.b_s + (MARLIN ? ((int64_t)g_lo * N + chunk * 64) * 2 : (int64_t)n0 * G * 2 - range.back);
    const uint32_t tab_last = (uint32_t)min(range.last, (int64_t)0x7fffffff), tab_back = (uint32_t)range.back;
    auto tab_at = [&](int idx, int& col, int& w, int& shift) {
        if constexpr (MARLIN) {                              // col: unit of four scales, w: group
            w = min(idx >> 4, GR - 1);
            col = idx & 15;
            shift = 0;
            return (uint32_t)w * (uint32_t)(N * 2) + (uint32_t)col * 8u;
        } else {
            col = (int)p.by_words((uint32_t)idx);
            w = idx - col * W;
            const uint32_t want = ((uint32_t)min(min(col, BN - 1), N - 1 - n0) * (uint32_t)G + (uint32_t)(g_lo + 4 * w)) * 2u + tab_back;
            const uint32_t at = min(want, tab_last);
            shift = (int)(want - at) * 8;
            return at;
        }
    };
    auto tab_put = [&](int col, int w, int shift, uint64_t v) {
        if constexpr (MARLIN) {
            // scale 8 c + 2 j + b of a chunk belongs to column 16 j + 8 b + c
            const int c = col >> 1, j = 2 * (col & 1);
#pragma unroll
            for (int e = 0; e < 4; ++e) *(unsigned short*)(tab + w * TR + 2 * (16 * (j + (e >> 1)) + 8 * (e & 1) + c)) = (unsigned short)(v >> (16 * e));
        } else {
            v = shift < 64 ? v >> shift : 0;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (4 * w + e < GR) *(unsigned short*)(tab + (4 * w + e) * TR + 2 * col) = (unsigned short)(v >> (16 * e));
        }
    };
    int t_col, t_w, t_shift;
    v2i t_s;
    {
        const uint32_t at = tab_at(tid, t_col, t_w, t_shift);
        t_s = ring_load_b64<0>(at, ring_base(tabp));
    }

    // ---- source offsets.  16-byte chunk c of activation row R lies at chunk c ^ swizzle(R): 16 rows x one chunk (row-packed) and
    // 16 rows x four dwords of one chunk (Marlin) then fall into different banks.
    auto swizzle = [](int row) { return MARLIN ? (((row >> 1) & 3) * 2) | ((row >> 3) & 1) : ((row >> 1) & 7); };
    uint32_t aoff[2 * MT], boff[NB];
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) {
        const int row = 8 * i + (lane >> 3), sw = swizzle(row);
        aoff[i] = (uint32_t)min(row, m_end - 1 - m0) * (uint32_t)(K * 2) + (uint32_t)((lane & 7) ^ sw) * 16u;
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        if constexpr (MARLIN) {
            // strip 2 i + (lane >> 5) of the step: 512 contiguous bytes per chunk
            boff[i] = (uint32_t)(2 * i + (lane >> 5)) * (uint32_t)(nchunks * 512) + (uint32_t)(lane & 31) * 16u;
        } else {
            // 64 bytes of each of 16 rows
            const int row = 16 * i + (lane >> 2);
            boff[i] = (uint32_t)min(row, N - 1 - n0) * (uint32_t)(K >> 1) + (uint32_t)((lane & 3) ^ (((row >> 2) & 1) << 1)) * 16u;
        }
    }
    const uint8_t* const ga = p.a + (int64_t)m0 * K * 2;
    const uint8_t* const gb = p.b + (MARLIN ? (int64_t)chunk * 512 : (int64_t)n0 * (K >> 1));
    const int64_t b_step = MARLIN ? (int64_t)nchunks * 4096 : 64;
    auto issue_a = [&](int s, int h) __attribute__((always_inline)) {
        const uint8_t* src = ga + ((int64_t)(kt0 + min(s, KT - 1)) * 2 + h) * 128;
#pragma unroll
        for (int i = 0; i < 2 * MT; ++i) dma16(mine_addr + i * 1024u, aoff[i], src);
    };
    auto issue_b = [&](int s, int slot) __attribute__((always_inline)) {
        const uint8_t* src = gb + (int64_t)(kt0 + min(s, KT - 1)) * b_step;
#pragma unroll
        for (int i = 0; i < NB; ++i) dma16(mine_addr + OFF_B + (uint32_t)slot * WB + i * 1024u, boff[i], src);
    };
    auto issue_step = [&](int s) __attribute__((always_inline)) {
        issue_b(s, 0);
        const uint8_t* src = ga + (int64_t)(kt0 + min(s, KT - 1)) * 256;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < 2 * MT; ++i) dma16(mine_addr + (uint32_t)(h * wh_a(MT)) + i * 1024u, aoff[i], src + h * 128);
    };
    if constexpr (WHOLE) {
        issue_step(s_lo);
    } else {
        issue_b(s_lo, 0);
        issue_a(s_lo, 0);
        issue_b(s_lo + 1, 1);
    }

    ring_wait<WHOLE ? 4 * MT + NB : 2 * MT + 2 * NB>(t_s);
    if (tid < tab_n) tab_put(t_col, t_w, t_shift, __builtin_bit_cast(uint64_t, t_s));
    for (int idx = tid + NW * 64; idx < tab_n; idx += NW * 64) {
        int col, w, shift;
        const uint32_t at = tab_at(idx, col, w, shift);
        uint64_t v;
        __builtin_memcpy(&v, tabp + at, 8);
        tab_put(col, w, shift, v);
    }
    __syncthreads();

    // acc[mt][j][i] = C[row 16 mt + r][column 16 j + 4 g + i] over this wave's K steps
    v4f acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};

    // a[mt][f]: activation fragment of 32 of the half's 64 elements, in the order of the unpacked weights
    struct Half {
        v4i a[MT][2];
        // w[j][f] (row-packed): the word of columns 16 j + r, elements 16 g + 8 f .. + 7 of the half
        // w[st][j] (Marlin): word j of unit (c, g) of strip st of the half
        unsigned w[MARLIN ? 4 : NT][MARLIN ? NT : 2];
    };
    const int swz = swizzle(r);
    // half h of a step: activation rows at ast, words at bst
    auto fetch = [&](Half& half, int h, const uint8_t* ast, const uint8_t* bst) __attribute__((always_inline)) {
        auto &a = half.a;
        auto &w = half.w;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                const uint8_t* row = ast + mt * 2048 + r * 128;
                if constexpr (MARLIN) {
                    // strips 2 f, 2 f + 1 of 16 elements: elements 2 g, 2 g + 1, 2 g + 8, 2 g + 9 of each
#pragma unroll
                    for (int st = 0; st < 2; ++st) {
                        a[mt][f][2 * st] = *(const int*)(row + (((4 * f + 2 * st) ^ swz) * 16) + 4 * g);
                        a[mt][f][2 * st + 1] = *(const int*)(row + (((4 * f + 2 * st + 1) ^ swz) * 16) + 4 * g);
                    }
                } else {
                    a[mt][f] = *(const v4i*)(row + (((2 * g + f) ^ swz) * 16));
                }
            }
        if constexpr (MARLIN) {
#pragma unroll
            for (int st = 0; st < 4; ++st) {
                const uint8_t* u = bst + (4 * h + st) * 512 + (4 * (r & 7) + g) * 16 + sub * (4 * NT);
                if constexpr (NT == 4) {
                    const v4i x = *(const v4i*)u;
#pragma unroll
                    for (int j = 0; j < 4; ++j) w[st][j] = (unsigned)x[j];
                } else if constexpr (NT == 2) {
                    const v2i x = *(const v2i*)u;
                    w[st][0] = (unsigned)x[0];
                    w[st][1] = (unsigned)x[1];
                } else {
                    w[st][0] = *(const unsigned*)u;
                }
            }
        } else {
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const v2i x = *(const v2i*)(bst + (16 * j + r) * 64 + (((2 * h + (g >> 1)) ^ (((r >> 2) & 1) << 1)) * 16) + 8 * (g & 1));
                w[j][0] = (unsigned)x[0];
                w[j][1] = (unsigned)x[1];
            }
        }
    };
    auto lo8 = [](unsigned x) { return w4_as_u32(w4_as_h2((x & 0x000f000fu) | 0x64006400u) - (v2h){(_Float16)1032.f, (_Float16)1032.f}); };
    auto hi8 = [](unsigned x) {
        return w4_as_u32(w4_as_h2((x & 0x00f000f0u) | 0x64006400u) * (v2h){(_Float16)0.0625f, (_Float16)0.0625f} - (v2h){(_Float16)72.f, (_Float16)72.f});
    };
    auto mma = [](const v4i& x, const v4i& y, v4f c) {
        if constexpr (BF) return mfma_bf16_16x16x32(__builtin_bit_cast(v8bf, x), __builtin_bit_cast(v8bf, y), c);
        else return mfma_f16_16x16x32(__builtin_bit_cast(v8h, x), __builtin_bit_cast(v8h, y), c);
    };
    const int mshift = 8 * (r >> 3);
    auto compute = [&](Half& half, int s) __attribute__((always_inline)) {
        auto &a = half.a;
        auto &w = half.w;
        const uint8_t* tr = tab + ((int)p.by_group((uint32_t)(kt0 + s)) - g_lo) * TR + 2 * (MARLIN ? sub * BN : 0) + (PRE ? 2 * r : 8 * g);
        v4f init[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            init[mt] = (v4f){0.f, 0.f, 0.f, 0.f};
            if constexpr (!MARLIN && !(BF && PRE)) {
                // a word unpacks in the order 0, 4, 1, 5, 2, 6, 3, 7: the same for the activations
#pragma unroll
                for (int f = 0; f < 2; ++f) {
                    const v4i x = a[mt][f];
                    a[mt][f] = (v4i){(int)__builtin_amdgcn_perm((unsigned)x[2], (unsigned)x[0], 0x05040100u), (int)__builtin_amdgcn_perm((unsigned)x[2], (unsigned)x[0], 0x07060302u),
                                     (int)__builtin_amdgcn_perm((unsigned)x[3], (unsigned)x[1], 0x05040100u), (int)__builtin_amdgcn_perm((unsigned)x[3], (unsigned)x[1], 0x07060302u)};
                }
            }
            if constexpr (BF && !PRE) {
                // bf16: a nibble becomes 128 + q, exactly; the missing - 136 of every product is where the sums start
                const v4i c136 = {(int)0xc308c308u, (int)0xc308c308u, (int)0xc308c308u, (int)0xc308c308u};
                init[mt] = mma(c136, a[mt][0], init[mt]);
                init[mt] = mma(c136, a[mt][1], init[mt]);
            }
        }
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            if constexpr (BF && PRE) {
                const float sc = f16_to_f32(*(const unsigned short*)(tr + 32 * j));
                const v4i b0 = w4_word_to_bf16x8(w[j][0], sc), b1 = w4_word_to_bf16x8(w[j][1], sc);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    acc[mt][j] = mma(b0, a[mt][0], acc[mt][j]);
                    acc[mt][j] = mma(b1, a[mt][1], acc[mt][j]);
                }
                continue;
            }
            v4i b[2];
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                if constexpr (MARLIN) {
                    const unsigned u0 = w[2 * f][j] >> mshift, u1 = w[2 * f + 1][j] >> mshift;
                    b[f] = (v4i){(int)lo8(u0), (int)hi8(u0), (int)lo8(u1), (int)hi8(u1)};
                } else if constexpr (BF) {
                    const unsigned x = w[j][f];
                    b[f] = (v4i){(int)((x & 0x000f000fu) | 0x43004300u), (int)(((x >> 4) & 0x000f000fu) | 0x43004300u),
                                 (int)(((x >> 8) & 0x000f000fu) | 0x43004300u), (int)(((x >> 12) & 0x000f000fu) | 0x43004300u)};
                } else {
                    const unsigned x = w[j][f], x8 = x >> 8;
                    b[f] = (v4i){(int)lo8(x), (int)hi8(x), (int)lo8(x8), (int)hi8(x8)};
                }
            }
            if constexpr (PRE) {
                const _Float16 s1 = *(const _Float16*)(tr + 32 * j);
                const v2h s2 = {s1, s1};
#pragma unroll
                for (int f = 0; f < 2; ++f)
#pragma unroll
                    for (int i = 0; i < 4; ++i) b[f][i] = (int)w4_as_u32(w4_as_h2((unsigned)b[f][i]) * s2);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    acc[mt][j] = mma(b[0], a[mt][0], acc[mt][j]);
                    acc[mt][j] = mma(b[1], a[mt][1], acc[mt][j]);
                }
                continue;
            }
            const uint64_t sw = *(const uint64_t*)(tr + 32 * j);
            v4f sc;
#pragma unroll
            for (int i = 0; i < 4; ++i) sc[i] = f16_to_f32((unsigned short)(sw >> (16 * i)));
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                v4f t = mma(b[0], a[mt][0], init[mt]);
                t = mma(b[1], a[mt][1], t);
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[mt][j][i] = fmaf(t[i], sc[i], acc[mt][j][i]);
            }
        }
    };
    // the registers hold what they need of the stage: the next loads may overwrite it
    auto fetched = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_s_waitcnt(0xc07f);                  // lgkmcnt(0)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };

    if constexpr (WHOLE) {
        // everything of step s is in registers before step s + 1 is requested into its place
        Half h0, h1;
        for (int i = 0; i < n; ++i) {
            const int s = s_lo + i;
            wv_wait_loads<0>();
            fetch(h0, 0, mine, mine + OFF_B);
            fetch(h1, 1, mine + wh_a(MT), mine + OFF_B);
            fetched();
            if (i + 1 < n) issue_step(s + 1);
            __builtin_amdgcn_sched_barrier(0);
            compute(h0, s);
            compute(h1, s);
            __builtin_amdgcn_sched_barrier(0);
        }
    } else {
        // Step s: half 0 needs the activations requested last and the words requested a step before them; the words of step
        // s + 1, requested behind those activations, may stay in flight.  Half 1 needs activations requested behind them.
        int slot = 0;
        Half half;
        for (int i = 0; i < n; ++i) {
            const int s = s_lo + i;
            const bool more = i + 1 < n;
            if (more) wv_wait_loads<NB>();
            else wv_wait_loads<0>();
            fetch(half, 0, mine, mine + OFF_B + slot * WB);
            fetched();
            issue_a(s, 1);
            __builtin_amdgcn_sched_barrier(0);
            compute(half, s);
            __builtin_amdgcn_sched_barrier(0);
            wv_wait_loads<0>();
            fetch(half, 1, mine, mine + OFF_B + slot * WB);
            fetched();
            if (more) {
                issue_a(s + 1, 0);
                if (i + 2 < n) issue_b(s + 2, slot);
            }
            __builtin_amdgcn_sched_barrier(0);
            compute(half, s);
            __builtin_amdgcn_sched_barrier(0);
            slot ^= 1;
        }
    }
    wv_wait_loads<0>();
    __syncthreads();

    float* red = (float*)lds;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int j = 0; j < NT; ++j) *(v4f*)(red + (wave * BM + 16 * mt + r) * (BN + 4) + 16 * j + 4 * g) = acc[mt][j];
    __syncthreads();
    wv_store<NW, MT, NT>(p, red, n0, m0, m_end);
}

template <int KIND, int NW, int MT, int NT, bool PRE>
int launch_w4a16_wave(const DirectArgs& p, int z, hipStream_t stream, const char* name) {
    static std::atomic<uint64_t> configured{0};
    auto kern = w4a16_wave_kernel<KIND, NW, MT, NT, PRE>;
    const int KT_all = p.K >> 7, per = (KT_all + z - 1) / z, groups = wh_groups(p.K, p.group, per);
    const int bytes = wh_lds(KIND, NW, MT, NT, groups);
    if (bytes > D_LDS_MAX) LLMK_FAIL(LLMK_ERR_SHAPE, "%s: %d bytes of LDS needed", name, bytes);
    if (bytes > 64 * 1024)       // (less needs no leave, and asking for it costs a decode call 0.1 us)
        if (int rc = llmk_reserve_lds((const void*)kern, D_LDS_MAX, configured, name)) return rc;
    DirectArgs q = p;
    q.ksplit = z;
    const int zg = (KT_all + per - 1) / per, rows = (p.M + 16 * MT - 1) / (16 * MT);
    const unsigned tiles = (unsigned)(((p.N + 16 * NT - 1) / (16 * NT)) * rows);
    q.by_rows = fast_div((uint32_t)rows);
    q.by_group = fast_div((uint32_t)p.group >> 7);
    q.words = (groups + 3) >> 2;
    q.by_words = fast_div((uint32_t)q.words);
    kern<<<dim3(tiles, 1, (unsigned)zg), NW * 64, bytes, stream>>>(q);
    LLMK_CHECK_LAUNCH(name);
    if (z > 1) return wv_sum_slices(p, zg, stream, name);
    return LLMK_OK;
}

// ------------------------------------------------------------------------------------------------------------
// 8-bit operands [M, K] and [N, K]: fp8 or int8 with a scale per row and 128 elements and per 128 x 128 weight block (K_FP8_BLOCK,
// K_I8_BLOCK), or int8 with a scale per row and per column (K_I8_ROWCOL: int32 sums, scaled at the end).  S32 as above.
// What it replaces at 1 to 16 rows kept activations in registers and walked column tiles with one barrier each; its fragment
// loads (16 rows x 64 bytes an instruction) cost the address path four times what coalesced ones to LDS do.  Bound by weights
// from L2 or HBM up to 16 rows (28672 x 4096: 6.1 TB/s from the memory-side cache, 4.6 from HBM), by the address path and the latency of
// one stage from there.  us per launch, before | now, weights in the memory-side cache: fp8 4 x 4096 x 14336 15.3 | 11.1, 9 x 14336 x 4096 14.2 |
// 11.3, 12 x 28672 x 4096 22.9 | 18.7, 16 x 4096 x 4096 6.9 | 4.6, int8 15 x 6144 x 4096 8.7 | 5.1, per token 9 x 3128 x 9472 11.2 |
// 5.4; weights from HBM, fp8: 1 x 4096 x 4096 6.5 | 5.8, 16 x 4096 x 4096 7.0 | 6.7, 16 x 14336 x 4096 15.4 | 15.5, 9 x 28672 x 4096 25.4
// | 23.4, 16 x 28672 x 4096 25.9 | 25.9, 12 x 128256 x 4096 98 | 95, 1 x 4096 x 14336 16.0 | 12.4, int8 12 x 4096 x 14336 16.4 | 14.1; int8
// on short rows is slower than before: 1 x 4096 x 1536 4.0 | 4.3, 1 x 1144 x 1024 3.0 | 3.6 (a K step or two a wave, tables and a barrier in
// front; with the block scales in registers instead 3.7).
constexpr int w8_stage(int mt, int nt) { return (16 * mt + 16 * nt) * 128 + 256; }
constexpr int w8_lds(int nw, int mt, int nt, int d, int steps) {
    const int a = nw * d * w8_stage(mt, nt) + 4 * steps, b = wv_red(nw, mt, nt);
    return a > b ? a : b;
}

template <int KIND, int NW, int MT, int NT, int D, bool S32>
__global__ __launch_bounds__(NW * 64) void w8_wave_kernel(DirectArgs p) {
    constexpr bool SCALED = (KIND != K_I8_ROWCOL);
    static_assert(KIND == K_FP8_BLOCK || KIND == K_I8_BLOCK || KIND == K_I8_ROWCOL, "8-bit operands");
    constexpr int BM = 16 * MT, BN = 16 * NT, STAGE = w8_stage(MT, NT), LPS = 2 * MT + 2 * NT + (SCALED ? 1 : 0);
    constexpr int OFF_B = BM * 128, OFF_S = OFF_B + BN * 128;
    wv_arguments(p);
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int N = p.N, K = p.K, KT_all = K >> 7;
    int kt0 = 0, KT = KT_all;
    if constexpr (SCALED) {
        if (p.ksplit > 1) {
            const int per = (KT_all + p.ksplit - 1) / p.ksplit;
            kt0 = (int)blockIdx.z * per;
            KT = min(per, KT_all - kt0);
        }
    }
    const WaveTile tile = wave_tile(p.M, BM, p.by_rows);
    const int n0 = tile.col * BN, m0 = tile.row * BM, m_end = min(p.M, m0 + BM);
    const int s_lo = wave * KT / NW, n = (wave + 1) * KT / NW - s_lo;
    uint8_t* const mine = lds + wave * (D * STAGE);
    const uint32_t mine_addr = lds_base + (uint32_t)wave * (D * STAGE);
    float* const bsl = (float*)(lds + NW * D * STAGE);       // block scale of the tile's columns per K step

    const bool s_f16 = p.s_dtype == LLMK_F16;
    auto scale_f32 = [&](unsigned raw) { return S32 ? __uint_as_float(raw) : (s_f16 ? f16_to_f32((unsigned short)raw) : bf16_to_f32((unsigned short)raw)); };
    constexpr uint32_t ssz = S32 ? 4u : 2u;
    int t_bs = 0;
    if constexpr (SCALED) {
        const RingBase bsb = ring_base((const uint8_t*)p.b_s + ((int64_t)(n0 >> 7) * KT_all + kt0) * ssz);
        const uint32_t bat = (uint32_t)min(tid, KT - 1) * ssz;
        if constexpr (S32) t_bs = ring_load_b32<0>(bat, bsb);
        else t_bs = ring_load_u16<0>(bat, bsb);
    }

    // ---- source offsets of the loads of a stage; 16-byte chunks swizzled within a row as in the tile kernels
    uint32_t aoff[2 * MT], boff[2 * NT];
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) {
        const int row = 8 * i + (lane >> 3);
        aoff[i] = (uint32_t)min(row, m_end - 1 - m0) * (uint32_t)K + (uint32_t)((lane & 7) ^ ((row >> 1) & 7)) * 16u;
    }
#pragma unroll
    for (int i = 0; i < 2 * NT; ++i) {
        const int row = 8 * i + (lane >> 3);
        boff[i] = (uint32_t)min(row, N - 1 - n0) * (uint32_t)K + (uint32_t)((lane & 7) ^ ((row >> 1) & 7)) * 16u;
    }
    const uint32_t soff = (uint32_t)min(min(lane, BM - 1), m_end - 1 - m0) * (uint32_t)KT_all * ssz;
    const uint8_t* const ga = p.a + (int64_t)m0 * K;
    const uint8_t* const gb = p.b + (int64_t)n0 * K;
    const uint8_t* const gs = (const uint8_t*)p.a_s + (int64_t)m0 * KT_all * ssz;
    auto issue = [&](int slot, int s) __attribute__((always_inline)) {
        const int kb = kt0 + min(s, KT - 1);
        const uint32_t st = mine_addr + (uint32_t)slot * STAGE;
#pragma unroll
        for (int i = 0; i < 2 * NT; ++i) dma16(st + OFF_B + i * 1024u, boff[i], gb + (int64_t)kb * 128);
#pragma unroll
        for (int i = 0; i < 2 * MT; ++i) dma16(st + i * 1024u, aoff[i], ga + (int64_t)kb * 128);
        if constexpr (SCALED) {
            if constexpr (S32) dma4(st + OFF_S, soff, gs + (int64_t)kb * 4);
            else dma2(st + OFF_S, soff, gs + (int64_t)kb * 2);
        }
    };
#pragma unroll
    for (int d = 0; d < D; ++d) issue(d, s_lo + d);
    if constexpr (SCALED) {
        ring_wait<D * LPS>(t_bs);
        if (tid < KT) bsl[tid] = scale_f32((unsigned)t_bs);
        for (int k = tid + NW * 64; k < KT; k += NW * 64) bsl[k] = ld_scale(p.b_s, (int64_t)(n0 >> 7) * KT_all + kt0 + k, p.s_dtype);
        __syncthreads();
    }

    // acc[mt][j][i] = C[row 16 mt + r][column 16 j + 4 g + i] over this wave's K steps (K_I8_ROWCOL: int32 bits)
    v4f acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};
    const int swz = (r >> 1) & 7;
    const int lo = r * 128 + ((g ^ swz) * 16), hi = r * 128 + (((g + 4) ^ swz) * 16);
    auto ldfrag = [&](const uint8_t* base) {
        const v4i x = *(const v4i*)(base + lo), y = *(const v4i*)(base + hi);
        return (v8i){x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
    };
    v8i af[MT], bf[NT];
    unsigned a_sc[MT];
    auto fetch = [&](int slot) __attribute__((always_inline)) {
        const uint8_t* st = mine + slot * STAGE;
#pragma unroll
        for (int j = 0; j < NT; ++j) bf[j] = ldfrag(st + OFF_B + j * 2048);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            af[mt] = ldfrag(st + mt * 2048);
            if constexpr (SCALED) a_sc[mt] = *(const unsigned*)(st + OFF_S + (16 * mt + r) * 4);
        }
    };
    auto compute = [&](int s) __attribute__((always_inline)) {
        if constexpr (SCALED) {
            const float bs = bsl[s];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const float sa = scale_f32(a_sc[mt]) * bs;
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    const v4f t = raw_f32<KIND>(step_raw<KIND>(bf[j], af[mt]));
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[mt][j][i] = fmaf(t[i], sa, acc[mt][j][i]);
                }
            }
        } else {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[mt][j] = mma_plain<KIND>(bf[j], af[mt], acc[mt][j]);
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

    float* red = (float*)lds;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int j = 0; j < NT; ++j) *(v4f*)(red + (wave * BM + 16 * mt + r) * (BN + 4) + 16 * j + 4 * g) = acc[mt][j];
    __syncthreads();
    wv_store<NW, MT, NT, KIND == K_I8_ROWCOL>(p, red, n0, m0, m_end);
}

template <int KIND, int NW, int MT, int NT, int D, bool S32>
int launch_w8_wave(const DirectArgs& p, hipStream_t stream, const char* name) {
    static std::atomic<uint64_t> configured{0};
    auto kern = w8_wave_kernel<KIND, NW, MT, NT, D, S32>;
    const int z = p.ksplit > 1 ? p.ksplit : 1;
    const int bytes = w8_lds(NW, MT, NT, D, ((p.K >> 7) + z - 1) / z);
    if (bytes > D_LDS_MAX) LLMK_FAIL(LLMK_ERR_SHAPE, "%s: %d bytes of LDS needed", name, bytes);
    if (bytes > 64 * 1024)       // (less needs no leave, and asking for it costs a decode call 0.1 us)
        if (int rc = llmk_reserve_lds((const void*)kern, D_LDS_MAX, configured, name)) return rc;
    const int rows = (p.M + 16 * MT - 1) / (16 * MT);
    const unsigned tiles = (unsigned)(((p.N + 16 * NT - 1) / (16 * NT)) * rows);
    DirectArgs q = p;
    q.by_rows = fast_div((uint32_t)rows);
    kern<<<dim3(tiles, 1, (unsigned)z), NW * 64, bytes, stream>>>(q);
    LLMK_CHECK_LAUNCH(name);
    return z > 1 ? wv_sum_slices(p, z, stream, name) : LLMK_OK;
}

// Launch shape: waves per workgroup, row and column tiles of a wave, K slices over workgroups, estimated microseconds.
struct WavePlan {
    int nw, mt, nt, z;
    double cost;
};

inline int wave_shape(const WavePlan& w, int form, int32_t* shape) {
    const int32_t v[5] = {w.nw, w.mt, w.nt, w.z, form};
    for (int i = 0; i < 5; ++i) shape[i] = v[i];
    return 1;
}

// Estimated microseconds of a launch without its K slices' sums.  Eight waves: base + rounds of 256 workgroups x (fixed + K steps
// of a wave x step).  Four waves (64 columns): several workgroups share a CU and cover each other's prologue and reduction, so
// their rounds count in fractions; slower on a single round (w4a8 64 x 14336 x 4096 18.2 against 17.0 us), faster from two on
// (64 x 28672 x 4096 27.6 against 30.2, 128 rows 46.8 against 54).  The numbers are a fit (5 to 8 % rms) to 100 to 180 shapes of M
// 1 to 520, N 1024 to 28672, K 1024 to 14336 a kind, every tile shape timed; [mt - 1][log2 nt], and [mt - 1] for four waves (0:
// shape not built).  They are of the kernels with a division in front of the loads and half steps on 16-row tiles.  On the present ones the tile that they
// choose takes, against the fastest one that is built (45 random shapes of 1 to 300 rows a kind, all tiles timed, mean of cached weights and weights from HBM),
// fp8 1.016 of its time, int8 and per token 1.010, w4a8 1.006, row-packed bf16 1.009, fp16 1.028, Marlin words 1.009.
struct WaveModel {
    float base8[4][3], fixed8[4][3], step8[4][3], base4[4], step4[4];
};
constexpr WaveModel WV_W4A8 = {{{3.78f, 3.77f, 3.94f}, {3.69f, 3.84f, 3.81f}, {4.04f, 3.99f, 1.38f}, {3.85f, 1.75f, 1.46f}},
                               {{0.10f, 0.00f, 0.00f}, {0.29f, 0.33f, 0.54f}, {0.00f, 0.39f, 3.16f}, {0.00f, 2.52f, 3.59f}},
                               {{0.45f, 0.73f, 1.16f}, {0.52f, 0.78f, 1.39f}, {0.70f, 0.97f, 1.71f}, {0.88f, 1.22f, 1.97f}},
                               {0.f, 0.f, 6.03f, 5.54f}, {0.f, 0.f, 1.06f, 1.28f}};
constexpr WaveModel WV_NK = {{{4.12f, 4.10f, 1.50f}, {3.89f, 3.63f, 1.48f}, {3.60f, 1.76f, 1.38f}, {2.14f, 1.85f, 1.60f}},
                             {{0.05f, 0.00f, 2.17f}, {0.05f, 0.36f, 2.65f}, {0.23f, 2.21f, 3.03f}, {1.75f, 1.91f, 2.86f}},
                             {{0.48f, 0.76f, 1.52f}, {0.72f, 1.03f, 1.85f}, {0.98f, 1.38f, 2.22f}, {1.27f, 1.75f, 2.68f}},
                             {5.42f, 4.67f, 4.98f, 0.f}, {0.80f, 1.17f, 1.49f, 0.f}};
constexpr WaveModel WV_NKB = {{{4.29f, 4.16f, 1.27f}, {4.05f, 3.52f, 0.87f}, {3.98f, 1.53f, 0.87f}, {1.65f, 1.31f, 1.29f}},
                              {{0.02f, 0.00f, 2.40f}, {0.00f, 0.27f, 3.23f}, {0.00f, 2.42f, 3.72f}, {2.45f, 3.05f, 3.77f}},
                              {{0.46f, 0.73f, 1.37f}, {0.74f, 1.05f, 1.70f}, {1.00f, 1.32f, 2.03f}, {1.21f, 1.55f, 2.51f}},
                              {4.12f, 3.88f, 4.64f, 0.f}, {0.90f, 1.21f, 1.52f, 0.f}};
constexpr WaveModel WV_NKB_PRE = {{{4.27f, 4.14f, 1.97f}, {3.67f, 4.35f, 1.77f}, {3.53f, 1.94f, 1.41f}, {2.02f, 1.92f, 1.23f}},
                                  {{0.23f, 0.00f, 1.85f}, {0.20f, 0.03f, 2.63f}, {0.21f, 2.07f, 3.39f}, {1.65f, 2.38f, 3.92f}},
                                  {{0.47f, 0.99f, 2.20f}, {0.71f, 1.18f, 2.36f}, {0.95f, 1.50f, 2.52f}, {1.26f, 1.66f, 2.74f}},
                                  {5.60f, 6.28f, 5.30f, 0.f}, {1.06f, 1.28f, 1.62f, 0.f}};
constexpr WaveModel WV_MARLIN = {{{1.94f, 1.67f, 1.52f}, {1.76f, 1.81f, 1.64f}, {2.06f, 1.78f, 1.59f}, {2.22f, 1.84f, 1.41f}},
                                 {{1.51f, 1.93f, 2.15f}, {1.76f, 2.14f, 2.51f}, {1.77f, 2.36f, 3.02f}, {1.89f, 2.46f, 3.45f}},
                                 {{0.82f, 1.04f, 1.44f}, {1.05f, 1.28f, 1.79f}, {1.31f, 1.61f, 2.12f}, {1.54f, 1.88f, 2.53f}},
                                 {4.60f, 5.15f, 5.21f, 0.f}, {0.84f, 1.15f, 1.50f, 0.f}};
// Shapes of the 16-bit kernels that are built: all but those that were the cheapest for one in all of 9 million calls of 1 to 512
// rows, N 8 to 300000 and K 128 to 153600.
template <int KIND, bool PRE>
constexpr bool wh_built(int nw, int mt, int nt) {
    if (nw == 4) return nt == 4 && mt < 4 && !(KIND == K_W4NKB && PRE && mt == 1);
    if (KIND == K_W4MARLIN) return mt < 4 || nt == 4;
    if (KIND == K_W4NKB && PRE) return mt > 1 || nt == 1;
    return PRE || !((mt == 4 && nt == 1) || (KIND == K_W4NK && mt == 1 && nt == 4));
}
template <int KIND, bool PRE>
constexpr const WaveModel& wave_model() {
    if constexpr (KIND == K_W4MARLIN) return WV_MARLIN;
    else if constexpr (KIND == K_W4NK) return WV_NK;             // (PRE or not)
    else if constexpr (PRE) return WV_NKB_PRE;
    else return WV_NKB;
}

// A launch has fewer than 2^32 threads.
constexpr bool wv_grid_ok(int64_t tiles, int nw) { return tiles * nw * 64 <= 0xffffffffll; }

// The cheapest shape whose LDS (bytes(nw, mt, nt, K steps of a workgroup)) and scratch fit; K slices cost a second launch and
// their fp32 sums.
template <class Bytes>
inline bool wave_plan(int64_t M, int64_t N, int64_t K, int64_t scratch, const WaveModel& m, Bytes bytes, WavePlan& best) {
    const int KT = (int)(K >> 7), zmin = (KT + WV_MAX_STEPS - 1) / WV_MAX_STEPS, zmax = zmin > 4 ? zmin : 4;
    const double us_sum = (double)(M * N) * 8.0 / 6e6;
    int64_t ct[3];
    for (int j = 0; j < 3; ++j) ct[j] = (N + (16 << j) - 1) >> (4 + j);
    bool found = false;
    for (int z = zmin; z <= zmax; z *= 2) {
        const int per = (KT + z - 1) / z, steps8 = (per + 7) >> 3, steps4 = (per + 3) >> 2;
        if (z > 1 && ((z > zmin && per < 8) || scratch < z * M * N * 4)) continue;
        for (int mt = 1; mt <= 4 && (mt == 1 || M > 16 * (mt - 1)); ++mt) {
            const int64_t rt = (M + 16 * mt - 1) / (16 * mt);
            for (int j = 0; j < 3; ++j) {
                const int64_t wgs = ct[j] * rt * z;
                if (z > zmin && wgs > LLMK_CUS + LLMK_CUS / 4) continue;
                for (int nw = 8; nw >= 4; nw -= 4) {
                    if (nw == 4 && (j < 2 || m.step4[mt - 1] == 0.f)) continue;
                    double cost;
                    if (nw == 8) cost = m.base8[mt - 1][j] + (double)((wgs + LLMK_CUS - 1) / LLMK_CUS) * (m.fixed8[mt - 1][j] + steps8 * m.step8[mt - 1][j]);
                    else cost = m.base4[mt - 1] + (wgs > LLMK_CUS ? (double)wgs / LLMK_CUS : 1.0) * steps4 * m.step4[mt - 1];
                    if (z > 1) cost += 3.0 + z * us_sum;
                    if ((found && cost >= best.cost) || bytes(nw, mt, 1 << j, per) > D_LDS_MAX || !wv_grid_ok(ct[j] * rt, nw)) continue;
                    best = WavePlan{nw, mt, 1 << j, z, cost};
                    found = true;
                }
            }
        }
    }
    return found;
}
// 8-bit operands: an estimate of at least the weights at 6.1 TB/s, and K slices (a second launch and a write and a read of the
// planes) only of block-scaled operands beyond 128 K steps, where few columns leave the chip idle: below they never won (fp8, us, whole
// | sliced: 16 x 1024 x 32768 17.1 | 10.0, 20 x 136 x 65664 21.2 | 7.6).
constexpr WaveModel WV_FP8 = {{{2.97f, 2.81f, 1.50f}, {2.68f, 2.71f, 1.46f}, {0.f, 1.67f, 1.34f}, {0.f, 1.56f, 1.38f}},
                              {{0.00f, 0.00f, 1.10f}, {0.00f, 0.00f, 1.16f}, {0.f, 0.96f, 1.48f}, {0.f, 0.84f, 1.76f}},
                              {{0.34f, 0.53f, 0.93f}, {0.55f, 0.85f, 1.21f}, {0.f, 1.04f, 1.46f}, {0.f, 1.31f, 1.73f}},
                              {0.f, 3.66f, 5.20f, 4.97f}, {0.f, 0.57f, 0.72f, 0.88f}};
constexpr WaveModel WV_I8 = {{{2.95f, 2.89f, 1.54f}, {3.03f, 2.96f, 1.47f}, {0.f, 1.84f, 1.44f}, {0.f, 1.81f, 1.28f}},
                             {{0.03f, 0.03f, 1.30f}, {0.00f, 0.01f, 1.57f}, {0.f, 1.20f, 1.99f}, {0.f, 1.37f, 2.53f}},
                             {{0.34f, 0.50f, 0.87f}, {0.51f, 0.73f, 1.13f}, {0.f, 0.97f, 1.39f}, {0.f, 1.19f, 1.63f}},
                             {0.f, 3.73f, 5.00f, 4.60f}, {0.f, 0.56f, 0.73f, 0.88f}};
constexpr WaveModel WV_I8_ROWCOL = {{{2.86f, 2.76f, 1.56f}, {2.90f, 2.76f, 1.28f}, {0.f, 1.65f, 1.10f}, {0.f, 1.55f, 0.95f}},
                                    {{0.00f, 0.08f, 1.26f}, {0.06f, 0.12f, 1.83f}, {0.f, 1.39f, 2.46f}, {0.f, 1.54f, 3.11f}},
                                    {{0.32f, 0.47f, 0.83f}, {0.45f, 0.65f, 1.02f}, {0.f, 0.80f, 1.20f}, {0.f, 0.96f, 1.38f}},
                                    {0.f, 3.20f, 5.00f, 4.05f}, {0.f, 0.54f, 0.67f, 0.79f}};
// Stages of a wave: two for 16 x 16 tiles where every wave has many K steps, and, on at most one workgroup a CU, where some wave has a
// second one: nothing else covers the latency of its weights there, while from two workgroups a CU on the loads of one cover the other's
// (us, weights from HBM, one | two stages: fp8 1 x 4096 x 4096 6.4 | 5.9, 1 x 2616 x 4096 6.0 | 5.3, int8 1 x 2408 x 3072 5.2 | 4.7, 1 x 4096 x
// 5120 7.4 | 6.7, but 1 x 6144 x 4096 7.6 | 8.1, 1 x 14336 x 4096 13.1 | 14.1).  From 9 rows on for weights below 16 MB only: more of
// them at once do not come faster behind a cache full of dirty lines (fp8 16 x 4096 x 4096 8.5 | 8.7, 16 x 2048 x 4096 7.35 | 7.15, 16 x 4096 x 2048
// 6.4 | 6.1).
constexpr int w8_depth(int mt, int nt, int steps, int64_t wgs, bool few) {
    return mt == 1 && nt == 1 && (steps >= 48 || (steps > 8 && wgs <= LLMK_CUS && few)) ? 2 : 1;
}
constexpr bool w8_few(int64_t M, int64_t N, int64_t K) { return M <= 8 || N * K < (16 << 20); }
template <int KIND>
inline bool w8_wave_plan(int64_t M, int64_t N, int64_t K, int64_t scratch, WavePlan& best) {
    constexpr const WaveModel& m = KIND == K_FP8_BLOCK ? WV_FP8 : (KIND == K_I8_BLOCK ? WV_I8 : WV_I8_ROWCOL);
    if (K < 128 || K > (1 << 22)) return false;
    const int KT_all = (int)(K >> 7);
    const int zmax = KIND == K_I8_ROWCOL || KT_all <= 128 ? 1 : 16;
    bool found = false;
    for (int z = 1; z <= zmax && (z == 1 || z * M * N * 4 <= scratch); ++z) {
        const int KT = (KT_all + z - 1) / z, steps8 = (KT + 7) >> 3, steps4 = (KT + 3) >> 2;
        if ((z - 1) * KT >= KT_all) continue;                // an empty slice
        const double slices = z == 1 ? 0.0 : 4.5 + (double)(z * M * N) / 1.0e6;
        for (int mt = 1; mt <= 4 && (mt == 1 || M > 16 * (mt - 1)); ++mt) {
            const int64_t rt = (M + 16 * mt - 1) / (16 * mt);
            for (int j = mt > 2; j < 3; ++j) {               // (16 columns with more than 32 rows: never the cheapest)
                const int64_t tiles = ((N + (16 << j) - 1) >> (4 + j)) * rt, rounds = (tiles * z + LLMK_CUS - 1) / LLMK_CUS;
                for (int nw = 8; nw >= 4; nw -= 4) {
                    if (nw == 4 && (j < 2 || m.step4[mt - 1] == 0.f)) continue;
                    const double cost = slices + (nw == 8 ? m.base8[mt - 1][j] + (double)rounds * (m.fixed8[mt - 1][j] + steps8 * m.step8[mt - 1][j])
                                                          : m.base4[mt - 1] + (double)rounds * steps4 * m.step4[mt - 1]);
                    if ((found && cost >= best.cost) || w8_lds(nw, mt, 1 << j, w8_depth(mt, 1 << j, KT, tiles * z, w8_few(M, N, K)), KT) > D_LDS_MAX || !wv_grid_ok(tiles, nw)) continue;
                    best = WavePlan{nw, mt, 1 << j, z, cost};
                    found = true;
                }
            }
        }
    }
    const double weights = 2.0 + (double)(N * K) / 6.1e6;
    if (found && best.cost < weights) {
        // Bound by the weights: tiles of 16 columns, four workgroups a CU, keep HBM busiest up to 8 rows, with K from 4096 on up to 12; beyond,
        // where activations and the tiles' ends weigh more, tiles of 32 columns where those make 2.5 workgroups a CU (us, weights from HBM, 16 | 32 columns: fp8 9 x
        // 28672 x 4096 23.6 | 24.8, 12 x 28672 x 4096 24.5 | 25.5, 10 x 24000 x 2304 13.4 | 12.5, 16 x 18000 x 4096 18.9 | 19.7, 14 x 20000 x 4096 19.1 | 20.0, 16 x 22000 x
        // 4096 22.8 | 21.5, 16 x 24576 x 4096 23.3 | 21.9, 16 x 28672 x 4096 26.3 | 26.1, 16 x 32000 x 6144 44.0 | 39.0, 16 x 57344 x 4096
        // 49.2 | 45.2, 16 x 128256 x 4096 104 | 95; weights in the cache 16 x 28672 x 4096 18.7 | 19.2; 64 columns: 1 x 28672 x 4096 32.2
        // against 29.8 with 16).
        const int j = M <= 8 || (M <= 12 && KT_all >= 32) || N < 80 * LLMK_CUS ? 0 : 1;
        const int64_t tiles = (N + (16 << j) - 1) >> (4 + j);
        const double narrow = m.base8[0][j] + (double)((tiles + LLMK_CUS - 1) / LLMK_CUS) * (m.fixed8[0][j] + ((KT_all + 7) >> 3) * m.step8[0][j]);
        const int d = w8_depth(1, 1 << j, KT_all, tiles, w8_few(M, N, K));
        if (M <= 16 && best.z == 1 && narrow <= weights && w8_lds(8, 1, 1 << j, d, KT_all) <= D_LDS_MAX && wv_grid_ok(tiles, 8)) best = WavePlan{8, 1, 1 << j, 1, weights};
        best.cost = weights;
    }
    return found;
}
inline int w8_depth(const WavePlan& w, int64_t M, int64_t N, int64_t K) {
    const int64_t tiles = ((N + 16 * w.nt - 1) / (16 * w.nt)) * ((M + 16 * w.mt - 1) / (16 * w.mt));
    return w8_depth(w.mt, w.nt, (int)(((K >> 7) + w.z - 1) / w.z), tiles * w.z, w8_few(M, N, K));
}
template <int KIND>
inline int launch_w8_wave_plan(DirectArgs p, const WavePlan& w, void* scratch, hipStream_t stream, const char* name) {
    if (w.z > 1) {
        p.partial = (float*)scratch;
        p.ksplit = w.z;
    }
    auto run = [&](auto nw, auto mt, auto nt, auto d) {
        constexpr int NW = decltype(nw)::value, MT = decltype(mt)::value, NT = decltype(nt)::value, D = decltype(d)::value;
        if constexpr (KIND == K_I8_BLOCK) {
            if (p.s_dtype != LLMK_F32) return launch_w8_wave<KIND, NW, MT, NT, D, false>(p, stream, name);
        }
        return launch_w8_wave<KIND, NW, MT, NT, D, true>(p, stream, name);
    };
    const std::integral_constant<int, 1> i1;
    const std::integral_constant<int, 2> i2;
    const std::integral_constant<int, 3> i3;
    const std::integral_constant<int, 4> i4;
    const std::integral_constant<int, 8> i8;
    auto rows = [&](auto mt) {
        if constexpr (decltype(mt)::value > 1) {
            if (w.nw == 4) return run(i4, mt, i4, i1);
        } else {
            if (w8_depth(w, p.M, p.N, p.K) == 2) return run(i8, mt, i1, i2);
        }
        if constexpr (decltype(mt)::value <= 2) {
            if (w.nt == 1) return run(i8, mt, i1, i1);
        }
        return w.nt == 4 ? run(i8, mt, i4, i1) : run(i8, mt, i2, i1);
    };
    return w.mt == 1 ? rows(i1) : (w.mt == 2 ? rows(i2) : (w.mt == 3 ? rows(i3) : rows(i4)));
}

inline bool w4a8_wave_plan(int64_t M, int64_t N, int64_t K, int64_t scratch, WavePlan& best) {
    return wave_plan(M, N, K, scratch, WV_W4A8, [](int nw, int mt, int nt, int per) { return wv_lds(nw, mt, nt, wv_depth(mt, nt, per), per); }, best);
}
// 16-bit activations: groups in whole K steps, a scale table of at least one load, and Marlin words whose eight strips of a K step, and
// scales whose groups, lie within 32-bit offsets (strips are 8 N bytes apart, groups 2 N).
template <int KIND, bool PRE>
inline bool w4a16_wave_plan(int64_t M, int64_t N, int64_t K, int group, int64_t scratch, WavePlan& best) {
    if (K % 128 || group % 128 || N * (K / group) < 4 || K > (1 << 24) || N * (K / 2) >= (1ll << 40)) return false;
    if (wh_marlin(KIND) && N * std::max<int64_t>(64, 2 * (K / group)) > 0xffffffffll) return false;
    return wave_plan(M, N, K, scratch, wave_model<KIND, PRE>(), [&](int nw, int mt, int nt, int per) {
        return wh_built<KIND, PRE>(nw, mt, nt) ? wh_lds(KIND, nw, mt, nt, wh_groups((int)K, group, per)) : D_LDS_MAX + 1;
    }, best);
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

template <int KIND, bool PRE>
inline int launch_w4a16_wave_plan(const DirectArgs& p, const WavePlan& w, hipStream_t stream, const char* name) {
    auto rows = [&](auto mt) {
        constexpr int MT = decltype(mt)::value;
        if constexpr (wh_built<KIND, PRE>(4, MT, 4)) {
            if (w.nw == 4) return launch_w4a16_wave<KIND, 4, MT, 4, PRE>(p, w.z, stream, name);
        }
        if constexpr (wh_built<KIND, PRE>(8, MT, 1)) {
            if (w.nt == 1) return launch_w4a16_wave<KIND, 8, MT, 1, PRE>(p, w.z, stream, name);
        }
        if constexpr (wh_built<KIND, PRE>(8, MT, 2)) {
            if (w.nt == 2) return launch_w4a16_wave<KIND, 8, MT, 2, PRE>(p, w.z, stream, name);
        }
        if constexpr (wh_built<KIND, PRE>(8, MT, 4)) {
            if (w.nt == 4) return launch_w4a16_wave<KIND, 8, MT, 4, PRE>(p, w.z, stream, name);
        }
        LLMK_FAIL(LLMK_ERR_ARG, "%s: no such tile", name);
    };
    const std::integral_constant<int, 1> i1;
    const std::integral_constant<int, 2> i2;
    const std::integral_constant<int, 3> i3;
    const std::integral_constant<int, 4> i4;
    return w.mt == 1 ? rows(i1) : (w.mt == 2 ? rows(i2) : (w.mt == 3 ? rows(i3) : rows(i4)));
}

}  // namespace llmk

// Tile kernel for problems of about one round of 32 MI x 128 tiles: two groups of four waves (one wave of each group per SIMD) take
// turns.  K goes by in sub-blocks of 128 bytes; group p multiplies the sub-blocks u with u mod 2 == p, each wave a 16 MI x 64 share of
// the tile.  In phase u group u mod 2 requests sub-block u + 3, fetches the fragments of sub-block u from LDS and (4-bit weights)
// expands the weight rows of sub-block u + 1, while the other group does nothing but multiply sub-block u - 1 from registers; one
// barrier ends the phase.  The two sums of an output meet in LDS at the end.
//
// K_W4A8: 1024 x 4096 x 4096 30.8 us in one launch, 36.7 as expansion pass and the int8 kernel (37.7 | 33.4 with the quantiser).
//
// What bounds it: the CU's path from L2 (the 32 KB of a phase of a 128 x 128 tile take 0.31 us, its products 0.25) and the start and end of
// every phase.  Against the eight waves of gemm_dma_kernel, which share one 128-byte step: a wave tile is 64 x 64 instead of 32 x 64
// (fragments of 16 KB instead of 24 for the same products), only waves that have nothing to multiply wait for the address path, and a
// workgroup can be any multiple of 32 rows high, which is worth most where a few rows over a tile height would start another round.
#pragma once
#include <algorithm>

#include "gemm_mid.hpp"

namespace llmk {

constexpr int DU_BN = 128, DU_THREADS = 512, DU_SLOTS = 4;
// 4-bit weights: activations in four slots, expanded weight rows in two; otherwise both operands of a sub-block in one slot
constexpr int du_a(int mi) { return 32 * mi * 128; }
constexpr int du_b() { return DU_BN * 128; }
constexpr int du_windows(int mi) { return 2 * 32 * mi * 4 * 4; }             // two windows of activation scales, four sub-blocks each
constexpr bool du_scaled(int kind) { return kind == K_FP8_BLOCK || kind == K_I8_BLOCK || kind == K_W4A8; }
constexpr bool du_w4a16(int kind) { return is_w4nk(kind) || kind == K_W4MARLIN; }
constexpr bool du_expands(int kind) { return du_w4a16(kind) || kind == K_W4A8; }
// 160 rows of block-scaled operands: the registers just suffice, see the end of the main loop.  (us, cached weights | from HBM, without this tile ->
// with it: fp8 145 x 25320 x 6528 45.7 | 60.1 -> 35.4 | 49.2, 918 x 4224 x 6528 42.9 | 51.2 -> 31.9 | 39.2, 1194 x 4096 x 14336 80 | 90 -> 69 | 78, int8 157 x
// 28672 x 4096 37.9 | 43.2 -> 28.7 | 37.0, 287 x 14336 x 4096 31.9 | 42.4 -> 26.1 | 29.8, 1262 x 4096 x 4096 35.7 | 34.7 -> 29.2 | 29.1)
constexpr bool du_tight(int kind, int mi) { return du_scaled(kind) && !du_expands(kind) && mi > 4; }
constexpr int du_lds(int kind, int mi) {                                      // K_W4A8: + du_table bytes
    return DU_SLOTS * du_a(mi) + (du_expands(kind) ? 2 : DU_SLOTS) * du_b() + (du_scaled(kind) ? du_windows(mi) + D_MAX_KT * 4 : 0);
}
constexpr int du_table(int sub_blocks) { return sub_blocks * DU_BN * 4; }     // second-level scales and zero points, see below

// An offset in a register of its own: the compiler multiplies and adds in 64 bits and then keeps both halves for as long as the lower one is used.
__device__ __forceinline__ uint32_t only32(uint32_t x) {
    uint32_t y;
    asm("v_mov_b32 %0, %1" : "=v"(y) : "v"(x));
    return y;
}

template <int KIND, int MI, int SDT = LLMK_F32, bool GROUPED = false>
__global__ __launch_bounds__(DU_THREADS) void gemm_duo_kernel(DirectArgs p) {
    static_assert(!GROUPED || KIND == K_FP8_BLOCK || KIND == K_I8_BLOCK, "grouped products: block-scaled 8-bit operands");
    constexpr bool AS16 = SDT != LLMK_F32;
    constexpr bool SCALED = du_scaled(KIND), ROWCOL = (KIND == K_I8_ROWCOL), W4A16 = du_w4a16(KIND), MARLIN = (KIND == K_W4MARLIN), W4A8 = (KIND == K_W4A8),
                   EXPANDS = W4A16 || W4A8;
    static_assert(SCALED || ROWCOL || W4A16, "8-bit operands, or 4-bit weights");
    constexpr int MATH = W4A8 ? K_I8_BLOCK : KIND;           // the products once the weights are expanded
    constexpr int ESZ = is_half(KIND) ? 2 : 1, BM = 32 * MI, WR = 16 * MI;
    constexpr int A_SLOT = du_a(MI), B_SLOT = du_b(), B0 = DU_SLOTS * A_SLOT, NB = EXPANDS ? 2 : DU_SLOTS, SW = B0 + NB * B_SLOT;
    constexpr bool TIGHT = du_tight(KIND, MI);
    constexpr int LP = MI + (W4A8 ? 2 : 4);                  // loads of a wave from one of its turns to the end of the next
    constexpr int NSW = (2 * MI + 7) / 8;                    // scale loads per wave and window (16 rows x 4 sub-blocks each)
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4, w4 = wave & 3;
    const int wm = (wave >> 1) & 1, wn = wave & 1;
    const int N = p.N;
    const int K = p.K * ESZ;                                 // row length in bytes
    const int KT_all = K >> 7;
    int kt0 = 0, KT = KT_all;                                // sub-blocks [kt0, kt0 + KT) of this workgroup
    if (!GROUPED && p.ksplit > 1) {
        const int per = (KT_all + p.ksplit - 1) / p.ksplit;
        kt0 = (int)blockIdx.z * per;
        KT = max(0, min(per, KT_all - kt0));
    }
    int tile_n = (int)blockIdx.x, tile_m = 0, m_start, m_end;
    const uint8_t* bbase = p.b;
    int64_t bs_off = 0;                                      // block scales in front of this expert's
    if constexpr (GROUPED) {
        const SegmentTile sg = segment_of(p.seg_indptr, p.E, BM, 1, (int)blockIdx.y);
        if (!sg.found) return;
        m_start = sg.s0 + sg.rest * BM;
        m_end = min(sg.s1, m_start + BM);
        const int64_t widx = p.weight_indices ? p.weight_indices[sg.e] : sg.e;
        bbase += widx * (int64_t)N * K;
        bs_off = widx * (int64_t)((N + 127) / 128) * KT_all;
    } else {
        xcd_tile((int)blockIdx.y * (int)gridDim.x + (int)blockIdx.x, (int)gridDim.x, (int)gridDim.y, tile_n, tile_m);
        m_start = tile_m * BM;
        m_end = min(p.M, m_start + BM);
    }
    const int n0 = tile_n * DU_BN;
    float* const bsl = (float*)(lds + SW + du_windows(MI));

    // ---- source offsets (bytes, 32 bit).  A piece = 8 rows x 128 bytes = one load instruction; chunks XOR-swizzled with (row >> 1) & 7
    // as everywhere.  Weight rows are permuted inside each 64 so that a lane ends up with two runs of 8 consecutive columns.
    auto column = [](int R) { const int rho = R & 63; return (R & 64) + 32 * (rho >> 5) + 8 * ((rho & 15) >> 2) + 4 * ((rho >> 4) & 1) + (rho & 3); };
    auto a_offset = [&](int i, int l) {
        const int R = 8 * (w4 * MI + i) + (l >> 3);
        const uint32_t off = (uint32_t)min(m_start + R, m_end - 1) * (uint32_t)K + (uint32_t)((l & 7) ^ ((R >> 1) & 7)) * 16u;
        return TIGHT ? only32(off) : off;
    };
    auto b_offset = [&](int i, int l) {
        const int R = 8 * (w4 * 4 + i) + (l >> 3);
        const uint32_t off = (uint32_t)min(n0 + column(R), N - 1) * (uint32_t)K + (uint32_t)((l & 7) ^ ((R >> 1) & 7)) * 16u;
        return TIGHT ? only32(off) : off;
    };
    uint32_t aoff[MI], boff[4];
#pragma unroll
    for (int i = 0; i < MI; ++i) aoff[i] = a_offset(i, lane);
    if constexpr (!EXPANDS) {
#pragma unroll
        for (int i = 0; i < 4; ++i) boff[i] = b_offset(i, lane);
    }
    // 4-bit weights: in phase f every thread expands 16 weights of sub-block f + 1 from a packed double word and its scales, requested four
    // phases ago (set f & 3).  Row-packed: quarter t & 3 of weight row t >> 2.  Marlin words: half h of the unit of strip sl, chunk ch, columns
    // c of eight, k pair q: words 2 h + jj hold columns 16 (2 h + jj) + 8 b + c of the chunk, elements 2 q, 2 q + 1 of the strip in the low
    // nibbles of byte b of both half words and 2 q + 8, 2 q + 9 in the high ones.  A wave holds all q, c & 3 and sl of one (h, c >> 2, ch):
    // its lanes then write 64 different banks (with a wave on one strip four lanes met in a bank).
    uint32_t w4_off = 0, w4_soff = 0, w4_dst = 0, w4_sw = 0;
    int w4_shift = 0;
    int64_t w4_step = 32, w4_sstep = 2;                      // bytes per sub-block, and per group of scales
    if constexpr (W4A16) w4_shift = __builtin_ctz((unsigned)(p.group >> 6));
    if constexpr (is_w4nk(KIND)) {
        const int R = tid >> 2, q = tid & 3;
        const uint32_t n = (uint32_t)min(n0 + column(R), N - 1);
        w4_off = n * (uint32_t)(p.K >> 1) + (uint32_t)q * 8u;
        w4_soff = n * (uint32_t)(p.K / p.group) * 2u;
        w4_dst = (uint32_t)(R * 128);
        w4_sw = (uint32_t)(((2 * q) ^ ((R >> 1) & 7)) * 16);                  // chunk 2 q; chunk 2 q + 1 is at ^ 16
    }
    if constexpr (MARLIN) {
        const int q = lane & 3, c3 = (lane >> 2) & 3, sl = lane >> 4, h = wave & 1, c4 = (wave >> 1) & 1, ch = wave >> 2, c = 4 * c4 + c3;
        const int chunks = N >> 6, chunk = min((n0 >> 6) + ch, chunks - 1);
        w4_off = (uint32_t)((sl * chunks + chunk) * 32 + 4 * c + q) * 16u + (uint32_t)h * 8u;
        w4_soff = (uint32_t)(64 * chunk + 8 * c + 4 * h) * 2u;
        w4_step = (int64_t)chunks * 2048;
        w4_sstep = (int64_t)N * 2;
        w4_dst = (uint32_t)((64 * ch + 32 * h + 16 * c4 + c3) * 128 + 4 * q);  // LDS row of jj = b = 0; 4 (2 jj + b) rows on for the others
        w4_sw = (uint32_t)(((2 * sl) ^ (c3 >> 1)) * 16);                       // its chunk; ^ 16 for the high nibbles, ^ 16 (4 jj + 2 b)
    }
    typedef typename std::conditional<MARLIN, uint64_t, unsigned>::type W4Scale;
    uint64_t w4_words[4] = {0, 0, 0, 0};
    W4Scale w4_scale[4] = {0, 0, 0, 0};
    auto request_words = [&](int set, int u) __attribute__((always_inline)) {
        if constexpr (W4A16) {
            const int kb = kt0 + min(u, KT - 1);
            const uint8_t* const sc = (const uint8_t*)p.b_s + (int64_t)(kb >> w4_shift) * w4_sstep;
            w4_words[set] = asm_load_b64(w4_off, (const uint8_t*)p.b + (int64_t)kb * w4_step);
            if constexpr (MARLIN) w4_scale[set] = asm_load_b64(w4_soff, sc);
            else w4_scale[set] = asm_load_u16(w4_soff, sc);
        }
    };
    // every use of the words comes behind this (the wait is the caller's business)
    auto words_landed = [&](int set) __attribute__((always_inline)) {
        if constexpr (W4A16) asm volatile("" : "+v"(w4_words[set]), "+v"(w4_scale[set]) : : "memory");
    };
    auto expand_word = [&](int set, int u, int c) __attribute__((always_inline)) {
        uint8_t* const dst = lds + B0 + (u & 1) * B_SLOT + w4_dst;
        if constexpr (is_w4nk(KIND)) *(v4i*)(dst + (w4_sw ^ (uint32_t)(c * 16))) = w4_word_x8<KIND>((unsigned)(w4_words[set] >> (32 * c)), w4_scale[set]);
        if constexpr (MARLIN) {
            const v2h k1032 = {(_Float16)1032.f, (_Float16)1032.f}, k16 = {(_Float16)0.0625f, (_Float16)0.0625f}, k72 = {(_Float16)72.f, (_Float16)72.f};
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const unsigned w = (unsigned)(w4_words[set] >> (32 * c)) >> (8 * b), s16 = (unsigned)(w4_scale[set] >> (16 * (2 * c + b))) & 0xffffu;
                const v2h sc = w4_as_h2(s16 | (s16 << 16));
                const uint32_t at = w4_sw ^ (uint32_t)(16 * (4 * c + 2 * b));
                *(v2h*)(dst + 512 * (2 * c + b) + at) = (w4_as_h2((w & 0x000f000fu) | 0x64006400u) - k1032) * sc;
                *(v2h*)(dst + 512 * (2 * c + b) + (at ^ 16u)) = (w4_as_h2((w & 0x00f000f0u) | 0x64006400u) * k16 - k72) * sc;
            }
        }
    };
    // int8 activations: its products keep the multiplying group's vector ALU busy, so the fetching one expands.  In its turn of phase u thread t
    // of the group takes eight words of sub-block u + 1, packed row (t >> 4) & 15, elements 8 (t & 15) .. + 7, requested four phases ago (set
    // (u >> 1) & 1).  A 16-bit lane holds q << 4 a, q being nibble a of a half word (a = 3: q); times s4 << (8 - 4 a) (a = 3: 8) plus
    // (-z4 s4) << 8 its high byte is the int8 weight with its wrap.  tab: that factor and that term of every row of the tile, [sub-block][row].
    unsigned* const tab = (unsigned*)(bsl + D_MAX_KT);
    uint32_t w8_off = 0, w8_dst[2] = {0, 0};
    if constexpr (W4A8) {
        const int pr = (tid >> 4) & 15, k8 = tid & 15;
        w8_off = (uint32_t)min((n0 >> 3) + pr, (N >> 3) - 1) * (uint32_t)(K * 4) + (uint32_t)k8 * 32u;
        // LDS rows of the packed row's columns i: R0 + 16 (i >> 2) + (i & 3)
        const int R0 = 64 * (pr >> 3) + 32 * ((pr >> 2) & 1) + 4 * (pr & 3);
#pragma unroll
        for (int h = 0; h < 2; ++h) w8_dst[h] = (uint32_t)((R0 + 2 * h) * 128 + (((k8 >> 1) ^ (((R0 + 2 * h) >> 1) & 7)) * 16) + (k8 & 1) * 8);
    }
    v4i w8_words[2][2] = {{{0, 0, 0, 0}, {0, 0, 0, 0}}, {{0, 0, 0, 0}, {0, 0, 0, 0}}};
    auto request_words8 = [&](int set, int u) __attribute__((always_inline)) {
        if constexpr (W4A8) {
            const uint8_t* const base = p.b + (int64_t)(kt0 + min(u, KT - 1)) * 512;
            w8_words[set][0] = asm_load_b128(w8_off, base);
            w8_words[set][1] = asm_load_b128<16>(w8_off, base);
        }
    };
    auto words8_landed = [&](int set) __attribute__((always_inline)) {
        if constexpr (W4A8) asm volatile("" : "+v"(w8_words[set][0]), "+v"(w8_words[set][1]) : : "memory");
    };
    auto expand8 = [&](int set, int u) __attribute__((always_inline)) {
        if constexpr (W4A8) {
            typedef unsigned short us2 __attribute__((ext_vector_type(2)));
            auto lanes = [](unsigned v) { return __builtin_bit_cast(us2, v); };
            auto bits = [](us2 v) { return __builtin_bit_cast(unsigned, v); };
            const v4i* const row = (const v4i*)(tab + u * DU_BN + 8 * ((tid >> 4) & 15));
            const v4i sc[2] = {row[0], row[1]};
            uint8_t* const dst = lds + B0 + (u & 1) * B_SLOT;
#pragma unroll
            for (int half = 0; half < 2; ++half) {           // nibbles 4 half .. + 3
                const unsigned sel = half ? 0x07060302u : 0x05040100u;
                unsigned h[4];                               // elements 2 e, 2 e + 1 of the eight
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    h[e] = __builtin_amdgcn_perm((unsigned)w8_words[set][e >> 1][2 * (e & 1) + 1], (unsigned)w8_words[set][e >> 1][2 * (e & 1)], sel);
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    const us2 v = lanes((unsigned)sc[half][a]), mul = __builtin_shufflevector(v, v, 0, 0), add = __builtin_shufflevector(v, v, 1, 1);
                    unsigned y[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const us2 x = a == 3 ? lanes(h[e]) >> (unsigned short)12 : lanes(h[e] & (0x000f000fu << (4 * a)));
                        y[e] = bits(x * mul + add);
                    }
                    const uint64_t o = (uint64_t)__builtin_amdgcn_perm(y[1], y[0], 0x07050301u) | (uint64_t)__builtin_amdgcn_perm(y[3], y[2], 0x07050301u) << 32;
                    *(uint64_t*)(dst + w8_dst[a >> 1] + (a & 1) * 128 + half * 2048) = o;
                }
            }
        }
    };
    auto request = [&](int u) {                              // operands of sub-block u, by the four waves of one group
        const uint32_t sa = lds_base + (uint32_t)(u & 3) * A_SLOT, sb = lds_base + B0 + (uint32_t)(u & 3) * B_SLOT;
        const uint8_t* ga = p.a + (int64_t)(kt0 + u) * 128;
        const uint8_t* gb = bbase + (int64_t)(kt0 + u) * 128;
#pragma unroll
        for (int i = 0; i < MI; ++i) dma16(sa + (uint32_t)(w4 * MI + i) * 1024u, aoff[i], ga);
        if constexpr (!EXPANDS) {
#pragma unroll
            for (int i = 0; i < 4; ++i) dma16(sb + (uint32_t)(w4 * 4 + i) * 1024u, boff[i], gb);
        }
    };
    // scale window w (sub-blocks 4 w .. 4 w + 3), [row][sub-block] dwords: lane l requests row l >> 2 of 16, sub-block 4 w + (l & 3)
    uint32_t srow[NSW];
#pragma unroll
    for (int i = 0; i < NSW; ++i)
        srow[i] = SCALED ? (uint32_t)min(m_start + 16 * min(wave + 8 * i, 2 * MI - 1) + (lane >> 2), m_end - 1) * (uint32_t)KT_all : 0;
    auto request_scales = [&](int window) {
        if constexpr (SCALED) {
            const int w = __builtin_amdgcn_readfirstlane(window);
            const uint32_t kb = (uint32_t)min(kt0 + 4 * w + (lane & 3), kt0 + KT - 1);
#pragma unroll
            for (int i = 0; i < NSW; ++i) {
                const uint32_t dst = lds_base + SW + (uint32_t)(w & 1) * (du_windows(MI) / 2) + (uint32_t)min(wave + 8 * i, 2 * MI - 1) * 256u;
                if constexpr (AS16) dma2(dst, (srow[i] + kb) * 2u, p.a_s);
                else dma4(dst, (srow[i] + kb) * 4u, p.a_s);
            }
        }
    };

    // acc[i][j][q] = C[row 16 i + r][column 32 (j >> 1) + 8 g + 4 (j & 1) + q] of the wave's tile, over the group's sub-blocks.  The
    // products of a tile row wait in t and are scaled while the next row is multiplied.
    v4f acc[MI][4], t[4];
    v8i bf[4], af[MI];
    float sa[MI];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int i = 0; i < MI; ++i) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};
        t[j] = (v4f){0.f, 0.f, 0.f, 0.f};
    }
    auto clear = [&]() {
#pragma unroll
        for (int j = 0; j < 4; ++j) bf[j] = (v8i){0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            af[i] = (v8i){0, 0, 0, 0, 0, 0, 0, 0};
            sa[i] = 0.f;
        }
    };
    clear();
    const int lo = r * 128 + ((g ^ ((r >> 1) & 7)) * 16);
    const int hi = r * 128 + (((g + 4) ^ ((r >> 1) & 7)) * 16);
    auto ldfrag = [&](const uint8_t* base) {
        const v4i x = *(const v4i*)(base + lo), y = *(const v4i*)(base + hi);
        return (v8i){x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
    };
    auto fetch = [&](int u) {
        const uint8_t* const As = lds + (u & 3) * A_SLOT + wm * WR * 128;
        const uint8_t* const Bs = lds + B0 + (u & (NB - 1)) * B_SLOT + wn * 64 * 128;
#pragma unroll
        for (int j = 0; j < 4; ++j) bf[j] = ldfrag(Bs + j * 2048);
#pragma unroll
        for (int i = 0; i < MI; ++i) af[i] = ldfrag(As + i * 2048);
        if constexpr (SCALED) {
            const float bs = bsl[u];
            const float* const Ss = (const float*)(lds + SW + ((u >> 2) & 1) * (du_windows(MI) / 2)) + (wm * WR + r) * 4 + (u & 3);
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                if constexpr (AS16) {
                    const unsigned raw = ((const unsigned*)Ss)[i * 64];
                    sa[i] = scale16_f32<SDT>(raw) * bs;
                } else {
                    sa[i] = Ss[i * 64] * bs;
                }
            }
        }
    };
    // 4-bit weights: in the shadow of its matrix instructions the multiplying group expands its half of sub-block f + 1 of phase f (the slot's
    // readers finished in the phase before), and requests the words of sub-block f + 5
    auto multiply = [&](auto expand_c, int f) __attribute__((always_inline)) {
        constexpr bool EXPAND = W4A16 && decltype(expand_c)::value;
        if constexpr (EXPAND) words_landed(f & 3);
        if constexpr (W4A16) __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            if constexpr (EXPAND) {
                if (i < 2) expand_word(f & 3, f + 1, i);
                if (i == (MI > 2 ? 2 : MI - 1)) request_words(f & 3, f + 5);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if constexpr (SCALED) {
                    if (i > 0) acc[i - 1][j] += raw_f32<MATH>(t[j]) * sa[i - 1];
                    t[j] = step_raw<MATH>(bf[j], af[i]);
                    __builtin_amdgcn_sched_barrier(0);
                } else {
                    acc[i][j] = mma_plain<KIND>(bf[j], af[i], acc[i][j]);
                }
            }
            if constexpr (EXPAND) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (SCALED) {
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[MI - 1][j] += raw_f32<MATH>(t[j]) * sa[MI - 1];
        }
        if constexpr (W4A16) __builtin_amdgcn_s_setprio(0);
    };
    auto meet = [&](auto left_c) {                           // this wave's LDS accesses, and its loads but the left_c youngest, are done
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (decltype(left_c)::value < 0) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(decltype(left_c)::value < 0 ? 0 : decltype(left_c)::value) : "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    const std::true_type yes;
    const std::false_type no;
    const std::integral_constant<int, -1> any;
    const std::integral_constant<int, 0> none;
    const std::integral_constant<int, LP> c_l;
    const std::integral_constant<int, LP + (SCALED ? NSW : 0)> c_ls;

    // Turn of the fetching group in phase u.  The operands requested in its last turn, two phases ago, have landed when only the loads since
    // are in flight: sub-block u + 1 is complete, and so are the words that the group expands in the next two phases.  SCALES: this turn also
    // requests the next scale window, behind its operands, so that the turn after it waits for it; the window it overwrites was last read
    // in phase u - 1 or before.
    auto turn = [&](int u, auto scales_c) __attribute__((always_inline)) {
        constexpr bool SCALES = SCALED && decltype(scales_c)::value;
        // (the wave that ends the phase goes first; us with the multiplying wave first | none | the fetching one, 1024 x 4096 x 4096: int8 25.8 | 25.1 |
        // 24.0, fp8 21.4 | 21.4 | 21.1, w4a8 35.5 | 31.7 | 30.8, per token the same, bf16 x 4-bit 42.0 | 43.3 | 44.7)
        if constexpr (SCALED) __builtin_amdgcn_s_setprio(1);
        // 4-bit weights, 16-bit activations: the LDS reads go first, so that the wave's requests, which wait for the address path one by one, run beside
        // them, and row-packed words are expanded in front of the requests too (Marlin words, whose expansion is eight scattered writes, behind
        // them).  us, requests first | reads first, then requests | expansion in front of the requests: rows 300 x 14336 x 4096 bf16 44.1 | 42.7 | 41.9, fp16
        // 44.9 | 43.4 | 42.6, bf16 512 x 6144 x 4096 36.7 | 37.9 | 35.8, fp16 1500 x 4096 x 4096 55.1 | 52.6 | 52.4, Marlin 320 x 14336 x 4096 47.0 | 43.4 |
        // 46.7, 768 x 4096 x 7168 61.6 | 58.5 | 60.9.  8-bit operands: no difference (fp8 1024 x 4096 x 4096 25.9 | 25.8, int8 200 x 14336 x 4096 25.0 | 25.3).
        // Random shapes of 65 to 520 rows, weights of 8 MB or more for the most part, cached (from HBM): Marlin words 1.08 (1.055) times as fast as with the requests first,
        // row-packed ones on tiles of 96 | 128 | 160 | 192 rows fp16 1.03 (1.01) | 1.06 (1.03) | 1.06 (1.03) | 1.06 (1.03), bf16 1.01 (0.99) | 1.02 (1.01) | 1.04 (1.03) |
        // 1.07 (1.03).  So bf16 on 96-row tiles keeps the requests first: little is expanded beside few rows, and wide weights wait for HBM (94 x 25864 x
        // 6016 with the reads first 8 % slower).  What is left are single shapes of wide weights from HBM, with an odd number of K steps for the most part
        // (rows of words then begin in the middle of a line): 2 to 8 % slower, 4 % faster cached (fp16 262 x 8896 x 8064).
        constexpr bool READS_FIRST = W4A16 && !(KIND == K_W4NKB && MI == 3);
        auto expand_words = [&]() __attribute__((always_inline)) {
            __builtin_amdgcn_sched_barrier(0);
            words_landed(u & 3);
            expand_word(u & 3, u + 1, 0);
            expand_word(u & 3, u + 1, 1);
            __builtin_amdgcn_sched_barrier(0);
        };
        if constexpr (READS_FIRST) {
            fetch(u);
            if constexpr (!MARLIN) expand_words();
            __builtin_amdgcn_sched_barrier(0);
        }
        request(u + 3);
        if constexpr (SCALES) request_scales((u >> 2) + 1);
        if constexpr (W4A16 && !READS_FIRST) fetch(u);
        if constexpr (W4A16) {
            if constexpr (MARLIN || !READS_FIRST) expand_words();
            request_words(u & 3, u + 5);
        }
        if constexpr (W4A8) {                                // (in front of the fragments, which leave no registers for it)
            words8_landed((u >> 1) & 1);
            expand8((u >> 1) & 1, u + 1);
            request_words8((u >> 1) & 1, u + 5);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (!W4A16) fetch(u);
        if constexpr (SCALED) __builtin_amdgcn_s_setprio(0);
        if constexpr (SCALES) meet(c_ls);
        else meet(c_l);
    };
    // The same where little or nothing is left to request: every phase waits for all of it, and the words move up a set a phase.
    auto last_words = [&](int f) __attribute__((always_inline)) {
        if constexpr (W4A16) {
            if (f + 1 < KT) {
                expand_word(0, f + 1, 0);
                expand_word(0, f + 1, 1);
            }
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                w4_words[i] = w4_words[i + 1];
                w4_scale[i] = w4_scale[i + 1];
            }
            request_words(3, f + 5);
        }
    };
    auto last_meet = [&]() __attribute__((always_inline)) {
        meet(none);
        words_landed(3);
    };
    auto last_turn = [&](int u) __attribute__((always_inline)) {
        if constexpr (TIGHT) {                               // (worked out again: no registers to keep them through these turns)
            int l = lane;
            asm volatile("" : "+v"(l));
#pragma unroll
            for (int i = 0; i < MI; ++i) aoff[i] = a_offset(i, l);
#pragma unroll
            for (int i = 0; i < 4; ++i) boff[i] = b_offset(i, l);
#pragma unroll
            for (int i = 0; i < NSW; ++i) srow[i] = (uint32_t)min(m_start + 16 * min(wave + 8 * i, 2 * MI - 1) + (l >> 2), m_end - 1) * (uint32_t)KT_all;
        }
        if (u + 3 < KT) request(u + 3);
        if constexpr (SCALED) if ((u & 3) < 2 && (u | 3) + 1 < KT) request_scales((u >> 2) + 1);
        if constexpr (W4A8) {
            if (u + 1 < KT) expand8(0, u + 1);
            w8_words[0][0] = w8_words[1][0];
            w8_words[0][1] = w8_words[1][1];
            request_words8(1, u + 5);
            __builtin_amdgcn_sched_barrier(0);
        }
        fetch(u);
        last_words(u);
        last_meet();
        words8_landed(1);
    };
    auto all_landed = [&]() __attribute__((always_inline)) {
        if constexpr (W4A16) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
            for (int i = 0; i < 4; ++i) words_landed(i);
        }
        if constexpr (W4A8) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            words8_landed(0);
            words8_landed(1);
        }
    };

    // ---- the first three sub-blocks; 4-bit weights: the weight rows of the first, and the words of the four behind it
    if (KT > 0) {
        request_words(0, 0);
        request_words8(0, 0);
        if (wave < 4) {
            if (KT > 1) request(1);
        } else {
            request(0);
            if (KT > 2) request(2);
        }
        request_scales(0);
        if constexpr (SCALED) {
            const int64_t bs_row = bs_off + (int64_t)tile_n * KT_all + kt0;
            for (int i = tid; i < KT; i += DU_THREADS) bsl[i] = ld_scale(p.b_s, bs_row + i, p.s_dtype);
        }
        if constexpr (W4A8) {
            // thread: four (or, at odd counts, one) sub-blocks of a row, rows of a wave side by side
            const int8_t* const s4 = p.w4_s4 + (int64_t)n0 * KT_all + kt0;
            const int8_t* const z4 = p.w4_z4 + (int64_t)n0 * KT_all + kt0;
            const uint32_t row = (uint32_t)min(tid & (DU_BN - 1), N - 1 - n0) * (uint32_t)KT_all;
            const int shift = (tid & 3) == 3 ? 8 : 8 - 4 * (tid & 3);
            auto put = [&](int kb, unsigned s, unsigned z) {
                tab[kb * DU_BN + (tid & (DU_BN - 1))] = (s & 0xffu) << shift | (0u - (z & 0xffu) * (s & 0xffu)) << 24;
            };
            if (((KT_all | KT | kt0) & 3) == 0) {
                for (int kb = 4 * (tid >> 7); kb < KT; kb += 16) {
                    const unsigned s = ((const Loose<unsigned, 1>*)(s4 + row + kb))->v, z = ((const Loose<unsigned, 1>*)(z4 + row + kb))->v;
#pragma unroll
                    for (int b = 0; b < 4; ++b) put(kb + b, s >> (8 * b), z >> (8 * b));
                }
            } else {
                for (int kb = tid >> 7; kb < KT; kb += 4) put(kb, (uint8_t)s4[row + kb], (uint8_t)z4[row + kb]);
            }
        }
        all_landed();
        if constexpr (W4A8) {
            meet(none);                                      // the table
            if (wave >= 4) expand8(0, 0);
            request_words8(0, wave < 4 ? 1 : 2);
            request_words8(1, wave < 4 ? 3 : 4);
        }
        expand_word(0, 0, 0);
        expand_word(0, 0, 1);
#pragma unroll
        for (int i = 0; i < 4; ++i) request_words(i, i + 1);
        all_landed();
    }
    meet(none);

    // ---- each group keeps half of the tile rows of its waves, passes the other half to its counterpart and stores the sums
    constexpr int H = (MI + 1) / 2;
    const bool split = !GROUPED && p.ksplit > 1;
    void* const cout = split ? (void*)(p.partial + (int64_t)blockIdx.z * p.M * N) : p.c;
    const int cdt = split ? LLMK_F32 : p.c_dtype;
    auto finish = [&](auto grp_c) {
        constexpr int G = decltype(grp_c)::value, KEEP = G ? H : 0, NKEEP = G ? MI - H : H, GIVE = G ? 0 : H, NGIVE = MI - NKEEP;
        v4f* const give = (v4f*)lds + wave * (H * 4 * 64) + lane;
        const v4f* const take = (const v4f*)lds + (wave ^ 4) * (H * 4 * 64) + lane;
#pragma unroll
        for (int i = 0; i < NGIVE; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) give[(i * 4 + j) * 64] = acc[GIVE + i][j];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NKEEP; ++i) {
            const int m = m_start + wm * WR + 16 * (KEEP + i) + r;
            if (m >= m_end) continue;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int nb = n0 + wn * 64 + 32 * h + 8 * g, nv = N - nb;
                if (nv <= 0) continue;
                v4f s[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const v4f o = take[(i * 4 + 2 * h + e) * 64], mine = acc[KEEP + i][2 * h + e];
                    if constexpr (ROWCOL) s[e] = __builtin_bit_cast(v4f, __builtin_bit_cast(v4i, o) + __builtin_bit_cast(v4i, mine));
                    else s[e] = o + mine;
                }
                const int64_t off = (int64_t)m * N + nb;
                if constexpr (ROWCOL) {
                    if (!split) {                            // (a K slice leaves its int32 sums, see splitk_sum_rowcol_kernel)
                        rowcol_epilogue8(p, s[0], s[1], m, off, nb, nv);
                        if (!p.c) continue;
                    }
                }
                if (cdt == LLMK_BF16) store_run8<LLMK_BF16>(cout, off, s[0], s[1], nv);
                else if (cdt == LLMK_F16) store_run8<LLMK_F16>(cout, off, s[0], s[1], nv);
                else store_run8<LLMK_F32>(cout, off, s[0], s[1], nv);
            }
        }
    };

    // Four phases a loop turn (the last operands they request are those of sub-block 4 q + 6), then phase by phase what is left.
    const int rounds = KT >= 7 ? (KT - 3) >> 2 : 0;
    auto nothing_left = [&]() __attribute__((always_inline)) {               // an odd number of sub-blocks: nothing left to multiply
        clear();
        meet(any);
    };
    if (wave < 4) {
        for (int q = 0; q < rounds; ++q) {
            turn(4 * q, yes);
            multiply(yes, 4 * q + 1);
            meet(any);
            turn(4 * q + 2, no);
            multiply(yes, 4 * q + 3);
            meet(any);
        }
        if constexpr (!TIGHT) {
            all_landed();
            for (int u = 4 * rounds; u < KT; u += 2) {
                last_turn(u);
                last_words(u + 1);
                multiply(no, 0);
                last_meet();
            }
            finish(std::integral_constant<int, 0>{});
        }
    } else {
        for (int q = 0; q < rounds; ++q) {
            multiply(yes, 4 * q);
            meet(any);
            turn(4 * q + 1, yes);
            multiply(yes, 4 * q + 2);
            meet(any);
            turn(4 * q + 3, no);
        }
        if constexpr (!TIGHT) {
            all_landed();
            for (int u = 4 * rounds; u < KT; u += 2) {
                last_words(u);
                multiply(no, 0);
                last_meet();
                if (u + 1 < KT) last_turn(u + 1);
                else nothing_left();
            }
            multiply(no, 0);
            finish(std::integral_constant<int, 1>{});
        }
    }
    if constexpr (TIGHT) {
        // one loop for both groups: with a loop each, the compiler keeps the registers of the second through the first and spills (a loop each is
        // 1.3 us faster where they suffice: the registers move between the main loops and this one)
        for (int f = 4 * rounds; f < ((KT + 1) & ~1); ++f) {
            if ((f & 1) != (wave >> 2)) {
                multiply(no, 0);
                last_meet();
            } else if (f < KT) {
                last_turn(f);
            } else {
                nothing_left();
            }
        }
        if (wave < 4) {
            finish(std::integral_constant<int, 0>{});
        } else {
            multiply(no, 0);
            finish(std::integral_constant<int, 1>{});
        }
    }
}

// p.a_s: fp32, or with AS16 the 16-bit scales of dtype p.s_dtype as the caller passed them; p.ksplit / p.partial select the K split.
template <int KIND, int MI, bool AS16 = false, bool GROUPED = false>
int launch_duo(const DirectArgs& p, hipStream_t stream, const char* name) {
    constexpr int fixed = du_lds(KIND, MI);
    static_assert(fixed <= D_LDS_MAX && 8 * ((MI + 1) / 2) * 4096 <= fixed, "slots, and the exchange of half the sums in them, fit in LDS");
    const int KT = (p.K * (is_half(KIND) ? 2 : 1)) >> 7, z = p.ksplit > 1 ? p.ksplit : 1;
    const int lds_bytes = fixed + (KIND == K_W4A8 ? du_table((KT + z - 1) / z) : 0);
    if (lds_bytes > D_LDS_MAX) LLMK_FAIL(LLMK_ERR_SHAPE, "%s: %d bytes of LDS needed", name, lds_bytes);
    const bool split = !GROUPED && p.ksplit > 1 && p.partial;
    DirectArgs q = p;
    q.ksplit = split ? p.ksplit : 1;
    const int tiles_m = GROUPED ? grouped_row_tiles(p.M, p.E, 32 * MI) : (p.M + 32 * MI - 1) / (32 * MI);
    dim3 grid((unsigned)((p.N + DU_BN - 1) / DU_BN), (unsigned)tiles_m, (unsigned)q.ksplit);
    if (grid.x == 0 || grid.y == 0) return LLMK_OK;
    auto launch = [&](auto sdt_c) {
        static std::atomic<uint64_t> configured{0};
        auto kern = gemm_duo_kernel<KIND, MI, decltype(sdt_c)::value, GROUPED>;
        if (int rc = llmk_reserve_lds((const void*)kern, KIND == K_W4A8 ? D_LDS_MAX : fixed, configured, name)) return rc;
        kern<<<grid, DU_THREADS, lds_bytes, stream>>>(q);
        LLMK_CHECK_LAUNCH(name);
        return (int)LLMK_OK;
    };
    if (int rc = with_scale_type<AS16>(p.s_dtype, launch)) return rc;
    return split ? launch_splitk_sum<KIND == K_W4A8 ? K_I8_BLOCK : KIND>(q, q.ksplit, stream, name) : LLMK_OK;
}

// Tile heights that are built (32 mi rows); at the next one the fragments of a sub-block, the sums and what waits to be expanded or scaled
// spill.
template <int KIND>
constexpr bool duo_built(int mi) {
    return mi >= 3 && mi <= (is_w4nk(KIND) ? 6 : (KIND == K_W4A8 ? 4 : 5));
}
// Estimated microseconds: base + rounds of 256 workgroups x (round + sub-blocks x step[mi - 3]) + out x MB of the output, and for K slices
// split + plane x MB of the fp32 planes.  A fit of 4 to 7 % rms to 300 random shapes a kind of M 64 to 4096, N 1024 to 28672, K 1024 to
// 14336, every height and up to eight slices timed, means of cached weights and of weights from HBM.
struct DuoModel {
    float base, round, step[4], split, plane, out;
};
template <int KIND>
constexpr DuoModel duo_model() {
    if (KIND == K_FP8_BLOCK) return {2.0f, 1.4f, {0.396f, 0.452f, 0.515f, 0.f}, 3.0f, 0.47f, 0.48f};
    if (KIND == K_I8_BLOCK) return {2.4f, 1.4f, {0.417f, 0.502f, 0.585f, 0.f}, 3.1f, 0.45f, 0.57f};
    if (KIND == K_W4MARLIN) return {3.03f, 2.53f, {0.460f, 0.519f, 0.589f, 0.f}, 2.9f, 0.45f, 0.31f};
    if (KIND == K_W4A8) return {1.76f, 2.62f, {0.614f, 0.683f, 0.f, 0.f}, 3.0f, 0.55f, 0.37f};
    if (KIND == K_I8_ROWCOL) return {2.79f, 1.59f, {0.355f, 0.406f, 0.470f, 0.f}, 2.9f, 0.47f, 0.57f};
    return {2.29f, 1.78f, {0.421f, 0.487f, 0.561f, 0.639f}, 3.7f, 0.46f, 0.43f};
}
struct DuoPlan {
    int mi, z;                                               // mi == 0: not for this kernel
    double cost;
};
// The cheapest height and number of K slices with `scratch` bytes for their planes (at most DU_MAX_PLANES: what is reported as scratch
// stays within the array that serves calls without any).
constexpr int64_t DU_MAX_PLANES = LLMK_STATIC_SCRATCH_BYTES;
template <int KIND>
DuoPlan duo_plan(const DirectArgs& p, int64_t scratch) {
    constexpr int ESZ = is_half(KIND) ? 2 : 1;
    constexpr DuoModel m = duo_model<KIND>();
    DuoPlan best{0, 1, 1e30};
    if (p.M <= 64 || !dma_eligible(p, ESZ) || (du_w4a16(KIND) && (p.group < 64 || (p.group & (p.group - 1))))) return best;
    const int KT = (p.K * ESZ) >> 7;
    const int64_t gx = (p.N + DU_BN - 1) / DU_BN, planes = std::min(scratch, DU_MAX_PLANES);
    const double out = (double)p.M * p.N * 1e-6;
    for (int mi = 3; mi <= 6; ++mi) {
        if (!duo_built<KIND>(mi)) continue;
        const int64_t tiles = gx * ((p.M + 32 * mi - 1) / (32 * mi));
        constexpr int Z[] = {1, 2, 3, 4, 6, 8};
        for (int z : Z) {
            if (z > 1 && (tiles * z > LLMK_CUS || KT / z < 6 || (int64_t)z * p.M * p.N * 4 > planes)) break;
            if (KIND == K_W4A8 && du_lds(KIND, mi) + du_table((KT + z - 1) / z) > D_LDS_MAX) continue;
            const double rounds = (double)((tiles * z + LLMK_CUS - 1) / LLMK_CUS);
            // the tight tile: its shared last loop costs 1.8 us a tile, and beyond 512 rows and a round of them the 256-column tiles are the
            // faster ones, which their estimates there do not show (fp8 2337 x 4096 x 4096 45.0 | 49.3 this one, int8 2375 x 28672 x 4096 320 | 333)
            if (du_tight(KIND, mi) && p.M > 512 && tiles > LLMK_CUS) break;
            const double round = m.round + (du_tight(KIND, mi) ? 1.8 : 0.0);
            const double c = m.base + rounds * (round + (KT + z - 1) / z * m.step[mi - 3]) + 2.0 * m.out * out + (z > 1 ? m.split + 4.0 * m.plane * out * z : 0.0);
            if (c < best.cost) best = {mi, z, c};
        }
    }
    return best;
}
inline bool duo_beyond_a_round(const DirectArgs& p, const DuoPlan& d) {
    return (int64_t)((p.N + DU_BN - 1) / DU_BN) * ((p.M + 32 * d.mi - 1) / (32 * d.mi)) * d.z > LLMK_CUS;
}
// A choice by two estimates: this kernel's has to be this much below the other one.
constexpr double DU_MARGIN = 1.08;
// The same in more than a round of workgroups against 256-row tiles of 4-bit weights: both estimates are 4 to 8 % off there, in opposite
// directions (a row of these tiles a CU more or less, and every one of them expands the weights again).  Of 195 shapes 64 fell between the two margins,
// 0.99 times as fast on this kernel (us, others | this one: fp16 976 x 10616 x 7168 161 | 176, 201 x 23784 x 9728 152 | 165, Marlin words 432 x 13056
// x 9472 140 | 158, 1920 x 4544 x 3968 84 | 90).
constexpr double DU_MARGIN_TALL = 1.20;
template <int KIND, bool AS16 = false>
int launch_duo_plan(DirectArgs p, const DuoPlan& pl, void* workspace, hipStream_t stream, const char* name) {
    if (pl.z > 1) { p.partial = (float*)workspace; p.ksplit = pl.z; }
    if constexpr (duo_built<KIND>(6)) if (pl.mi == 6) return launch_duo<KIND, 6, AS16>(p, stream, name);
    if constexpr (duo_built<KIND>(5)) if (pl.mi == 5) return launch_duo<KIND, 5, AS16>(p, stream, name);
    return pl.mi == 4 ? launch_duo<KIND, 4, AS16>(p, stream, name) : launch_duo<KIND, 3, AS16>(p, stream, name);
}

// Grouped products: tile height (mi; 0: not for this kernel) where an expert's rows are one tile and all tiles one round of the chip.
// The rows of a segment are only known on the device: mean + 1.5 standard deviations of an even routing are taken for the longest.
// There each workgroup reads its share of the weights once, and the deeper queue of loads is what counts (us, the 64- and 128-row
// tiles of gemm_dma_kernel | these: fp8 8 experts of 4096 x 14336, 362 rows 88 | 84, 512 98 | 88, 860 135 | 101; int8 452 rows 158 | 88;
// over 299 random shapes inside the rule 1.13 fp8, 1.20 int8).  Outside it they are level or behind:
// above 200 tiles of up to 64 rows from 7168 columns or fewer, two workgroups a CU of the 64-row tile keep as much in flight
// (8 x 4096 x 7168, 256 rows 37 | 39), and with more than one round (16 experts of 4096 x 4096, 1448 rows) the 256-column tiles
// take 44 us, these 54.  From 5120 columns: 16 x 4096 x 2048, 980 rows 27 | 28.
// Up to half a round and from some 85 rows on, two 64-row tiles an expert stream the weights on twice the CUs: 77 shapes there were 0.92 times
// as fast on these tiles, with weights from HBM 0.85 (8 experts of 592 x 6912, 684 rows 24.2 | 24.2 cached, 29.7 | 37.0 from HBM; int8 2 of
// 1448 x 9856, 167 rows 39 | 49).  128-row tiles from 90 rows: a segment beyond 96 would start another round of 96-row ones (int8 8 of
// 4096 x 14336, 645 rows 117 | 128).
inline int grouped_duo_mi(const DirectArgs& p) {
    if (p.E <= 0 || p.K < 5120 || !dma_eligible(p)) return 0;
    const double rows = (double)p.M / p.E, longest = rows + 1.5 * __builtin_sqrt(rows);
    const int64_t tiles = (int64_t)p.E * ((p.N + DU_BN - 1) / DU_BN);
    if (rows < 20.0 || longest > 128.0 || tiles > LLMK_CUS || (tiles > 200 && p.K < 8192 && rows < 64.0)) return 0;
    if (longest > 85.0 && tiles <= LLMK_CUS / 2) return 0;
    return longest <= 64.0 ? 2 : (longest <= 90.0 ? 3 : 4);
}
template <int KIND, bool AS16>
int launch_grouped_duo(const DirectArgs& p, int mi, hipStream_t stream, const char* name) {
    if (mi == 2) return launch_duo<KIND, 2, AS16, true>(p, stream, name);
    return mi == 3 ? launch_duo<KIND, 3, AS16, true>(p, stream, name) : launch_duo<KIND, 4, AS16, true>(p, stream, name);
}

}  // namespace llmk

// Single-GPU expert-parallel MoE path: segment bookkeeping, token permute / un-permute,
// gated activation, and the grouped GEMM over one GPU's experts.
#include "gemm_duo.hpp"
#include "gemm_wide.hpp"
#include "quant_util.hpp"

using namespace llmk;

namespace {

// seg_indptr[e + 1] = number of sorted ids <= e (binary search for the right boundary)
__global__ void seg_indptr_kernel(const int64_t* __restrict__ sorted_ids, int64_t* __restrict__ seg_indptr,
                                  int64_t num_toks, int num_experts) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= num_experts) return;
    int64_t lo = 0, hi = num_toks;       // first index with id > e
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (sorted_ids[mid] > e) hi = mid; else lo = mid + 1;
    }
    seg_indptr[e + 1] = lo;
    if (e == 0) seg_indptr[0] = 0;
}

__global__ void src2dst_kernel(const int64_t* __restrict__ reorder_ids, int32_t* __restrict__ src2dst, int64_t n) {
    const int64_t d = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (d < n) src2dst[reorder_ids[d]] = (int32_t)d;
}

__device__ __forceinline__ int64_t ld_id(const void* p, int64_t i, int bytes) {
    return bytes == 8 ? ((const int64_t*)p)[i] : (int64_t)((const int32_t*)p)[i];
}

// Stable counting sort of the flattened expert ids, with the segment pointers and the source -> destination
// map as by-products: what torch.sort(stable) + seg_indptr_kernel + src2dst_kernel produce in eight launches.
// Bucket 0 takes negative ids, bucket e + 1 expert e, bucket E + 1 ids >= E (both out-of-range buckets keep
// their arrival order; a well-formed input leaves them empty).
// Workgroup g places the ids [g THREADS, (g + 1) THREADS).  It counts, per bucket, all ids (-> bucket starts) and
// the ids in front of its chunk, by reading the whole id list (at most PP_MAX_IDS ids, from L2); a lane's
// position is then bucket start + ids of the bucket in earlier chunks + those in the lower waves of the
// chunk + its rank among the equal ids of its own wave.  No workgroup waits for another.
// Bound by latency: a chain of one load, three barriers and a scan.  Few buckets are counted in 64 columns per bucket, one
// per lane, so that the ids of a wave never meet on one LDS address (ballots per bucket, the form before, took
// 12.2 us for 8192 ids of 8 experts, this one 8.4); lists that one workgroup holds have a kernel of their own.  What is left grows
// with the list: a workgroup's LDS additions, about one a clock (21816 ids of 64 experts 18.2 us, 32768 22.2; 23.4 and 26.2 with half the loads
// in flight and a pass per distinct bucket in the ranking).
constexpr int PP_THREADS = 1024, PP_MAX_EXPERTS = 512, PP_BUCKETS = PP_MAX_EXPERTS + 2, PP_FEW = 66;

__global__ __launch_bounds__(PP_THREADS) void ep_preprocess_kernel(const void* __restrict__ ids, int ids_bytes, int n, int E,
                                                                   void* __restrict__ sorted_out, int32_t* __restrict__ src2dst,
                                                                   int64_t* __restrict__ seg_indptr) {
    constexpr int THREADS = PP_THREADS, WAVES = THREADS / 64;
    __shared__ int tot[PP_BUCKETS];      // ids per bucket, then the bucket's first position
    __shared__ int pre[PP_BUCKETS];      // ids per bucket in front of this workgroup's chunk
    // either the columns of a few buckets (two counts per cell: ids in front of the chunk in the low half, the others in
    // the high half; at most PP_MAX_IDS / 64 ids a column) or nothing; afterwards the counts per wave
    constexpr int CELLS = PP_FEW * 64, WCELLS = WAVES * PP_BUCKETS;
    __shared__ int cells[CELLS > WCELLS ? CELLS : WCELLS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nb = E + 2;
    const int c0 = blockIdx.x * THREADS;
    auto bucket_at = [&](int i) {
        if (i >= n) return -1;
        const int64_t id = ld_id(ids, i, ids_bytes);
        return id < 0 ? 0 : (id >= E ? E + 1 : (int)id + 1);
    };
    const int b = bucket_at(c0 + tid);   // the id this thread places: requested before anything else
    const bool few = nb <= PP_FEW;
    for (int k = tid; k < nb; k += THREADS) { tot[k] = 0; pre[k] = 0; }
    if (few) for (int i = tid; i < nb * 64; i += THREADS) cells[i] = 0;
    __syncthreads();
    constexpr int U = 8;                 // rounds whose loads are in flight together
    for (int r0 = 0; r0 < n; r0 += U * THREADS) {
        int v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = bucket_at(r0 + u * THREADS + tid);
#pragma unroll
        for (int u = 0; u < U; ++u) if (v[u] >= 0) {
            const bool before = r0 + u * THREADS < c0;           // whole rounds lie in front of the chunk or not
            if (few) {
                atomicAdd(&cells[v[u] * 64 + lane], before ? 1 : 1 << 16);
            } else {
                atomicAdd(&tot[v[u]], 1);
                if (before) atomicAdd(&pre[v[u]], 1);
            }
        }
    }
    __syncthreads();
    if (few) {
        for (int k = wave; k < nb; k += WAVES) {
            const int c = cells[k * 64 + lane];
            int lo = c & 0xffff, all = lo + (c >> 16);
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) { lo += __shfl_xor(lo, o, 64); all += __shfl_xor(all, o, 64); }
            if (lane == 0) { pre[k] = lo; tot[k] = all; }
        }
        __syncthreads();
    }
    for (int i = tid; i < WAVES * nb; i += THREADS) cells[i] = 0;
    if (wave == 0) {
        // exclusive scan of the bucket counts: a run of buckets per lane, then a scan over the lanes
        const int per = (nb + 63) / 64, b0 = lane * per;
        int sum = 0;
        for (int k = 0; k < per; ++k) if (b0 + k < nb) sum += tot[b0 + k];
        int incl = sum;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int t = __shfl_up(incl, o, 64);
            if (lane >= o) incl += t;
        }
        int run = incl - sum;
        for (int k = 0; k < per; ++k) if (b0 + k < nb) {
            const int c = tot[b0 + k];
            tot[b0 + k] = run;
            run += c;
        }
    }
    __syncthreads();
    // seg_indptr[e + 1] = number of ids <= e = start of bucket e + 2; seg_indptr[0] = 0
    if (blockIdx.x == 0)
        for (int e = tid; e <= E; e += THREADS) seg_indptr[e] = e == 0 ? 0 : (int64_t)tot[e + 1];

    // rank of a lane among the lanes of its wave with the same bucket, one leader per bucket publishes the count
    // (one ballot per bit of the bucket number; a pass per distinct bucket of the wave is up to 64 of them with 64 experts)
    uint64_t same = __ballot(b >= 0);
    for (int bit = 0; nb >> bit; ++bit) {
        const bool one = (b >> bit) & 1;
        const uint64_t m = __ballot(one);
        same &= one ? m : ~m;
    }
    const int rank = __popcll(same & ((1ull << lane) - 1ull));
    if (b >= 0 && rank == 0) cells[wave * nb + b] = __popcll(same);
    __syncthreads();
    if (b >= 0) {
        int pos = tot[b] + pre[b] + rank;
        for (int w = 0; w < wave; ++w) pos += cells[w * nb + b];
        const int i = c0 + tid;
        const int64_t id = (b >= 1 && b <= E) ? (int64_t)(b - 1) : ld_id(ids, i, ids_bytes);
        if (ids_bytes == 8) ((int64_t*)sorted_out)[pos] = id; else ((int32_t*)sorted_out)[pos] = (int32_t)id;
        src2dst[i] = pos;
    }
}

// The same for a list that one workgroup holds, an id per thread: the counts of its waves are all there is to count, so there
// are no columns to clear, fill and add up, and the code is short (see below).  (us,
// the kernel above | this one: 96 ids of 64 experts 8.9 | 2.8, 256 of 8 4.7 | 2.6, 588 of 16 5.0 | 3.2, 1000 of 64 7.6 | 3.9.)
template <int THREADS>
__global__ __launch_bounds__(THREADS) void ep_preprocess_one_kernel(const void* __restrict__ ids, int ids_bytes, int n, int E,
                                                                    void* __restrict__ sorted_out, int32_t* __restrict__ src2dst,
                                                                    int64_t* __restrict__ seg_indptr) {
    constexpr int WAVES = THREADS / 64;
    __shared__ int first[PP_BUCKETS];            // the bucket's first position
    __shared__ int cells[WAVES * PP_BUCKETS];    // ids per wave and bucket
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nb = E + 2;
    const bool live = tid < n;
    const int64_t id = live ? ld_id(ids, tid, ids_bytes) : 0;
    const int b = id < 0 ? 0 : (id >= E ? E + 1 : (int)id + 1);
    for (int i = tid; i < WAVES * nb; i += THREADS) cells[i] = 0;
    uint64_t same = __ballot(live);
    for (int bit = 0; nb >> bit; ++bit) {
        const bool one = (b >> bit) & 1;
        const uint64_t m = __ballot(one);
        same &= one ? m : ~m;
    }
    const int rank = __popcll(same & ((1ull << lane) - 1ull));
    __syncthreads();
    if (live && rank == 0) cells[wave * nb + b] = __popcll(same);
    __syncthreads();
    if (wave == 0) {
        // starts of the buckets, and of a bucket's waves in it: a run of buckets per lane, then a scan over the lanes
        const int per = (nb + 63) / 64, b0 = lane * per, b1 = min(b0 + per, nb);
        int sum = 0;
        for (int k = b0; k < b1; ++k)
            for (int w = 0; w < WAVES; ++w) sum += cells[w * nb + k];
        int incl = sum;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int t = __shfl_up(incl, o, 64);
            if (lane >= o) incl += t;
        }
        int run = incl - sum;
        for (int k = b0; k < b1; ++k) {
            first[k] = run;
            for (int w = 0; w < WAVES; ++w) {
                const int c = cells[w * nb + k];
                cells[w * nb + k] = run;
                run += c;
            }
        }
    }
    __syncthreads();
    for (int e = tid; e <= E; e += THREADS) seg_indptr[e] = e == 0 ? 0 : (int64_t)first[e + 1];
    if (live) {
        const int pos = cells[wave * nb + b] + rank;
        if (ids_bytes == 8) ((int64_t*)sorted_out)[pos] = id; else ((int32_t*)sorted_out)[pos] = (int32_t)id;
        src2dst[tid] = pos;
    }
}

// The same for at most 64 ids: one wave, a lane per id, no LDS.  Every lane counts the ids of lower buckets and the equal
// ids of lower lanes, one pass per distinct bucket.  What such a launch costs behind a kernel that streamed the experts'
// weights is fetching its code from memory again, so the code is short (32 ids, 8 experts: launches back to back 5.4 us in
// the general form, 2.0 here; in an expert layer of 16 tokens 5.9 and 4.7).
__global__ __launch_bounds__(64) void ep_preprocess_wave_kernel(const void* __restrict__ ids, int ids_bytes, int n, int E,
                                                                void* __restrict__ sorted_out, int32_t* __restrict__ src2dst,
                                                                int64_t* __restrict__ seg_indptr) {
    const int lane = threadIdx.x;
    const bool live = lane < n;
    const int64_t id = live ? ld_id(ids, lane, ids_bytes) : 0;
    const int b = !live ? E + 2 : (id < 0 ? 0 : (id >= E ? E + 1 : (int)id + 1));
    int pos = 0;
    for (int e0 = 0; e0 <= E; e0 += 64) {
        int below = 0;                                   // ids of the buckets up to e0 + lane
        uint64_t todo = __ballot(live);
        while (todo) {
            const int v = __builtin_amdgcn_readlane(b, __ffsll((unsigned long long)todo) - 1);
            const uint64_t m = __ballot(b == v);
            const int c = __popcll(m);
            if (v <= e0 + lane) below += c;
            if (e0 == 0) pos += v < b ? c : (v == b ? __popcll(m & ((1ull << lane) - 1ull)) : 0);
            todo &= ~m;
        }
        const int e = e0 + lane;
        if (e <= E) seg_indptr[e] = e == 0 ? 0 : below;
    }
    if (live) {
        if (ids_bytes == 8) ((int64_t*)sorted_out)[pos] = id; else ((int32_t*)sorted_out)[pos] = (int32_t)id;
        src2dst[lane] = pos;
    }
}

// ---------------------------------------------------------------- softmax top-k router
// L lanes own one token, V experts each (expert v * L + lane), topk <= L; a wave owns 64 / L tokens.  Bound by latency: a token is a few
// dozen bytes, and what the launch costs is one dependent chain (load, max, sum, topk rounds of an arg-max over the lanes),
// so everything stays in registers and lanes.  As five torch kernels the same routing took 31 us of GPU time for 16 tokens
// and 43 us for 4096; one launch here takes 1.9 and 2.8 us back to back, 5.3 and 5.0 in a layer of 8 experts, where its code
// has to be fetched again behind the kernels that streamed the weights.
// A probability is ranked by its bit pattern (monotone for the non-negative values, a NaN above all of them), joined with
// the complement of the index, so equal values go to the lower index and one 64-bit maximum decides a round.
template <int DT, int L, int V>
__global__ __launch_bounds__(256) void softmax_topk_kernel(const void* __restrict__ logits, int64_t* __restrict__ ids,
                                                           float* __restrict__ wts, int64_t T, int E, int topk, bool renorm) {
    const int64_t t = ((int64_t)blockIdx.x * 256 + threadIdx.x) / L;
    const int lane = threadIdx.x & (L - 1);
    const bool live = t < T;
    float x[V];
    float m = -INFINITY;
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const int e = v * L + lane;
        x[v] = (live && e < E) ? FloatIO<DT>::ld(logits, t * E + e) : -INFINITY;
        m = fmaxf(m, x[v]);
    }
#pragma unroll
    for (int o = L / 2; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));      // (signed: group_max is for magnitudes)
    float sum = 0.f;
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const int e = v * L + lane;
        x[v] = e < E ? expf(x[v] - m) : 0.f;
        sum += x[v];
    }
#pragma unroll
    for (int o = L / 2; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
    uint64_t key[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const int e = v * L + lane;
        key[v] = e < E ? ((uint64_t)__float_as_uint(x[v] / sum) << 32) | (uint64_t)(0xffffffffu - (unsigned)e) : 0;
    }
    float total = 0.f, mine = 0.f;                       // lane k keeps the k-th weight (topk <= L)
    unsigned mine_e = 0;
    for (int k = 0; k < topk; ++k) {
        uint64_t best = key[0];
#pragma unroll
        for (int v = 1; v < V; ++v) best = key[v] > best ? key[v] : best;
#pragma unroll
        for (int o = L / 2; o > 0; o >>= 1) {
            const uint64_t other = __shfl_xor((unsigned long long)best, o, 64);
            best = other > best ? other : best;
        }
        const float w = __uint_as_float((unsigned)(best >> 32));
        total += w;
        if (lane == k) { mine = w; mine_e = 0xffffffffu - (unsigned)best; }
#pragma unroll
        for (int v = 0; v < V; ++v) if (key[v] == best) key[v] = 0;
    }
    if (live && lane < topk) {
        ids[t * topk + lane] = (int64_t)mine_e;
        wts[t * topk + lane] = renorm ? mine / total : mine;
    }
}

// one workgroup per token: copy (x * 1/a1_scale[e]) into each destination row of its local experts
template <int IDT, int ODT>
__global__ void pre_reorder_kernel(const void* __restrict__ x, void* __restrict__ out, const int32_t* __restrict__ src2dst,
                                   const void* __restrict__ topk_ids, int ids_bytes, const float* __restrict__ a1_scales,
                                   int start_e, int end_e, int topk, int64_t hidden) {
    const int64_t t = blockIdx.x;
    for (int j = 0; j < topk; ++j) {
        const int64_t e = ld_id(topk_ids, t * topk + j, ids_bytes);
        if (e < start_e || e > end_e) continue;
        const float scale = a1_scales ? 1.0f / a1_scales[e - start_e] : 1.0f;
        const int64_t dst = src2dst[t * topk + j];
        for (int64_t c = threadIdx.x; c < hidden; c += blockDim.x)
            FloatIO<ODT>::st(out, dst * hidden + c, FloatIO<IDT>::ld(x, t * hidden + c) * scale);
    }
}

// groups per thread of the fused activation + quantisation kernel (8192 x 28672 bf16 -> e4m3: 121 us with 1,
// 117 us with 2, 131 us with 4, 146 us with 8)
constexpr int AMQ_UNROLL = 2;

template <int IDT, int ODT>
__global__ void act_and_mul_kernel(const void* __restrict__ gateup, void* __restrict__ out,
                                   const void* __restrict__ reorder_topk_ids, int ids_bytes,
                                   const float* __restrict__ scales, int start_e, int end_e, int64_t two_i, int act) {
    const int64_t row = blockIdx.x;
    const int64_t e = ld_id(reorder_topk_ids, row, ids_bytes);
    if (e < start_e || e > end_e) return;
    const int64_t I = two_i / 2;
    const bool has_scale = scales != nullptr;
    const float scale = has_scale ? rnd<IDT>(1.0f / scales[e - start_e]) : 1.0f;
    for (int64_t c = threadIdx.x; c < I; c += blockDim.x) {
        const float gv = FloatIO<IDT>::ld(gateup, row * two_i + c);
        const float up = FloatIO<IDT>::ld(gateup, row * two_i + I + c);
        const float r = gated_act<IDT>(gv, up, act, has_scale, scale);
        FloatIO<ODT>::st(out, row * I + c, r);
    }
}

// the same with 8 outputs per thread and pass (I a multiple of 8, 16-byte aligned tensors); a thread requests
// the operands of two passes before it converts the first
template <int IDT, int ODT>
__global__ void act_and_mul_vec_kernel(const void* __restrict__ gateup, void* __restrict__ out,
                                       const void* __restrict__ reorder_topk_ids, int ids_bytes,
                                       const float* __restrict__ scales, int start_e, int end_e, int64_t two_i, int act) {
    const int64_t row = blockIdx.x;
    const int64_t e = ld_id(reorder_topk_ids, row, ids_bytes);
    if (e < start_e || e > end_e) return;
    const int64_t I = two_i / 2;
    const bool has_scale = scales != nullptr;
    const float scale = has_scale ? rnd<IDT>(1.0f / scales[e - start_e]) : 1.0f;
    const int64_t step = (int64_t)blockDim.x * EPL;
    for (int64_t c0 = (int64_t)threadIdx.x * EPL; c0 < I; c0 += 2 * step) {
        const int64_t c1 = c0 + step;
        const bool two = c1 < I;
        float gv[2][EPL], up[2][EPL], r[EPL];
        load8<IDT>(gateup, row * two_i + c0, gv[0]);
        load8<IDT>(gateup, row * two_i + I + c0, up[0]);
        if (two) {
            load8<IDT>(gateup, row * two_i + c1, gv[1]);
            load8<IDT>(gateup, row * two_i + I + c1, up[1]);
        }
        gated_act8<IDT>(gv[0], up[0], act, has_scale, scale, r);
        store8<ODT>(out, row * I + c0, r);
        if (two) {
            gated_act8<IDT>(gv[1], up[1], act, has_scale, scale, r);
            store8<ODT>(out, row * I + c1, r);
        }
    }
}

// Gated activation and 1 x 128 activation quantisation in one pass: 16 lanes own one group of 128 outputs,
// 8 each.  The values quantised are exactly those the separate activation kernel would have stored in the
// tensor dtype, so q and s equal those of the two-kernel sequence bit for bit.
// EIGHT: the branch on the activation stands around a thread's eight elements (gated_act8), faster where few waves share a SIMD: elements run beside each
// other there.  With the chip full of waves those do so anyway, and a branch around each element is faster.  us, a branch around each | around
// eight, bf16 to e4m3, SiLU (GELU): 32 x 14336 5.0 (5.05) | 4.6 (4.75), 1024 x 1408 5.5 (5.65) | 5.1 (5.4), 2048 x 2048 7.5 (7.8) | 7.4 (8.1), 8192 x
// 2048 20.5 (21.9) | 21.7 (23.3), 8192 x 14336 121 (131) | 128 (144); to int8 4.4 (4.7) | 4.15 (4.3), 4.95 (5.2) | 4.7 (5.2), 6.9 (7.2) | 6.8 (7.5), 20.0
// (21.7) | 20.7 (23.0), 118 (127) | 123 (139).  The line is two workgroups a CU, between 1024 x 1408 and 2048 x 2048.
template <int IDT, bool FP8, bool EIGHT>
__global__ void act_mul_quant_kernel(const void* __restrict__ gateup, void* __restrict__ q_out, void* __restrict__ s_out,
                                     const void* __restrict__ reorder_topk_ids, int ids_bytes,
                                     const float* __restrict__ scales, int start_e, int end_e, int64_t M, int64_t two_i,
                                     int act, int mode) {
    // a workgroup owns AMQ_UNROLL x 16 consecutive groups; a thread requests the operands of all its groups
    // before it converts the first one
    const int64_t I = two_i / 2, gpr = I / 128;
    const int sub = threadIdx.x & 15;
    int64_t grp[AMQ_UNROLL], row[AMQ_UNROLL], col[AMQ_UNROLL];
    bool live[AMQ_UNROLL];
    float gv[AMQ_UNROLL][EPL], up[AMQ_UNROLL][EPL];
#pragma unroll
    for (int k = 0; k < AMQ_UNROLL; ++k) {
        grp[k] = ((int64_t)blockIdx.x * AMQ_UNROLL + k) * (blockDim.x >> 4) + (threadIdx.x >> 4);
        live[k] = grp[k] < M * gpr;
        const int64_t gs = live[k] ? grp[k] : 0;
        row[k] = gs / gpr;
        col[k] = (gs - row[k] * gpr) * 128 + sub * EPL;
        load8<IDT>(gateup, row[k] * two_i + col[k], gv[k]);
        load8<IDT>(gateup, row[k] * two_i + I + col[k], up[k]);
    }
#pragma unroll
    for (int k = 0; k < AMQ_UNROLL; ++k) {
        const int64_t e = ld_id(reorder_topk_ids, row[k], ids_bytes);
        const bool local = e >= start_e && e <= end_e;
        const bool has_scale = scales != nullptr && local;
        const float scale = has_scale ? rnd<IDT>(1.0f / scales[e - start_e]) : 1.0f;
        float r[EPL];
        float m = 0.f;
        if constexpr (EIGHT) gated_act8<IDT>(gv[k], up[k], act, has_scale, scale, r);
#pragma unroll
        for (int j = 0; j < EPL; ++j) {
            if constexpr (!EIGHT) r[j] = gated_act<IDT>(gv[k][j], up[k][j], act, has_scale, scale);
            m = fmaxf(m, fabsf(r[j]));
        }
        m = group_max<16>(m);
        if (!live[k] || !local) continue;
        quant_store8<FP8>(r, m, q_out, row[k] * I + col[k], s_out, grp[k], sub == 0, mode);
    }
}

// Token permutation and 1 x 128 activation quantisation in one pass: a token's row is read once, quantised
// (after the optional per-expert scale, rounded to the tensor dtype as the separate kernels do) and written
// to the destination row of each of its local experts.  Without per-expert scales the values are the same for
// every expert and are quantised once (bound by HBM then: 4096 tokens x 2 experts x 4096 bf16 19.6 us; quantising per
// expert took 25.8 us).
template <int IDT, bool FP8, bool SCALED>
__global__ void pre_reorder_quant_kernel(const void* __restrict__ x, void* __restrict__ q_out, void* __restrict__ s_out,
                                         const int32_t* __restrict__ src2dst, const void* __restrict__ topk_ids,
                                         int ids_bytes, const float* __restrict__ a1_scales, int start_e, int end_e,
                                         int topk, int64_t T, int64_t hidden, int mode) {
    const int64_t gpr = hidden / 128;
    const int sub = threadIdx.x & 15;
    const int64_t grp = (int64_t)blockIdx.x * (blockDim.x >> 4) + (threadIdx.x >> 4);
    const bool live = grp < T * gpr;
    const int64_t gs = live ? grp : 0;
    const int64_t t = gs / gpr, gi = gs - t * gpr, col = gi * 128 + sub * EPL;
    float v[EPL];
    load8<IDT>(x, t * hidden + col, v);
    float sc = 0.f;
    uint2 w = make_uint2(0, 0);
    if constexpr (!SCALED) {
        float m = 0.f;
#pragma unroll
        for (int k = 0; k < EPL; ++k) m = fmaxf(m, fabsf(v[k]));
        w = quant8<FP8>(v, group_max<16>(m), mode, sc);
    }
    for (int j = 0; j < topk; ++j) {
        const int64_t e = ld_id(topk_ids, t * topk + j, ids_bytes);
        const bool local = e >= start_e && e <= end_e;
        if constexpr (SCALED) {
            const float scale = local ? 1.0f / a1_scales[e - start_e] : 1.0f;
            float u[EPL];
            float m = 0.f;
#pragma unroll
            for (int k = 0; k < EPL; ++k) {
                u[k] = rnd<IDT>(v[k] * scale);
                m = fmaxf(m, fabsf(u[k]));
            }
            w = quant8<FP8>(u, group_max<16>(m), mode, sc);
        }
        if (!live || !local) continue;
        const int64_t dst = src2dst[t * topk + j];
        store_quant8<FP8>(w, sc, q_out, dst * hidden + col, s_out, dst * gpr + gi, sub == 0);
    }
}

template <int DT, int WDT>
__global__ void post_reorder_kernel(const void* __restrict__ down, void* __restrict__ out, const int32_t* __restrict__ src2dst,
                                    const void* __restrict__ topk_ids, int ids_bytes, const void* __restrict__ topk_w,
                                    int start_e, int end_e, int topk, int64_t hidden) {
    const int64_t t = blockIdx.x;
    if constexpr (DT != LLMK_F32) {
        // 16-bit rows of whole 16-byte chunks: 8 columns per lane and load
        if (hidden % EPL == 0 && (((uintptr_t)down | (uintptr_t)out) & 15) == 0) {
            for (int64_t c = (int64_t)threadIdx.x * EPL; c < hidden; c += (int64_t)blockDim.x * EPL) {
                float sum[EPL] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                for (int j = 0; j < topk; ++j) {
                    const int64_t e = ld_id(topk_ids, t * topk + j, ids_bytes);
                    if (e < start_e || e > end_e) continue;
                    const int64_t dst = src2dst[t * topk + j];
                    const float w = rnd<DT>(FloatIO<WDT>::ld(topk_w, t * topk + j));
                    float v[EPL];
                    load8<DT>(down, dst * hidden + c, v);
#pragma unroll
                    for (int k = 0; k < EPL; ++k) sum[k] = rnd<DT>(sum[k] + rnd<DT>(v[k] * w));
                }
                uint4 o;
                if constexpr (DT == LLMK_BF16) {
                    o.x = pack_bf16x2(sum[0], sum[1]); o.y = pack_bf16x2(sum[2], sum[3]);
                    o.z = pack_bf16x2(sum[4], sum[5]); o.w = pack_bf16x2(sum[6], sum[7]);
                } else {
                    o.x = pack_f16x2(sum[0], sum[1]); o.y = pack_f16x2(sum[2], sum[3]);
                    o.z = pack_f16x2(sum[4], sum[5]); o.w = pack_f16x2(sum[6], sum[7]);
                }
                *(uint4*)((unsigned short*)out + t * hidden + c) = o;
            }
            return;
        }
    }
    for (int64_t c = threadIdx.x; c < hidden; c += blockDim.x) {
        float sum = 0.f;
        for (int j = 0; j < topk; ++j) {
            const int64_t e = ld_id(topk_ids, t * topk + j, ids_bytes);
            if (e < start_e || e > end_e) continue;
            const int64_t dst = src2dst[t * topk + j];
            const float w = rnd<DT>(FloatIO<WDT>::ld(topk_w, t * topk + j));
            const float v = FloatIO<DT>::ld(down, dst * hidden + c);
            sum = rnd<DT>(sum + rnd<DT>(v * w));     // product and running sum both live in the tensor dtype
        }
        FloatIO<DT>::st(out, t * hidden + c, sum);
    }
}

// ---------------------------------------------------------------- per-expert scalar scales -> block-scale layout
// scale_a[r, :] = sa[e(r)] for the rows of segment e, scale_b[w, :, :] = sb[w]; rows outside every segment get 0.
// Blocks [0, M) write one activation-scale row each, blocks [M, M + Eb) one expert's weight scales.
template <int SDT>
__global__ void expert_scales_kernel(const float* __restrict__ sa, const float* __restrict__ sb,
                                     const int64_t* __restrict__ seg, int E, int64_t M, int kb, int64_t nbkb,
                                     void* __restrict__ scale_a, void* __restrict__ scale_b) {
    const int64_t blk = blockIdx.x;
    if (blk < M) {
        float v = 0.f;
        for (int e = 0; e < E; ++e)
            if (blk >= seg[e] && blk < seg[e + 1]) { v = sa[e]; break; }
        for (int i = threadIdx.x; i < kb; i += blockDim.x) FloatIO<SDT>::st(scale_a, blk * kb + i, v);
    } else {
        const int64_t w = blk - M;
        const float v = sb[w];
        for (int64_t i = threadIdx.x; i < nbkb; i += blockDim.x) FloatIO<SDT>::st(scale_b, w * nbkb + i, v);
    }
}

}  // namespace

extern "C" int llmk_moe_expert_scales(const float* sa, const float* sb, const int64_t* seg_indptr, int E, int Eb,
                                      int64_t M, int64_t N, int64_t K, void* scale_a, void* scale_b, int s_dtype,
                                      void* stream) {
    if (M < 0 || N < 0 || K < 0 || E < 0 || Eb < 0 || K % 128) LLMK_FAIL(LLMK_ERR_SHAPE, "moe_expert_scales: bad shape");
    if (M + Eb == 0 || K == 0) return LLMK_OK;
    if (!sa || !sb || !seg_indptr || !scale_a || !scale_b) LLMK_FAIL(LLMK_ERR_ARG, "moe_expert_scales: null pointer");
    const int kb = (int)(K / 128);
    const int64_t nbkb = ((N + 127) / 128) * kb;
    LLMK_DISPATCH_FLOAT(s_dtype, SDT, (expert_scales_kernel<SDT><<<(unsigned)(M + Eb), 64, 0, (hipStream_t)stream>>>(
        sa, sb, seg_indptr, E, M, kb, nbkb, scale_a, scale_b)));
    LLMK_CHECK_LAUNCH("moe_expert_scales");
    return LLMK_OK;
}

extern "C" int llmk_moe_seg_indptr(const int64_t* sorted_ids, int64_t* seg_indptr, int64_t num_toks, int num_experts,
                                   void* stream) {
    if (num_experts < 0 || num_toks < 0) LLMK_FAIL(LLMK_ERR_SHAPE, "moe_seg_indptr: negative size");
    if (!seg_indptr || (num_toks && !sorted_ids)) LLMK_FAIL(LLMK_ERR_ARG, "moe_seg_indptr: null pointer");
    if (num_experts == 0) return LLMK_OK;
    seg_indptr_kernel<<<(unsigned)cdiv64(num_experts, 64), 64, 0, (hipStream_t)stream>>>(sorted_ids, seg_indptr, num_toks, num_experts);
    LLMK_CHECK_LAUNCH("moe_seg_indptr");
    return LLMK_OK;
}

extern "C" int llmk_moe_src2dst(const int64_t* reorder_ids, int32_t* src2dst, int64_t num_toks, void* stream) {
    if (num_toks < 0) LLMK_FAIL(LLMK_ERR_SHAPE, "moe_src2dst: negative size");
    if (num_toks == 0) return LLMK_OK;
    if (!reorder_ids || !src2dst) LLMK_FAIL(LLMK_ERR_ARG, "moe_src2dst: null pointer");
    src2dst_kernel<<<(unsigned)cdiv64(num_toks, 256), 256, 0, (hipStream_t)stream>>>(reorder_ids, src2dst, num_toks);
    LLMK_CHECK_LAUNCH("moe_src2dst");
    return LLMK_OK;
}

extern "C" int llmk_moe_ep_preprocess(const void* topk_ids, int ids_bytes, int64_t num_toks, int num_experts,
                                      void* sorted_ids, int32_t* src2dst, int64_t* seg_indptr, void* stream) {
    if (num_experts < 0 || num_toks < 0) LLMK_FAIL(LLMK_ERR_SHAPE, "moe_ep_preprocess: negative size");
    if (num_experts > LLMK_MOE_PREPROCESS_MAX_EXPERTS || num_toks > LLMK_MOE_PREPROCESS_MAX_IDS)
        LLMK_FAIL(LLMK_ERR_SHAPE, "moe_ep_preprocess: %lld ids of %d experts exceed the limits %d / %d of the one-launch sort",
                  (long long)num_toks, num_experts, LLMK_MOE_PREPROCESS_MAX_IDS, LLMK_MOE_PREPROCESS_MAX_EXPERTS);
    if (ids_bytes != 4 && ids_bytes != 8) LLMK_FAIL(LLMK_ERR_DTYPE, "moe_ep_preprocess: ids_bytes %d", ids_bytes);
    if (!seg_indptr || (num_toks && (!topk_ids || !sorted_ids || !src2dst))) LLMK_FAIL(LLMK_ERR_ARG, "moe_ep_preprocess: null pointer");
    static_assert(LLMK_MOE_PREPROCESS_MAX_EXPERTS == PP_MAX_EXPERTS, "header limit and kernel table size differ");
    const unsigned grid = (unsigned)(num_toks > 0 ? cdiv64(num_toks, PP_THREADS) : 1);
    // one workgroup of the smallest size that holds the ids, chunks of PP_THREADS beyond
    if (num_toks <= 64) ep_preprocess_wave_kernel<<<1, 64, 0, (hipStream_t)stream>>>(topk_ids, ids_bytes, (int)num_toks, num_experts, sorted_ids, src2dst, seg_indptr);
    else if (num_toks <= 256) ep_preprocess_one_kernel<256><<<1, 256, 0, (hipStream_t)stream>>>(topk_ids, ids_bytes, (int)num_toks, num_experts, sorted_ids, src2dst, seg_indptr);
    else if (num_toks <= PP_THREADS) ep_preprocess_one_kernel<PP_THREADS><<<1, PP_THREADS, 0, (hipStream_t)stream>>>(topk_ids, ids_bytes, (int)num_toks, num_experts, sorted_ids, src2dst, seg_indptr);
    else ep_preprocess_kernel<<<grid, PP_THREADS, 0, (hipStream_t)stream>>>(topk_ids, ids_bytes, (int)num_toks, num_experts, sorted_ids, src2dst, seg_indptr);
    LLMK_CHECK_LAUNCH("moe_ep_preprocess");
    return LLMK_OK;
}

template <int DT>
static int launch_router(const void* logits_all, int64_t* ids_all, float* w_all, int64_t T_all, int E, int topk, bool renorm, hipStream_t st) {
    // the narrowest group of lanes that holds a token's experts one each, then more experts per lane; 2^24 tokens a launch
    // (64 lanes each are a quarter of the 2^32 threads a grid may have)
    constexpr int64_t ROWS = 1ll << 24;
    for (int64_t t0 = 0; t0 < T_all; t0 += ROWS) {
        const void* logits = (const uint8_t*)logits_all + t0 * E * (DT == LLMK_F32 ? 4 : 2);
        int64_t* ids = ids_all + t0 * topk;
        float* w = w_all + t0 * topk;
        const int64_t T = std::min(ROWS, T_all - t0);
#define CALL(L, V) softmax_topk_kernel<DT, L, V><<<(unsigned)cdiv64(T * L, 256), 256, 0, st>>>(logits, ids, w, T, E, topk, renorm)
        if (E <= 8) CALL(8, 1);
        else if (E <= 16) CALL(16, 1);
        else if (E <= 32) CALL(32, 1);
        else if (E <= 64) CALL(64, 1);
        else if (E <= 128) CALL(64, 2);
        else if (E <= 256) CALL(64, 4);
        else CALL(64, 8);
#undef CALL
        LLMK_CHECK_LAUNCH("moe_softmax_topk");
    }
    return LLMK_OK;
}

extern "C" int llmk_moe_softmax_topk(const void* logits, int dtype, int64_t* ids, float* weights, int64_t T, int E, int topk,
                                     int renormalize, void* stream) {
    if (T < 0 || E < 1 || topk < 1 || topk > E || E > LLMK_ROUTER_MAX_EXPERTS || topk > LLMK_ROUTER_MAX_TOPK)
        LLMK_FAIL(LLMK_ERR_SHAPE, "moe_softmax_topk: T=%lld E=%d topk=%d", (long long)T, E, topk);
    if (T == 0) return LLMK_OK;
    if (!logits || !ids || !weights) LLMK_FAIL(LLMK_ERR_ARG, "moe_softmax_topk: null pointer");
    int rc = LLMK_OK;
    LLMK_DISPATCH_FLOAT(dtype, DT, rc = launch_router<DT>(logits, ids, weights, T, E, topk, renormalize != 0, (hipStream_t)stream));
    return rc;
}

extern "C" int llmk_moe_pre_reorder(const void* x, int x_dtype, void* out, int out_dtype, const int32_t* src2dst,
                                    const void* topk_ids, int ids_bytes, const float* a1_scales, int start_expert,
                                    int end_expert, int topk, int64_t T, int64_t hidden, void* stream) {
    if (T < 0 || hidden < 0 || topk < 0) LLMK_FAIL(LLMK_ERR_SHAPE, "moe_pre_reorder: negative size");
    if (ids_bytes != 4 && ids_bytes != 8) LLMK_FAIL(LLMK_ERR_DTYPE, "moe_pre_reorder: ids_bytes %d", ids_bytes);
    if (T == 0 || hidden == 0 || topk == 0) return LLMK_OK;
    if (!x || !out || !src2dst || !topk_ids) LLMK_FAIL(LLMK_ERR_ARG, "moe_pre_reorder: null pointer");
    LLMK_DISPATCH_FLOAT(x_dtype, IDT, LLMK_DISPATCH_FLOAT(out_dtype, ODT,
        (pre_reorder_kernel<IDT, ODT><<<(unsigned)T, 256, 0, (hipStream_t)stream>>>(x, out, src2dst, topk_ids, ids_bytes, a1_scales, start_expert, end_expert, topk, hidden))));
    LLMK_CHECK_LAUNCH("moe_pre_reorder");
    return LLMK_OK;
}

extern "C" int llmk_moe_act_and_mul(const void* gateup, int in_dtype, void* out, int out_dtype,
                                    const void* reorder_topk_ids, int ids_bytes, const float* scales, int start_expert,
                                    int end_expert, int64_t M, int64_t two_i, int act, void* stream) {
    if (M < 0 || two_i < 0 || two_i % 2) LLMK_FAIL(LLMK_ERR_SHAPE, "moe_act_and_mul: bad shape");
    if (ids_bytes != 4 && ids_bytes != 8) LLMK_FAIL(LLMK_ERR_DTYPE, "moe_act_and_mul: ids_bytes %d", ids_bytes);
    if (act != 0 && act != 1) LLMK_FAIL(LLMK_ERR_DTYPE, "moe_act_and_mul: act %d", act);
    if (M == 0 || two_i == 0) return LLMK_OK;
    if (!gateup || !out || !reorder_topk_ids) LLMK_FAIL(LLMK_ERR_ARG, "moe_act_and_mul: null pointer");
    const int in_al = in_dtype == LLMK_F32 ? 31 : 15, out_al = out_dtype == LLMK_F32 ? 31 : 15;
    if ((two_i / 2) % 8 == 0 && ((uintptr_t)gateup & in_al) == 0 && ((uintptr_t)out & out_al) == 0) {
        LLMK_DISPATCH_FLOAT(in_dtype, IDT, LLMK_DISPATCH_FLOAT(out_dtype, ODT,
            (act_and_mul_vec_kernel<IDT, ODT><<<(unsigned)M, 256, 0, (hipStream_t)stream>>>(gateup, out, reorder_topk_ids, ids_bytes, scales, start_expert, end_expert, two_i, act))));
        LLMK_CHECK_LAUNCH("moe_act_and_mul");
        return LLMK_OK;
    }
    LLMK_DISPATCH_FLOAT(in_dtype, IDT, LLMK_DISPATCH_FLOAT(out_dtype, ODT,
        (act_and_mul_kernel<IDT, ODT><<<(unsigned)M, 256, 0, (hipStream_t)stream>>>(gateup, out, reorder_topk_ids, ids_bytes, scales, start_expert, end_expert, two_i, act))));
    LLMK_CHECK_LAUNCH("moe_act_and_mul");
    return LLMK_OK;
}

extern "C" int llmk_moe_act_and_mul_quant(const void* gateup, int in_dtype, void* q_out, void* s_out, int kind,
                                          int round_mode, const void* reorder_topk_ids, int ids_bytes,
                                          const float* scales, int start_expert, int end_expert, int64_t M,
                                          int64_t two_i, int act, void* stream) {
    if (M < 0 || two_i < 0 || two_i % 256) LLMK_FAIL(LLMK_ERR_SHAPE, "moe_act_and_mul_quant: 2I=%lld must be a multiple of 256", (long long)two_i);
    if (ids_bytes != 4 && ids_bytes != 8) LLMK_FAIL(LLMK_ERR_DTYPE, "moe_act_and_mul_quant: ids_bytes %d", ids_bytes);
    if (act != 0 && act != 1) LLMK_FAIL(LLMK_ERR_DTYPE, "moe_act_and_mul_quant: act %d", act);
    if (kind != LLMK_KIND_I8 && kind != LLMK_KIND_FP8) LLMK_FAIL(LLMK_ERR_DTYPE, "moe_act_and_mul_quant: kind %d", kind);
    if (round_mode != LLMK_ROUND_HALF_AWAY && round_mode != LLMK_ROUND_HALF_UP) LLMK_FAIL(LLMK_ERR_DTYPE, "moe_act_and_mul_quant: round_mode %d", round_mode);
    if (in_dtype == LLMK_F32) LLMK_FAIL(LLMK_ERR_DTYPE, "moe_act_and_mul_quant: fp16 / bf16 inputs only");
    if (M == 0 || two_i == 0) return LLMK_OK;
    if (!gateup || !q_out || !s_out || !reorder_topk_ids) LLMK_FAIL(LLMK_ERR_ARG, "moe_act_and_mul_quant: null pointer");
    if (((uintptr_t)gateup | (uintptr_t)q_out) & 15) LLMK_FAIL(LLMK_ERR_ARG, "moe_act_and_mul_quant: buffers must be 16-byte aligned");
    const int64_t threads = M * (two_i / 256) * 16;
    const unsigned grid = (unsigned)cdiv64(threads, 256 * AMQ_UNROLL);
    const bool eight = grid <= 2 * LLMK_CUS;
#define CALL(FP8, EIGHT) act_mul_quant_kernel<IDT, FP8, EIGHT><<<grid, 256, 0, (hipStream_t)stream>>>(gateup, q_out, s_out, reorder_topk_ids, ids_bytes, scales, start_expert, end_expert, M, two_i, act, round_mode)
    LLMK_DISPATCH_FLOAT(in_dtype, IDT, {
        if (kind == LLMK_KIND_FP8) { if (eight) CALL(true, true); else CALL(true, false); }
        else { if (eight) CALL(false, true); else CALL(false, false); }
    });
#undef CALL
    LLMK_CHECK_LAUNCH("moe_act_and_mul_quant");
    return LLMK_OK;
}

extern "C" int llmk_moe_pre_reorder_quant(const void* x, int x_dtype, void* q_out, void* s_out, int kind, int round_mode,
                                          const int32_t* src2dst, const void* topk_ids, int ids_bytes,
                                          const float* a1_scales, int start_expert, int end_expert, int topk,
                                          int64_t T, int64_t hidden, void* stream) {
    if (T < 0 || hidden < 0 || topk < 0 || hidden % 128) LLMK_FAIL(LLMK_ERR_SHAPE, "moe_pre_reorder_quant: hidden=%lld must be a multiple of 128", (long long)hidden);
    if (ids_bytes != 4 && ids_bytes != 8) LLMK_FAIL(LLMK_ERR_DTYPE, "moe_pre_reorder_quant: ids_bytes %d", ids_bytes);
    if (kind != LLMK_KIND_I8 && kind != LLMK_KIND_FP8) LLMK_FAIL(LLMK_ERR_DTYPE, "moe_pre_reorder_quant: kind %d", kind);
    if (round_mode != LLMK_ROUND_HALF_AWAY && round_mode != LLMK_ROUND_HALF_UP) LLMK_FAIL(LLMK_ERR_DTYPE, "moe_pre_reorder_quant: round_mode %d", round_mode);
    if (x_dtype == LLMK_F32) LLMK_FAIL(LLMK_ERR_DTYPE, "moe_pre_reorder_quant: fp16 / bf16 inputs only");
    if (T == 0 || hidden == 0 || topk == 0) return LLMK_OK;
    if (!x || !q_out || !s_out || !src2dst || !topk_ids) LLMK_FAIL(LLMK_ERR_ARG, "moe_pre_reorder_quant: null pointer");
    if (((uintptr_t)x | (uintptr_t)q_out) & 15) LLMK_FAIL(LLMK_ERR_ARG, "moe_pre_reorder_quant: buffers must be 16-byte aligned");
    const int64_t threads = T * (hidden / 128) * 16;
    const unsigned grid = (unsigned)cdiv64(threads, 256);
#define CALL(FP8, SCALED) pre_reorder_quant_kernel<IDT, FP8, SCALED><<<grid, 256, 0, (hipStream_t)stream>>>(x, q_out, s_out, src2dst, topk_ids, ids_bytes, a1_scales, start_expert, end_expert, topk, T, hidden, round_mode)
    LLMK_DISPATCH_FLOAT(x_dtype, IDT, {
        if (kind == LLMK_KIND_FP8) { if (a1_scales) CALL(true, true); else CALL(true, false); }
        else { if (a1_scales) CALL(false, true); else CALL(false, false); }
    });
#undef CALL
    LLMK_CHECK_LAUNCH("moe_pre_reorder_quant");
    return LLMK_OK;
}

extern "C" int llmk_moe_post_reorder(const void* down_out, void* out, int dtype, const int32_t* src2dst,
                                     const void* topk_ids, int ids_bytes, const void* topk_weights, int w_dtype,
                                     int start_expert, int end_expert, int topk, int64_t T, int64_t hidden,
                                     void* stream) {
    if (T < 0 || hidden < 0 || topk < 0) LLMK_FAIL(LLMK_ERR_SHAPE, "moe_post_reorder: negative size");
    if (ids_bytes != 4 && ids_bytes != 8) LLMK_FAIL(LLMK_ERR_DTYPE, "moe_post_reorder: ids_bytes %d", ids_bytes);
    if (T == 0 || hidden == 0) return LLMK_OK;
    if (!down_out || !out || !src2dst || !topk_ids || !topk_weights) LLMK_FAIL(LLMK_ERR_ARG, "moe_post_reorder: null pointer");
    LLMK_DISPATCH_FLOAT(dtype, DT, LLMK_DISPATCH_FLOAT(w_dtype, WDT,
        (post_reorder_kernel<DT, WDT><<<(unsigned)T, 256, 0, (hipStream_t)stream>>>(down_out, out, src2dst, topk_ids, ids_bytes, topk_weights, start_expert, end_expert, topk, hidden))));
    LLMK_CHECK_LAUNCH("moe_post_reorder");
    return LLMK_OK;
}

// Tile kernels when the average segment is longer than 64 rows, and from two rows per expert up when the
// expert weights are large (measured on 8 experts of 4096 x 14336, whole forward, tile vs weight-streaming
// kernel: 256 vs 158 us at 1 token, 295 vs 289 us at 8, 344 vs 374 us at 16, 362 vs 481 us at 64).
// Also with several short segments: the weight-streaming kernel spreads its workgroups over the row tiles and
// leaves each of them a fraction of the column workgroups (measured: tile kernels faster from six row tiles).
static bool grouped_tiles(const DirectArgs& p) {
    return p.M > 64 * (int64_t)p.E || (p.M > 2 * (int64_t)p.E && (int64_t)p.N * p.K >= ((int64_t)20 << 20)) || grouped_row_tiles(p.M, p.E, 16) >= 6;
}

extern "C" int llmk_grouped_gemm_duo_rows(int E, int64_t M, int64_t N, int64_t K) {
    if (E <= 0 || M <= 0 || N <= 0 || K <= 0 || K % 128 || M > 0x7fffffff || N > 0x7fffffff || K > 0x7fffffff) return 0;
    DirectArgs p{};
    p.M = (int)M; p.N = (int)N; p.K = (int)K; p.E = E;
    return grouped_tiles(p) ? 32 * grouped_duo_mi(p) : 0;
}

extern "C" int llmk_grouped_gemm(const void* a, const void* b, void* c, int kind, int c_dtype, int E, int64_t M,
                                 int64_t N, int64_t K, const int64_t* seg_indptr, const int64_t* weight_indices,
                                 const void* scale_a, const void* scale_b, int s_dtype, void* workspace,
                                 int64_t workspace_bytes, void* stream) {
    if (M < 0 || N < 0 || K < 0 || E < 0) LLMK_FAIL(LLMK_ERR_SHAPE, "grouped_gemm: negative dimension");
    if (c_dtype != LLMK_F32 && c_dtype != LLMK_F16 && c_dtype != LLMK_BF16) LLMK_FAIL(LLMK_ERR_DTYPE, "grouped_gemm: c_dtype %d", c_dtype);
    const bool scaled = (kind == LLMK_KIND_I8 || kind == LLMK_KIND_FP8);
    const int kstep = scaled ? 128 : 64;
    if (K % kstep) LLMK_FAIL(LLMK_ERR_SHAPE, "grouped_gemm: K=%lld must be a multiple of %d for this element kind", (long long)K, kstep);
    if (M > 0x7fffffff || N > 0x7fffffff || K > 0x7fffffff) LLMK_FAIL(LLMK_ERR_SHAPE, "grouped_gemm: dimension exceeds int32");
    if (M == 0 || N == 0 || E == 0) return LLMK_OK;
    if (!a || !b || !c || !seg_indptr) LLMK_FAIL(LLMK_ERR_ARG, "grouped_gemm: null pointer");
    if (scaled && (!scale_a || !scale_b)) LLMK_FAIL(LLMK_ERR_ARG, "grouped_gemm: block scales required for int8 / fp8 operands");
    if ((((uintptr_t)a) | ((uintptr_t)b)) & 15) LLMK_FAIL(LLMK_ERR_ARG, "grouped_gemm: operands must be 16-byte aligned");
    DirectArgs p{};
    p.a = (const uint8_t*)a; p.b = (const uint8_t*)b; p.c = c; p.a_s = scale_a; p.b_s = scale_b;
    p.seg_indptr = seg_indptr; p.weight_indices = weight_indices;
    p.c_dtype = c_dtype; p.s_dtype = s_dtype; p.M = (int)M; p.N = (int)N; p.K = (int)K; p.E = E;
    hipStream_t st = (hipStream_t)stream;
    const bool big = grouped_tiles(p);
    const int duo = big && scaled && (kind == LLMK_KIND_I8 || s_dtype == LLMK_F32) ? grouped_duo_mi(p) : 0;
    if (duo && kind == LLMK_KIND_FP8) return launch_grouped_duo<K_FP8_BLOCK, false>(p, duo, st, "grouped_gemm(fp8, duo)");
    if (duo && s_dtype == LLMK_F32) return launch_grouped_duo<K_I8_BLOCK, false>(p, duo, st, "grouped_gemm(i8, duo)");
    if (duo) return launch_grouped_duo<K_I8_BLOCK, true>(p, duo, st, "grouped_gemm(i8, duo)");
    if (big && kind == LLMK_KIND_I8) return launch_big<K_I8_BLOCK, true>(p, workspace, workspace_bytes, st, "grouped_gemm(i8, tiled)");
    if (big && kind == LLMK_KIND_FP8) return launch_big<K_FP8_BLOCK, true>(p, workspace, workspace_bytes, st, "grouped_gemm(fp8, tiled)");
    if (big && kind == LLMK_KIND_F16 && dma_eligible(p, 2)) return launch_big_half<K_F16, true>(p, st, "grouped_gemm(f16, tiled)");
    if (big && kind == LLMK_KIND_BF16 && dma_eligible(p, 2)) return launch_big_half<K_BF16, true>(p, st, "grouped_gemm(bf16, tiled)");
    switch (kind) {
        case LLMK_KIND_I8:   return launch_direct<K_I8_BLOCK, true>(p, (int)M, st, "grouped_gemm(i8)");
        case LLMK_KIND_FP8:  return launch_direct<K_FP8_BLOCK, true>(p, (int)M, st, "grouped_gemm(fp8)");
        case LLMK_KIND_F16:  return launch_direct<K_F16, true>(p, (int)M, st, "grouped_gemm(f16)");
        case LLMK_KIND_BF16: return launch_direct<K_BF16, true>(p, (int)M, st, "grouped_gemm(bf16)");
        default: LLMK_FAIL(LLMK_ERR_DTYPE, "grouped_gemm: kind %d", kind);
    }
}

// which tile kernel the gated-activation form would run on for this shape: 8 / 4 = tile rows per wave of the 256-column
// kernel, 0 = none (the caller runs the grouped GEMM and the activation kernel instead)
static int swiglu_tile_rows(int kind, const DirectArgs& p, TileChoice* tile = nullptr) {
    if (p.N % 256 || p.K % 128 || !dma_eligible(p)) return 0;
    if (!grouped_tiles(p)) return 0;
    const TileChoice c = kind == LLMK_KIND_FP8 ? dma_tile_estimate<K_FP8_BLOCK, true>(p) : dma_tile_estimate<K_I8_BLOCK, true>(p);
    if (tile) *tile = c;
    return c.choice == 8 ? 8 : (c.choice == 9 ? 4 : 0);
}

extern "C" int llmk_grouped_gemm_swiglu_quant_fused(int kind, int E, int64_t M, int64_t two_i, int64_t K) {
    if ((kind != LLMK_KIND_I8 && kind != LLMK_KIND_FP8) || E <= 0 || M <= 0 || two_i <= 0 || K <= 0) return 0;
    if (M > 0x7fffffff || two_i > 0x7fffffff || K > 0x7fffffff) return 0;
    DirectArgs p{};
    p.M = (int)M; p.N = (int)two_i; p.K = (int)K; p.E = E;
    return swiglu_tile_rows(kind, p) ? 1 : 0;
}

extern "C" int llmk_grouped_gemm_swiglu_quant(const void* a, const void* b, void* q_out, void* s_out, int kind, int mid_dtype,
                                              int round_mode, int E, int64_t M, int64_t two_i, int64_t K,
                                              const int64_t* seg_indptr, const int64_t* weight_indices, const void* scale_a,
                                              const void* scale_b, int s_dtype, int act, void* workspace,
                                              int64_t workspace_bytes, void* stream) {
    if (M < 0 || two_i < 0 || K < 0 || E < 0) LLMK_FAIL(LLMK_ERR_SHAPE, "grouped_gemm_swiglu_quant: negative dimension");
    if (kind != LLMK_KIND_I8 && kind != LLMK_KIND_FP8) LLMK_FAIL(LLMK_ERR_DTYPE, "grouped_gemm_swiglu_quant: kind %d", kind);
    if (mid_dtype != LLMK_F16 && mid_dtype != LLMK_BF16) LLMK_FAIL(LLMK_ERR_DTYPE, "grouped_gemm_swiglu_quant: mid_dtype %d (the dtype the gate / up sums are rounded to: fp16 or bf16)", mid_dtype);
    if (act != 0 && act != 1) LLMK_FAIL(LLMK_ERR_ARG, "grouped_gemm_swiglu_quant: act %d", act);
    if (round_mode != LLMK_ROUND_HALF_AWAY && round_mode != LLMK_ROUND_HALF_UP) LLMK_FAIL(LLMK_ERR_DTYPE, "grouped_gemm_swiglu_quant: round_mode %d", round_mode);
    if (M > 0x7fffffff || two_i > 0x7fffffff || K > 0x7fffffff) LLMK_FAIL(LLMK_ERR_SHAPE, "grouped_gemm_swiglu_quant: dimension exceeds int32");
    if (M == 0 || two_i == 0 || E == 0) return LLMK_OK;
    if (!a || !b || !q_out || !s_out || !seg_indptr || !scale_a || !scale_b) LLMK_FAIL(LLMK_ERR_ARG, "grouped_gemm_swiglu_quant: null pointer");
    if ((((uintptr_t)a) | ((uintptr_t)b)) & 15 || ((uintptr_t)q_out & 7)) LLMK_FAIL(LLMK_ERR_ARG, "grouped_gemm_swiglu_quant: operands must be 16-byte aligned, q_out 8-byte aligned");
    DirectArgs p{};
    p.a = (const uint8_t*)a; p.b = (const uint8_t*)b; p.c = q_out; p.q_scale = s_out; p.a_s = scale_a; p.b_s = scale_b;
    p.seg_indptr = seg_indptr; p.weight_indices = weight_indices;
    p.c_dtype = mid_dtype; p.s_dtype = s_dtype; p.M = (int)M; p.N = (int)two_i; p.K = (int)K; p.E = E;
    p.act = act; p.round_mode = round_mode;
    TileChoice tile{};
    const int rows = swiglu_tile_rows(kind, p, &tile);
    if (!rows) LLMK_FAIL(LLMK_ERR_SHAPE, "grouped_gemm_swiglu_quant: shape E=%d M=%lld 2I=%lld K=%lld is not one the fused kernel takes (ask llmk_grouped_gemm_swiglu_quant_fused first)", E, (long long)M, (long long)two_i, (long long)K);
    hipStream_t st = (hipStream_t)stream;
    if (s_dtype != LLMK_F32) {
        // 16-bit activation scales are widened first, as in front of the plain kernel, fp16 ones of int8 operands where that is worth it and there is room
        const int64_t n = M * (K >> 7);
        const bool room = workspace && workspace_bytes >= n * 4 && !((uintptr_t)workspace & 15);
        const unsigned blocks = (unsigned)cdiv64(n, 256);
        if (kind == LLMK_KIND_I8 && wide_f16_scales(tile, p.K, s_dtype, room))
            return rows == 8 ? launch_wide_swiglu<K_I8_BLOCK, 8, LLMK_F16>(p, st, "grouped_gemm_swiglu_quant(i8)") : launch_wide_swiglu<K_I8_BLOCK, 4, LLMK_F16>(p, st, "grouped_gemm_swiglu_quant(i8)");
        if (!room) LLMK_FAIL(LLMK_ERR_ARG, "grouped_gemm_swiglu_quant: 16-bit activation scales need %lld bytes of workspace", (long long)(n * 4));
        if (s_dtype == LLMK_F16) scales_to_f32_kernel<LLMK_F16><<<blocks, 256, 0, st>>>(scale_a, (float*)workspace, n);
        else if (s_dtype == LLMK_BF16) scales_to_f32_kernel<LLMK_BF16><<<blocks, 256, 0, st>>>(scale_a, (float*)workspace, n);
        else LLMK_FAIL(LLMK_ERR_DTYPE, "grouped_gemm_swiglu_quant: s_dtype %d", s_dtype);
        LLMK_CHECK_LAUNCH("grouped_gemm_swiglu_quant(scales)");
        p.a_s = workspace;
    }
    if (kind == LLMK_KIND_FP8)
        return rows == 8 ? launch_wide_swiglu<K_FP8_BLOCK, 8>(p, st, "grouped_gemm_swiglu_quant(fp8)") : launch_wide_swiglu<K_FP8_BLOCK, 4>(p, st, "grouped_gemm_swiglu_quant(fp8)");
    return rows == 8 ? launch_wide_swiglu<K_I8_BLOCK, 8>(p, st, "grouped_gemm_swiglu_quant(i8)") : launch_wide_swiglu<K_I8_BLOCK, 4>(p, st, "grouped_gemm_swiglu_quant(i8)");
}

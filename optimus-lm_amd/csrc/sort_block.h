// A stable counting sort of a few (token, k) pairs by local expert, by one block: what sort.hip's one-launch forms and the router that
// sorts its own selections (route.hip) have in common.
#pragma once
#include "common.h"

namespace {

// Mask of the lanes of this wavefront that hold the same key (keys < 2^nbits).
__device__ __forceinline__ unsigned long long match_key(int key, int nbits) {
    unsigned long long m = ~0ull;
    for (int b = 0; b < nbits; b++) {
        const unsigned long long vote = __ballot((key >> b) & 1);
        m &= ((key >> b) & 1) ? vote : ~vote;
    }
    return m;
}

__device__ __forceinline__ unsigned long long lanemask_lt(int lane) { return (1ull << lane) - 1ull; }

// Inclusive prefix sum over the 64 lanes of a wavefront.
__device__ __forceinline__ int wave_incl_scan(int v, int lane) {
    for (int o = 1; o < 64; o <<= 1) {
        const int u = __shfl_up(v, o, 64);
        if (lane >= o) v += u;
    }
    return v;
}

inline int key_bits(int NR) {  // keys 0..NR (NR = "not local")
    int b = 1;
    while ((1 << b) <= NR) b++;
    return b;
}

// Few pairs: count, scan and scatter by one block, in one launch.  A thread keeps its pair's key, weight and rank in registers between the
// passes.  A decode batch or a small training batch spends nothing on bandwidth here, only on latencies.  So pairs past the end are read
// as the last one, not behind a condition, and the rank of a pair within its expert comes from the counting pass.
constexpr int SORT_BLOCK_MAX_NR = 256;
// Of a block that sorts some of the pairs: the first of them, and how many pairs of an expert come before the first and after the last, as
// SPREAD_COPIES counts each that are added up here.
constexpr int SPREAD_COPIES = 8;
struct SpreadPart {
    int first;
    const int *before, *after;   // LDS, [expert][SPREAD_COPIES]
};
// e and weight: of this thread's pair; past the last pair anything.  SPREAD: the block sorts the pairs from part.first on, otherwise all of
// them.
constexpr int SORT_BLOCK_WAVES = 16, SORT_BLOCK_PAIRS = SORT_BLOCK_WAVES * 64;
template <bool SPREAD = false, typename TI>
__device__ __forceinline__ void sort_block(const TI e, const float weight, int n_pairs, int K, int start, int end, int NR, int nbits,
                                           int32_t *__restrict__ cum_token_counts, int32_t *__restrict__ cum_expert_counts_ep,
                                           int32_t *__restrict__ input_indices, int32_t *__restrict__ output_indices,
                                           int32_t *__restrict__ selected_experts_indices, float *__restrict__ row_weights,
                                           const SpreadPart part = {}) {
    constexpr int WAVES = SORT_BLOCK_WAVES;
    __shared__ int off[WAVES][SORT_BLOCK_MAX_NR];   // counts, then the first position of a wavefront's rows of an expert
    __shared__ __attribute__((aligned(16))) int wave_hits[WAVES], chunk_total[SORT_BLOCK_MAX_NR / 64];
    __shared__ int kept_total, kept_before[SORT_BLOCK_MAX_NR / 64];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int j = (SPREAD ? part.first : 0) + tid;
    volatile int *mine = off[wv];
    for (int i = lane; i < NR; i += 64) mine[i] = 0;
    __builtin_amdgcn_wave_barrier();
    const long long v = static_cast<long long>(e);
    const bool kept = j < n_pairs && v >= start && v < end;
    const int key = kept ? static_cast<int>(v - start) : NR;
    const unsigned long long m = match_key(key, nbits), all = __ballot(kept);
    const int rank = __popcll(m & lanemask_lt(lane));
    if (kept && (__ffsll(static_cast<long long>(m)) - 1) == lane) mine[key] = __popcll(m);
    if (lane == 0) wave_hits[wv] = __popcll(all);
    __syncthreads();
    // thread e: expert e's total over the wavefronts, exclusive positions of the wavefronts within it
    int total = 0, ahead = 0, at[WAVES];   // ahead: SPREAD, the expert's pairs before this block's
    if (tid < NR) {
#pragma unroll
        for (int w = 0; w < WAVES; w++) at[w] = off[w][tid];
#pragma unroll
        for (int w = 0; w < WAVES; w++) {
            const int c = at[w];
            at[w] = total;
            total += c;
        }
        if (SPREAD) {
#pragma unroll
            for (int x = 0; x < SPREAD_COPIES; x++) {
                ahead += part.before[tid * SPREAD_COPIES + x];
                total += part.after[tid * SPREAD_COPIES + x];
            }
            total += ahead;
        }
    }
    if (SPREAD && tid < SORT_BLOCK_MAX_NR) {
        const int kept_ahead = wave_sum_i(ahead);
        if (lane == 0) kept_before[wv] = kept_ahead;
    }
    const int incl = wave_incl_scan(total, lane);
    if (tid < SORT_BLOCK_MAX_NR && lane == 63) chunk_total[wv] = incl;
    __syncthreads();
    int before = incl - total;   // rows of the experts before this one
#pragma unroll
    for (int w = 0; w < SORT_BLOCK_MAX_NR / 64; w++) before += w < wv ? chunk_total[w] : 0;
    if (tid < NR) {
#pragma unroll
        for (int w = 0; w < WAVES; w++) off[w][tid] = before + ahead + at[w];
        const bool first = !SPREAD || part.first == 0;
        if (first) cum_token_counts[tid] = before;
        if (tid == NR - 1) {
            if (first) {
                cum_token_counts[NR] = before + total;
                cum_expert_counts_ep[n_pairs / K] = before + total;
            }
            kept_total = before + total;
        }
    }
    __syncthreads();
    int oi = __popcll(all & lanemask_lt(lane));   // kept pairs before this one: of its wavefront, the block and the blocks before
#pragma unroll
    for (int w = 0; w < WAVES; w++) oi += w < wv ? wave_hits[w] : 0;
    if (SPREAD) {
#pragma unroll
        for (int w = 0; w < SORT_BLOCK_MAX_NR / 64; w++) oi += kept_before[w];
    }
    if (j >= n_pairs) return;
    if (j >= kept_total) {   // past the kept pairs: see sort_scatter_kernel
        output_indices[j] = -1;
        input_indices[j] = 0;
        selected_experts_indices[j] = 0;
    }
    const uint32_t t = static_cast<uint32_t>(j) / static_cast<uint32_t>(K);
    const int k = j - static_cast<int>(t) * K;
    if (k == 0) cum_expert_counts_ep[t] = oi;
    if (kept) {
        const int pos = off[wv][key] + rank;
        input_indices[pos] = static_cast<int32_t>(t);
        output_indices[oi] = pos;
        selected_experts_indices[oi] = k;
        if (row_weights) row_weights[pos] = weight;
    }
}

}  // namespace

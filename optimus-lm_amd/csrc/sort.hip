// Token permutation for the fast MoE block: a stable counting sort of the (token, k) pairs by
// local expert, producing exactly the arrays the reference builds with its two index kernels and
// two cumsums.  Up to 65536 pairs are one launch: of one block up to 1024 (sort_small_kernel), of a block for every 1024 beyond
// (sort_spread_kernel); more pairs, or more than 256 local experts, are three:
//   count   — every block histograms its chunk of pairs per expert (wave ballots -> LDS);
//   scan    — one block (16 wavefront-wide scans at a time) turns the [block][expert] table into exclusive offsets in
//             (expert-major, block-minor) order = the stable order, and writes cum_token_counts;
//   scatter — every block re-reads its chunk and places each pair at offset + stable rank.
// Ranks come from wavefront ballots (lanes holding the same expert form a mask; rank = popcount of
// the mask below the lane), per-wave running offsets live in LDS.  Atomics only count (sort_spread_kernel,
// whole numbers in LDS, a sum that no order changes), so the result is deterministic.
// The three launches move a few bytes per pair and wait all the time: a wavefront's steps are a serial chain.
// Hence eight wavefronts of four steps per block (it was four of eight), and a wavefront's keys and weights
// fetched at once, not step by step: us, count + scan + scatter, 32768 pairs of 64 experts 9.2 + 6.7 + 21.4 ->
// 5.3 + 6.3 + 11.6, 9003 pairs of 12 7.0 + 3.1 + 16.3 -> 4.0 + 3.0 + 8.4 (sizes that took three launches then; 131072 pairs, which do
// now, 21.3 in all).
// Also: the reference's two index operators with their own [expert][column] table layout, one
// wavefront per column.
#include "sort_block.h"
#include <mutex>
#include <type_traits>

namespace {

constexpr int SORT_THREADS = 512;
constexpr int SORT_WAVES = SORT_THREADS / 64;
constexpr int SORT_ITERS = 4;                                    // 64-pair steps per wavefront
constexpr int SORT_CHUNK = SORT_THREADS * SORT_ITERS;            // pairs per block
constexpr int SORT_MAX_NR = 1024;                                // local experts supported

// The routing weight of every sorted row, for expert kernels that apply it themselves: row_weights[pos] =
// routing_weights[pair], float32 or bf16 -> float32.  Absent (row_weights null) where nobody asks for it.
struct RowWeights {
    const void *routing_weights = nullptr;
    float *row_weights = nullptr;
    int bf16 = 0;
    // fetched for all of a wavefront's pairs before the first is placed: a load per placement would be waited for each time
    __device__ __forceinline__ float get(int64_t pair, int64_t n_pairs) const {
        if (!row_weights || pair >= n_pairs) return 0.0f;
        return bf16 ? bf16_bits_to_f32(static_cast<const uint16_t *>(routing_weights)[pair])
                    : static_cast<const float *>(routing_weights)[pair];
    }
    __device__ __forceinline__ void put(int pos, float weight) const {
        if (row_weights) row_weights[pos] = weight;
    }
};

template <typename TI>
__device__ __forceinline__ int local_key(const TI *selected_experts, int64_t j, int64_t n_pairs,
                                         int start, int end, int NR) {
    if (j >= n_pairs) return NR;
    const long long e = static_cast<long long>(selected_experts[j]);
    return (e >= start && e < end) ? static_cast<int>(e - start) : NR;
}

// The keys of a wavefront's SORT_ITERS*64 pairs, all loads in flight at once.
template <typename TI>
__device__ __forceinline__ void wave_keys(const TI *selected_experts, int64_t wave_base, int64_t n_pairs, int start,
                                          int end, int NR, int lane, int (&key)[SORT_ITERS]) {
    TI e[SORT_ITERS];
#pragma unroll
    for (int it = 0; it < SORT_ITERS; it++) e[it] = selected_experts[min(wave_base + it * 64 + lane, n_pairs - 1)];
#pragma unroll
    for (int it = 0; it < SORT_ITERS; it++) {
        const long long v = static_cast<long long>(e[it]);
        key[it] = wave_base + it * 64 + lane < n_pairs && v >= start && v < end ? static_cast<int>(v - start) : NR;
    }
}

// Per-wave histogram of these keys into wave_hist[wave][0..NR).
__device__ __forceinline__ int wave_histogram(const int (&key)[SORT_ITERS], int NR, int nbits, int lane, volatile int *hist) {
    int hits = 0;
#pragma unroll
    for (int it = 0; it < SORT_ITERS; it++) {
        const unsigned long long m = match_key(key[it], nbits);
        const bool leader = (__ffsll(static_cast<long long>(m)) - 1) == lane;
        if (leader && key[it] < NR) hist[key[it]] += __popcll(m);
        hits += __popcll(__ballot(key[it] < NR));
        __builtin_amdgcn_wave_barrier();
    }
    return hits;
}

template <typename TI>
__global__ __launch_bounds__(SORT_THREADS) void sort_count_kernel(const TI *__restrict__ selected_experts,
                                                                  int64_t n_pairs, int start, int end,
                                                                  int NR, int nbits,
                                                                  int32_t *__restrict__ block_hist) {
    extern __shared__ int lds[];  // [SORT_WAVES][NR]
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int64_t wave_base = static_cast<int64_t>(blockIdx.x) * SORT_CHUNK + wv * (SORT_ITERS * 64);
    int key[SORT_ITERS];
    wave_keys(selected_experts, wave_base, n_pairs, start, end, NR, lane, key);
    for (int i = threadIdx.x; i < SORT_WAVES * NR; i += SORT_THREADS) lds[i] = 0;
    __syncthreads();
    wave_histogram(key, NR, nbits, lane, lds + wv * NR);
    __syncthreads();
    for (int e = threadIdx.x; e < NR; e += SORT_THREADS) {
        int s = 0;
        for (int w = 0; w < SORT_WAVES; w++) s += lds[w * NR + e];
        block_hist[static_cast<int64_t>(blockIdx.x) * NR + e] = s;
    }
}

// One block.  block_hist [NB][NR] -> in place: exclusive offset of (expert e, block b) in the
// stable order; hits_base [NB] = pairs kept by blocks before b; cum_token_counts [NR+1].
// Every phase is spread over the 16 wavefronts (lanes over blocks or over experts, wavefront
// scans), so nothing walks the table serially.
__global__ __launch_bounds__(1024) void sort_scan_kernel(int32_t *__restrict__ block_hist,
                                                          int32_t *__restrict__ hits_base, int NB,
                                                          int NR, int32_t *__restrict__ cum_token_counts,
                                                          int32_t *__restrict__ cum_expert_counts_ep,
                                                          int64_t T) {
    __shared__ int totals[SORT_MAX_NR + 1];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, n_waves = blockDim.x >> 6;
    // per-expert exclusive scan over blocks: one wavefront per expert, lanes over blocks
    for (int e = wv; e < NR; e += n_waves) {
        int run = 0;
        for (int b0 = 0; b0 < NB; b0 += 64) {
            const int b = b0 + lane;
            const int c = b < NB ? block_hist[static_cast<int64_t>(b) * NR + e] : 0;
            const int incl = wave_incl_scan(c, lane);
            if (b < NB) block_hist[static_cast<int64_t>(b) * NR + e] = run + incl - c;
            run += __shfl(incl, 63, 64);
        }
        if (lane == 0) totals[e] = run;
    }
    __syncthreads();
    if (wv == 0) {  // exclusive scan of the per-expert totals
        int run = 0;
        for (int e0 = 0; e0 < NR; e0 += 64) {
            const int e = e0 + lane;
            const int c = e < NR ? totals[e] : 0;
            const int incl = wave_incl_scan(c, lane);
            if (e < NR) {
                totals[e] = run + incl - c;
                cum_token_counts[e] = run + incl - c;
            }
            run += __shfl(incl, 63, 64);
        }
        if (lane == 0) {
            totals[NR] = run;
            cum_token_counts[NR] = run;
            cum_expert_counts_ep[T] = run;
        }
    }
    __syncthreads();
    // add the expert's base, and per block sum what its experts hold before it:
    // kept_before(b) = sum_e (off[b][e] - totals[e]) = sum_e of the within-expert offsets
    for (int b = wv; b < NB; b += n_waves) {
        int kept_before = 0;
        for (int e0 = 0; e0 < NR; e0 += 64) {
            const int e = e0 + lane;
            if (e < NR) {
                const int within = block_hist[static_cast<int64_t>(b) * NR + e];
                kept_before += within;
                block_hist[static_cast<int64_t>(b) * NR + e] = within + totals[e];
            }
        }
        kept_before = wave_sum_i(kept_before);
        if (lane == 0) hits_base[b] = kept_before;
    }
}

template <typename TI>
__global__ __launch_bounds__(SORT_THREADS) void sort_scatter_kernel(
    const TI *__restrict__ selected_experts, int64_t n_pairs, int K, int start, int end, int NR,
    int nbits, const int32_t *__restrict__ block_offsets, const int32_t *__restrict__ hits_base,
    int32_t *__restrict__ cum_expert_counts_ep, int32_t *__restrict__ input_indices,
    int32_t *__restrict__ output_indices, int32_t *__restrict__ selected_experts_indices, const RowWeights rw) {
    extern __shared__ int lds[];  // [SORT_WAVES][NR] then [SORT_WAVES] wave hit counts
    int *wave_hits = lds + SORT_WAVES * NR;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int64_t wave_base = static_cast<int64_t>(blockIdx.x) * SORT_CHUNK + wv * (SORT_ITERS * 64);
    int key[SORT_ITERS];
    float weight[SORT_ITERS];
    wave_keys(selected_experts, wave_base, n_pairs, start, end, NR, lane, key);
#pragma unroll
    for (int it = 0; it < SORT_ITERS; it++) weight[it] = rw.get(wave_base + it * 64 + lane, n_pairs);
    for (int i = threadIdx.x; i < SORT_WAVES * NR; i += SORT_THREADS) lds[i] = 0;
    __syncthreads();
    const int hits = wave_histogram(key, NR, nbits, lane, lds + wv * NR);
    if (lane == 0) wave_hits[wv] = hits;
    __syncthreads();
    // counts -> running offsets: off[w][e] = block offset + counts of the waves before w
    for (int e = threadIdx.x; e < NR; e += SORT_THREADS) {
        int run = block_offsets[static_cast<int64_t>(blockIdx.x) * NR + e];
        for (int w = 0; w < SORT_WAVES; w++) {
            const int c = lds[w * NR + e];
            lds[w * NR + e] = run;
            run += c;
        }
    }
    __syncthreads();
    int oi_base = hits_base[blockIdx.x];
    for (int w = 0; w < wv; w++) oi_base += wave_hits[w];
    volatile int *off = lds + wv * NR;
    // Entries past the number of kept pairs (an expert window keeps fewer than T*K) are given fixed
    // values, so that a caller who sizes its work by T*K instead of reading the count back can tell
    // them apart: output_indices -1 (no row), the other two 0 (a valid token / slot).
    const int total_kept = cum_expert_counts_ep[static_cast<uint32_t>(n_pairs) / static_cast<uint32_t>(K)];
#pragma unroll
    for (int it = 0; it < SORT_ITERS; it++) {
        const int64_t j = wave_base + it * 64 + lane;
        if (j < n_pairs && j >= total_kept) {
            output_indices[j] = -1;
            input_indices[j] = 0;
            selected_experts_indices[j] = 0;
        }
        const unsigned long long m = match_key(key[it], nbits);
        const unsigned long long kept = __ballot(key[it] < NR);
        const int oi = oi_base + __popcll(kept & lanemask_lt(lane));
        const bool valid = j < n_pairs;
        const uint32_t t = valid ? static_cast<uint32_t>(j) / static_cast<uint32_t>(K) : 0;   // (pairs are counted in int32)
        const int k = valid ? static_cast<int>(static_cast<uint32_t>(j) - t * K) : 0;
        if (valid && k == 0) cum_expert_counts_ep[t] = oi;
        if (key[it] < NR) {
            const int pos = off[key[it]] + __popcll(m & lanemask_lt(lane));
            __builtin_amdgcn_wave_barrier();
            const bool leader = (__ffsll(static_cast<long long>(m)) - 1) == lane;
            if (leader) off[key[it]] += __popcll(m);
            input_indices[pos] = static_cast<int32_t>(t);
            output_indices[oi] = pos;
            selected_experts_indices[oi] = k;
            rw.put(pos, weight[it]);
        } else {
            __builtin_amdgcn_wave_barrier();
        }
        oi_base += __popcll(kept);
        __builtin_amdgcn_wave_barrier();
    }
}

// Few pairs: count, scan and scatter by one block, in one launch (sort_block.h).
template <typename TI>
__global__ __launch_bounds__(SORT_BLOCK_PAIRS) void sort_small_kernel(
    const TI *__restrict__ selected_experts, int n_pairs, int K, int start, int end, int NR, int nbits,
    int32_t *__restrict__ cum_token_counts, int32_t *__restrict__ cum_expert_counts_ep,
    int32_t *__restrict__ input_indices, int32_t *__restrict__ output_indices,
    int32_t *__restrict__ selected_experts_indices, const RowWeights rw) {
    sort_block(selected_experts[min(static_cast<int>(threadIdx.x), n_pairs - 1)], rw.get(threadIdx.x, n_pairs), n_pairs, K, start, end, NR, nbits,
               cum_token_counts, cum_expert_counts_ep, input_indices, output_indices, selected_experts_indices, rw.row_weights);
}

// More pairs in one launch: a block sorts 1024 of them, as above, and counts all the others by itself, with LDS atomics on eight
// copies of the counts, so that the lanes of a wavefront that meet at one expert are few.  That is more work in all than count, scan
// and scatter, but not for a compute unit: 64 pairs a thread at the line, against two more launches and the waits in each.  us, as
// before (up to 8192 pairs one block of eight steps a wavefront, then three launches) -> so, operands in the caches / caches full of written data: 4096
// pairs of 64 experts 8.7 -> 6.5 / 11.8 -> 9.1, 8000 14.7 -> 6.8 / 18.2 -> 9.6, 16384 17 -> 7.6 / 20.4 -> 10.4, 32768 17 -> 9.5 / 20.7 -> 12.5 (uneven
// the same), 65536 17.9 -> 13.8 / 21.5 -> 17.1, 131072 21.3 -> 22.5 / 25.1 -> 26; 9003 of 12 13.2 -> 6.6 / 17 -> 9.2.
constexpr int64_t SPREAD_PAIRS = 1 << 16;
// VEC: selections in a load, 16 bytes of them where they are aligned
template <typename TI, int VEC>
__global__ __launch_bounds__(SORT_BLOCK_PAIRS) void sort_spread_kernel(
    const TI *__restrict__ selected_experts, int n_pairs, int K, int start, int end, int NR, int nbits,
    int32_t *__restrict__ cum_token_counts, int32_t *__restrict__ cum_expert_counts_ep,
    int32_t *__restrict__ input_indices, int32_t *__restrict__ output_indices,
    int32_t *__restrict__ selected_experts_indices, const RowWeights rw) {
    constexpr int THREADS = SORT_BLOCK_PAIRS, AHEAD = 8, CELLS = SORT_BLOCK_MAX_NR * SPREAD_COPIES;
    typedef TI vec __attribute__((ext_vector_type(VEC)));
    __shared__ int counts[2 * CELLS];   // of the pairs before this block's and of those after them
    const int tid = threadIdx.x, first = blockIdx.x * THREADS, last = min(first + THREADS, n_pairs);
    const TI e = selected_experts[min(first + tid, n_pairs - 1)];
    const float weight = rw.get(first + tid, n_pairs);
    for (int i = tid; i < 2 * CELLS; i += THREADS) counts[i] = 0;
    __syncthreads();
    const int n_vec = n_pairs / VEC, copy = tid % SPREAD_COPIES;
    auto count = [&](TI value, int at) {
        const long long v = static_cast<long long>(value);
        if (v >= start && v < end && (at < first || at >= last))
            atomicAdd(&counts[(at < first ? 0 : CELLS) + static_cast<int>(v - start) * SPREAD_COPIES + copy], 1);
    };
    for (int v0 = 0; v0 < n_vec; v0 += AHEAD * THREADS) {
        vec q[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; u++) q[u] = reinterpret_cast<const vec *>(selected_experts)[min(v0 + u * THREADS + tid, n_vec - 1)];
#pragma unroll
        for (int u = 0; u < AHEAD; u++) {
            const int at = v0 + u * THREADS + tid;
            if (at < n_vec)
#pragma unroll
                for (int x = 0; x < VEC; x++) count(q[u][x], at * VEC + x);
        }
    }
    if (tid < n_pairs - n_vec * VEC) count(selected_experts[n_vec * VEC + tid], n_vec * VEC + tid);
    // (sort_block's first barrier comes before it reads the counts)
    sort_block<true>(e, weight, n_pairs, K, start, end, NR, nbits, cum_token_counts, cum_expert_counts_ep, input_indices, output_indices,
                     selected_experts_indices, rw.row_weights, {first, counts, counts + CELLS});
}

// ---- the reference's table layout [expert][column] ---------------------------------------------
// The pybind ops keep a table with one column per group of TB = T / TH consecutive tokens
// (partial_token_counts [NR][TH], then its flattened cumsum, then a same-shaped table of running
// increments).  Here one wavefront owns one column: its TB*K (token, k) pairs are walked in
// row-major order 64 at a time, equal experts are matched by ballots (match_key), and the
// column's per-expert running values live in the wavefront's slice of LDS.  Same results as the
// reference's one-work-item-per-column serial loops, entry for entry.
constexpr int COL_WAVES = 4;   // columns per block

template <typename TI>
__global__ __launch_bounds__(COL_WAVES * 64) void column_counts_kernel(
    const TI *__restrict__ selected_experts, int32_t *__restrict__ partial_token_counts,
    int32_t *__restrict__ expert_counts_ep, int start, int end, int NR, int nbits, int K, int64_t TB,
    int64_t TH) {
    extern __shared__ int lds[];   // [COL_WAVES][NR]
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int64_t col = static_cast<int64_t>(blockIdx.x) * COL_WAVES + wv;
    if (col >= TH) return;   // whole wavefronts leave; no block-wide barrier below
    volatile int *hist = lds + wv * NR;
    for (int e = lane; e < NR; e += 64) hist[e] = 0;
    __builtin_amdgcn_wave_barrier();
    const int64_t j0 = col * TB * K, j1 = j0 + TB * K;
    for (int64_t base = j0; base < j1; base += 64) {
        const int key = local_key(selected_experts, base + lane, j1, start, end, NR);
        const unsigned long long m = match_key(key, nbits);
        if (key < NR && (__ffsll(static_cast<long long>(m)) - 1) == lane) hist[key] += __popcll(m);
        __builtin_amdgcn_wave_barrier();
    }
    for (int e = lane; e < NR; e += 64) {
        const int c = hist[e];
        if (c) partial_token_counts[static_cast<int64_t>(e) * TH + col] += c;   // the table is updated in place
    }
    // local hits per token: lanes over the column's tokens
    for (int64_t t = col * TB + lane; t < (col + 1) * TB; t += 64) {
        int hits = 0;
        for (int k = 0; k < K; k++) {
            const long long e = static_cast<long long>(selected_experts[t * K + k]);
            hits += (e >= start && e < end) ? 1 : 0;
        }
        expert_counts_ep[t] = hits;
    }
}

template <typename TI>
__global__ __launch_bounds__(COL_WAVES * 64) void column_scatter_kernel(
    const TI *__restrict__ selected_experts, const int32_t *__restrict__ partial_cum_token_counts,
    int32_t *__restrict__ input_increment_buffer, const int32_t *__restrict__ cum_expert_counts_ep,
    int32_t *__restrict__ selected_experts_indices, int32_t *__restrict__ input_indices,
    int32_t *__restrict__ output_indices, int start, int end, int NR, int nbits, int K, int64_t TB,
    int64_t TH) {
    extern __shared__ int lds[];   // [COL_WAVES][NR]: next free position of every expert in this column
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int64_t col = static_cast<int64_t>(blockIdx.x) * COL_WAVES + wv;
    if (col >= TH) return;
    volatile int *off = lds + wv * NR;
    for (int e = lane; e < NR; e += 64) {
        const int64_t cell = static_cast<int64_t>(e) * TH + col;
        off[e] = partial_cum_token_counts[cell] + input_increment_buffer[cell];
    }
    __builtin_amdgcn_wave_barrier();
    const int64_t j0 = col * TB * K, j1 = j0 + TB * K;
    // kept pairs of the token that straddles into the current 64-pair step
    int64_t carry_token = -1;
    int carry_kept = 0;
    for (int64_t base = j0; base < j1; base += 64) {
        const int64_t j = base + lane;
        const bool valid = j < j1;
        const int key = local_key(selected_experts, j, j1, start, end, NR);
        const unsigned long long m = match_key(key, nbits);
        const unsigned long long kept = __ballot(key < NR);
        const int64_t t = valid ? j / K : -2;
        const int k = valid ? static_cast<int>(j - t * K) : 0;
        // lanes of this step that hold earlier pairs of the same token: [first, lane)
        const int64_t first64 = t * K - base;
        const int first = first64 > 0 ? static_cast<int>(first64) : 0;
        const unsigned long long same_before = lanemask_lt(lane) & ~lanemask_lt(first);
        if (key < NR) {
            const int oi = cum_expert_counts_ep[t] + __popcll(kept & same_before) +
                           (t == carry_token ? carry_kept : 0);
            const int pos = off[key] + __popcll(m & lanemask_lt(lane));
            input_indices[pos] = static_cast<int32_t>(t);
            output_indices[oi] = pos;
            selected_experts_indices[oi] = k;
        }
        __builtin_amdgcn_wave_barrier();
        if (key < NR && (__ffsll(static_cast<long long>(m)) - 1) == lane) off[key] += __popcll(m);
        // the step's last token may continue in the next step: hand its kept pairs on
        const int64_t t_last = __shfl(t, 63, 64);
        if (t_last >= 0) {
            const int here = __popcll(kept & __ballot(t == t_last));
            carry_kept = (t_last == carry_token ? carry_kept : 0) + here;
            carry_token = t_last;
        }
        __builtin_amdgcn_wave_barrier();
    }
    for (int e = lane; e < NR; e += 64) {   // leave the increments as the reference's loop leaves them
        const int64_t cell = static_cast<int64_t>(e) * TH + col;
        input_increment_buffer[cell] = off[e] - partial_cum_token_counts[cell];
    }
}

}  // namespace

extern "C" int64_t om_moe_sort_workspace_bytes(int64_t T, int K, int NR) {
    if (T < 0 || K < 1 || NR < 1) return 0;
    const int64_t n_pairs = T * K;
    const int64_t NB = (n_pairs + SORT_CHUNK - 1) / SORT_CHUNK;
    return (NB * NR + NB + 1) * static_cast<int64_t>(sizeof(int32_t));
}

namespace {

// Launches count, scan and scatter with `workspace` holding the [NB][NR] block table and the
// [NB] kept-pair bases.  Arguments are validated by the two entry points below.
int moe_sort_launch(const void *selected_experts, int index_dtype, int64_t T, int K,
                    int expert_start_idx, int expert_end_idx, int32_t *cum_token_counts,
                    int32_t *cum_expert_counts_ep, int32_t *input_indices, int32_t *output_indices,
                    int32_t *selected_experts_indices, int32_t *workspace, hipStream_t st,
                    const RowWeights &rw = RowWeights()) {
    const int NR = expert_end_idx - expert_start_idx;
    const int64_t n_pairs = T * K;
    if (n_pairs > 0 && n_pairs <= SPREAD_PAIRS && NR <= SORT_BLOCK_MAX_NR) {
        const unsigned blocks = static_cast<unsigned>((n_pairs + SORT_BLOCK_PAIRS - 1) / SORT_BLOCK_PAIRS);
        auto sort = [&](const auto *experts) {
            using TI = std::remove_const_t<std::remove_pointer_t<decltype(experts)>>;
            auto launch = [&](auto kernel) {
                kernel<<<blocks, SORT_BLOCK_PAIRS, 0, st>>>(experts, static_cast<int>(n_pairs), K, expert_start_idx, expert_end_idx, NR, key_bits(NR),
                                                            cum_token_counts, cum_expert_counts_ep, input_indices, output_indices,
                                                            selected_experts_indices, rw);
            };
            if (blocks == 1) launch(sort_small_kernel<TI>);
            else if (om_aligned16(experts)) launch(sort_spread_kernel<TI, 16 / sizeof(TI)>);
            else launch(sort_spread_kernel<TI, 1>);
        };
        if (index_dtype == OM_I64) sort(static_cast<const int64_t *>(selected_experts));
        else sort(static_cast<const int32_t *>(selected_experts));
        return om_launch_status();
    }
    const int64_t NB = (n_pairs + SORT_CHUNK - 1) / SORT_CHUNK;
    int32_t *block_hist = workspace;
    int32_t *hits_base = block_hist + NB * NR;
    const int nbits = key_bits(NR);
    const size_t lds_count = static_cast<size_t>(SORT_WAVES) * NR * sizeof(int);
    const size_t lds_scatter = lds_count + SORT_WAVES * sizeof(int);
    if (NB > 0) {
        if (index_dtype == OM_I64)
            sort_count_kernel<int64_t><<<static_cast<unsigned>(NB), SORT_THREADS, lds_count, st>>>(
                static_cast<const int64_t *>(selected_experts), n_pairs, expert_start_idx,
                expert_end_idx, NR, nbits, block_hist);
        else
            sort_count_kernel<int32_t><<<static_cast<unsigned>(NB), SORT_THREADS, lds_count, st>>>(
                static_cast<const int32_t *>(selected_experts), n_pairs, expert_start_idx,
                expert_end_idx, NR, nbits, block_hist);
    }
    sort_scan_kernel<<<1, 1024, 0, st>>>(block_hist, hits_base, static_cast<int>(NB), NR,
                                         cum_token_counts, cum_expert_counts_ep, T);
    if (NB > 0) {
        if (index_dtype == OM_I64)
            sort_scatter_kernel<int64_t><<<static_cast<unsigned>(NB), SORT_THREADS, lds_scatter, st>>>(
                static_cast<const int64_t *>(selected_experts), n_pairs, K, expert_start_idx,
                expert_end_idx, NR, nbits, block_hist, hits_base, cum_expert_counts_ep, input_indices,
                output_indices, selected_experts_indices, rw);
        else
            sort_scatter_kernel<int32_t><<<static_cast<unsigned>(NB), SORT_THREADS, lds_scatter, st>>>(
                static_cast<const int32_t *>(selected_experts), n_pairs, K, expert_start_idx,
                expert_end_idx, NR, nbits, block_hist, hits_base, cum_expert_counts_ep, input_indices,
                output_indices, selected_experts_indices, rw);
    }
    return om_launch_status();
}

int moe_sort_check(const void *selected_experts, int index_dtype, int64_t T, int K,
                   int expert_start_idx, int expert_end_idx, const int32_t *cum_token_counts,
                   const int32_t *cum_expert_counts_ep, const int32_t *input_indices,
                   const int32_t *output_indices, const int32_t *selected_experts_indices) {
    if (index_dtype != OM_I32 && index_dtype != OM_I64) return OM_ERR_DTYPE;
    const int NR = expert_end_idx - expert_start_idx;
    if (T < 0 || K < 1 || NR < 1 || NR > SORT_MAX_NR || expert_start_idx < 0) return OM_ERR_SHAPE;
    if (T * K > 0x7fffffffLL) return OM_ERR_SHAPE;
    if (!cum_token_counts || !cum_expert_counts_ep) return OM_ERR_NULL;
    if (T > 0 && (!selected_experts || !input_indices || !output_indices || !selected_experts_indices))
        return OM_ERR_NULL;
    return OM_OK;
}

}  // namespace

extern "C" int om_moe_sort_weighted(const void *selected_experts, int index_dtype, int64_t T, int K,
                                    int expert_start_idx, int expert_end_idx, int32_t *cum_token_counts,
                                    int32_t *cum_expert_counts_ep, int32_t *input_indices,
                                    int32_t *output_indices, int32_t *selected_experts_indices,
                                    const void *routing_weights, int weights_dtype, float *row_weights,
                                    void *workspace, int64_t workspace_bytes, void *stream) {
    const int rc = moe_sort_check(selected_experts, index_dtype, T, K, expert_start_idx, expert_end_idx,
                                  cum_token_counts, cum_expert_counts_ep, input_indices, output_indices,
                                  selected_experts_indices);
    if (rc != OM_OK) return rc;
    if (row_weights) {
        if (weights_dtype != OM_F32 && weights_dtype != OM_BF16) return OM_ERR_DTYPE;
        if (T > 0 && !routing_weights) return OM_ERR_NULL;
    }
    if (workspace_bytes < om_moe_sort_workspace_bytes(T, K, expert_end_idx - expert_start_idx))
        return OM_ERR_WORKSPACE;
    if (!workspace || (reinterpret_cast<uintptr_t>(workspace) & 3u)) return OM_ERR_ALIGN;
    RowWeights rw;
    rw.routing_weights = routing_weights;
    rw.row_weights = row_weights;
    rw.bf16 = weights_dtype == OM_BF16;
    return moe_sort_launch(selected_experts, index_dtype, T, K, expert_start_idx, expert_end_idx,
                           cum_token_counts, cum_expert_counts_ep, input_indices, output_indices,
                           selected_experts_indices, static_cast<int32_t *>(workspace), om_stream(stream), rw);
}

extern "C" int om_moe_sort(const void *selected_experts, int index_dtype, int64_t T, int K,
                           int expert_start_idx, int expert_end_idx, int32_t *cum_token_counts,
                           int32_t *cum_expert_counts_ep, int32_t *input_indices,
                           int32_t *output_indices, int32_t *selected_experts_indices,
                           void *workspace, int64_t workspace_bytes, void *stream) {
    return om_moe_sort_weighted(selected_experts, index_dtype, T, K, expert_start_idx, expert_end_idx, cum_token_counts,
                                cum_expert_counts_ep, input_indices, output_indices, selected_experts_indices, nullptr,
                                OM_F32, nullptr, workspace, workspace_bytes, stream);
}

// ---- om_moe_sort for callers that cannot allocate ----------------------------------------------
// The block table lives in a file-scope device array instead of a caller's workspace.  The array's
// name is only a host-side handle: its device address is asked from the runtime once per device
// (with that device current) and kept; kernels and everything else in host code use that address.
constexpr int64_t SORT_SCRATCH_BYTES = 4ll << 20;
constexpr int SORT_MAX_DEVICES = 64;

static __device__ __align__(256) int32_t sort_scratch[SORT_SCRATCH_BYTES / sizeof(int32_t)];

namespace {

std::mutex sort_scratch_mutex;
int32_t *sort_scratch_ptr[SORT_MAX_DEVICES] = {};

// Device address of sort_scratch on the current device; nullptr if the runtime refuses.
int32_t *sort_scratch_on_current_device() {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= SORT_MAX_DEVICES) return nullptr;
    std::lock_guard<std::mutex> lock(sort_scratch_mutex);
    if (!sort_scratch_ptr[dev]) {
        void *p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(sort_scratch)) != hipSuccess || !p) {
            (void)hipGetLastError();
            return nullptr;
        }
        sort_scratch_ptr[dev] = static_cast<int32_t *>(p);
    }
    return sort_scratch_ptr[dev];
}

}  // namespace

extern "C" int64_t om_moe_sort_static_capacity_bytes(void) { return SORT_SCRATCH_BYTES; }

extern "C" int om_moe_sort_static(const void *selected_experts, int index_dtype, int64_t T, int K,
                                  int expert_start_idx, int expert_end_idx, int32_t *cum_token_counts,
                                  int32_t *cum_expert_counts_ep, int32_t *input_indices,
                                  int32_t *output_indices, int32_t *selected_experts_indices,
                                  void *stream) {
    const int rc = moe_sort_check(selected_experts, index_dtype, T, K, expert_start_idx, expert_end_idx,
                                  cum_token_counts, cum_expert_counts_ep, input_indices, output_indices,
                                  selected_experts_indices);
    if (rc != OM_OK) return rc;
    if (om_moe_sort_workspace_bytes(T, K, expert_end_idx - expert_start_idx) > SORT_SCRATCH_BYTES)
        return OM_ERR_WORKSPACE;
    int32_t *scratch = sort_scratch_on_current_device();
    if (!scratch) return OM_ERR_LAUNCH;
    // count writes every cell of the block table it later reads and scan writes every base, so
    // nothing left in the array by an earlier call needs clearing
    return moe_sort_launch(selected_experts, index_dtype, T, K, expert_start_idx, expert_end_idx,
                           cum_token_counts, cum_expert_counts_ep, input_indices, output_indices,
                           selected_experts_indices, scratch, om_stream(stream));
}

extern "C" int om_compute_partial_token_counts(const void *selected_experts, int index_dtype,
                                               int32_t *partial_token_counts,
                                               int32_t *expert_counts_ep, int expert_start_idx,
                                               int expert_end_idx, int64_t T, int K, int64_t TH,
                                               void *stream) {
    if (index_dtype != OM_I32 && index_dtype != OM_I64) return OM_ERR_DTYPE;
    const int NR = expert_end_idx - expert_start_idx;
    if (T < 0 || K < 1 || TH < 1 || T % TH != 0 || NR < 1 || NR > SORT_MAX_NR) return OM_ERR_SHAPE;
    if (T == 0) return OM_OK;
    if (!selected_experts || !partial_token_counts || !expert_counts_ep) return OM_ERR_NULL;
    hipStream_t st = om_stream(stream);
    const unsigned nb = static_cast<unsigned>((TH + COL_WAVES - 1) / COL_WAVES);
    const size_t lds = static_cast<size_t>(COL_WAVES) * NR * sizeof(int);
    const int nbits = key_bits(NR);
    if (index_dtype == OM_I64)
        column_counts_kernel<int64_t><<<nb, COL_WAVES * 64, lds, st>>>(
            static_cast<const int64_t *>(selected_experts), partial_token_counts, expert_counts_ep,
            expert_start_idx, expert_end_idx, NR, nbits, K, T / TH, TH);
    else
        column_counts_kernel<int32_t><<<nb, COL_WAVES * 64, lds, st>>>(
            static_cast<const int32_t *>(selected_experts), partial_token_counts, expert_counts_ep,
            expert_start_idx, expert_end_idx, NR, nbits, K, T / TH, TH);
    return om_launch_status();
}

extern "C" int om_compute_input_and_output_indices(
    const void *selected_experts, int index_dtype, const int32_t *partial_cum_token_counts,
    int32_t *input_increment_buffer, const int32_t *cum_expert_counts_ep,
    int32_t *selected_experts_indices, int32_t *input_indices, int32_t *output_indices,
    int expert_start_idx, int expert_end_idx, int64_t T, int K, int64_t TH, void *stream) {
    if (index_dtype != OM_I32 && index_dtype != OM_I64) return OM_ERR_DTYPE;
    const int NR = expert_end_idx - expert_start_idx;
    if (T < 0 || K < 1 || TH < 1 || T % TH != 0 || NR < 1 || NR > SORT_MAX_NR) return OM_ERR_SHAPE;
    if (T == 0) return OM_OK;
    if (!selected_experts || !partial_cum_token_counts || !input_increment_buffer ||
        !cum_expert_counts_ep || !selected_experts_indices || !input_indices || !output_indices)
        return OM_ERR_NULL;
    hipStream_t st = om_stream(stream);
    const unsigned nb = static_cast<unsigned>((TH + COL_WAVES - 1) / COL_WAVES);
    const size_t lds = static_cast<size_t>(COL_WAVES) * NR * sizeof(int);
    const int nbits = key_bits(NR);
    if (index_dtype == OM_I64)
        column_scatter_kernel<int64_t><<<nb, COL_WAVES * 64, lds, st>>>(
            static_cast<const int64_t *>(selected_experts), partial_cum_token_counts,
            input_increment_buffer, cum_expert_counts_ep, selected_experts_indices, input_indices,
            output_indices, expert_start_idx, expert_end_idx, NR, nbits, K, T / TH, TH);
    else
        column_scatter_kernel<int32_t><<<nb, COL_WAVES * 64, lds, st>>>(
            static_cast<const int32_t *>(selected_experts), partial_cum_token_counts,
            input_increment_buffer, cum_expert_counts_ep, selected_experts_indices, input_indices,
            output_indices, expert_start_idx, expert_end_idx, NR, nbits, K, T / TH, TH);
    return om_launch_status();
}

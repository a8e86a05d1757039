// Grouped expert products y = x W^T for the handful of rows per expert that generation has: a stream of
// weights that are used once (one token's top-8 of 64 experts: 101 MB; 37 tokens: nearly all 805 MB).
//
// What bounds it: the rate at which weights arrive, and the launch's own chain of latencies.  The tiles of
// ggemm.hip give a one-token call 128 blocks of a possible 512, and each walks the contraction in 64-deep
// steps with two in flight behind barriers.  Here a block owns 32 weight rows (16 gate and 16 up rows, or 32
// output columns) and its eight wavefronts split the contraction: each takes every eighth 64-deep (128-byte)
// piece, loads its weights straight into the fragments of v_mfma_f32_16x16x32_bf16 (a weight is used by one
// wavefront only, so LDS would only add a barrier), one group of pieces ahead, and the eight partial sums
// meet in LDS once at the end, added in the order of the wavefronts.  The weights are the instruction's
// first operand, so a lane ends with four neighbouring output columns of one token.  What mattered, measured
// on one token of OLMoE's sizes (gate+up + down, us): loads past the end issued and thrown away 17 + 14.5,
// plain loads instead of non-temporal ones -20 %, ends masked by address so that nothing is copied
// 13.7 + 7.1 (4.8 TB/s); the tiled kernels 22 + 12.3.
// Rows of an expert come in tiles of 64 (1, 2 or 4 fragments of 16 by how many there are); a further tile
// streams the weights again, mostly out of the caches.
//
// The grid is (column tiles) x (an upper bound on row tiles); a wavefront finds its row tile with a scan
// over cum_token_counts, 64 experts at a time, so experts without rows cost nothing.
#include "common.h"

namespace {

constexpr int WAVES = 8;
constexpr int ROWS = 64;       // rows of a row tile
constexpr int PIECE = 64;      // contraction indices per piece: one 128-byte line of a weight row

__device__ __attribute__((aligned(16))) const uint16_t zero_chunk[8] = {};

struct StreamParams {
    const uint16_t *x;
    const uint16_t *w[2];      // SWIGLU: gate and up; else w[0] twice
    uint16_t *out[3];          // SWIGLU: g, u (or neither), h; else out[0]
    const int32_t *cum;
    const int32_t *row_index;  // != null: sorted row r is row row_index[r] of x
    const float *row_scale;    // != null: h is scaled by it
    int64_t w_stride;
    int n_experts, n_cols, kc;
};

// Fragments of MB x 16 rows against 2 x 16 weight rows.  `xr`: this lane's source rows, `wr`: its two weight
// rows, all at its first contraction index.
template <int MB, int GROUP, int SETS>
__device__ __forceinline__ void stream_product(const uint16_t *const (&xr)[MB], const uint16_t *const (&wr)[2], int wave,
                                               int lane, int kc, f32x4 (&acc)[2][MB]) {
    const int q8 = (lane >> 4) * 8;
    const int pieces = (kc + PIECE - 1) / PIECE;
    const int mine = max(0, (pieces - wave + WAVES - 1) / WAVES);   // pieces wave, wave + 8, ...
    const int groups = (mine + GROUP - 1) / GROUP;
    u32x4 xf[SETS][GROUP][2][MB], wf[SETS][GROUP][2][2];
    auto load = [&](int group, int set) {                      // the weights first: a row index may still be on its way
        // past the end of the rows: zeros on both sides (selected by address, nothing is masked afterwards)
#pragma unroll
        for (int i = 0; i < GROUP; i++)
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const int k = (wave + (group * GROUP + i) * WAVES) * PIECE + t * 32 + q8;
#pragma unroll
                for (int m = 0; m < 2; m++)
                    wf[set][i][t][m] = *reinterpret_cast<const u32x4 *>(k < kc ? wr[m] + k : zero_chunk);
            }
#pragma unroll
        for (int i = 0; i < GROUP; i++)
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const int k = (wave + (group * GROUP + i) * WAVES) * PIECE + t * 32 + q8;
#pragma unroll
                for (int b = 0; b < MB; b++)
                    xf[set][i][t][b] = *reinterpret_cast<const u32x4 *>(k < kc ? xr[b] + k : zero_chunk);
            }
    };
    auto multiply = [&](int set) {
#pragma unroll
        for (int i = 0; i < GROUP; i++)
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int m = 0; m < 2; m++)
#pragma unroll
                    for (int b = 0; b < MB; b++)
                        acc[m][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            __builtin_bit_cast(bf16x8, wf[set][i][t][m]), __builtin_bit_cast(bf16x8, xf[set][i][t][b]),
                            acc[m][b], 0, 0, 0);
    };
    if (SETS == 1) {
#pragma unroll 1
        for (int group = 0; group < groups; group++) {
            load(group, 0);
            multiply(0);
        }
        return;
    }
    // (the loop is left where nothing is in flight: a load inside a branch would be waited for at its end)
    load(0, 0);
#pragma unroll 1
    for (int group = 1;; group += 2) {
        if (group >= groups) { multiply(0); return; }
        load(group, SETS - 1);
        multiply(0);
        if (group + 1 >= groups) { multiply(SETS - 1); return; }
        load(group + 1, 0);
        multiply(SETS - 1);
    }
}

template <bool SWIGLU, int MB, int GROUP, int SETS>
__device__ __forceinline__ void stream_tile(const StreamParams &p, int expert, int row0, int row_end, int n0,
                                            f32x4 (*part)[2][64]) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int l16 = lane & 15;
    const uint16_t *wr[2], *xr[MB];
#pragma unroll
    for (int m = 0; m < 2; m++) {
        // weight rows past the last one (a partial column tile) re-read it; masked on store
        const int n = min(n0 + (SWIGLU ? 0 : m * 16) + l16, p.n_cols - 1);
        wr[m] = p.w[m] + expert * p.w_stride + static_cast<int64_t>(n) * p.kc;
    }
#pragma unroll
    for (int b = 0; b < MB; b++) {
        int64_t r = min(row0 + b * 16 + l16, row_end - 1);       // rows past the segment: results unused
        if (p.row_index) r = p.row_index[r];
        xr[b] = p.x + r * p.kc;
    }
    f32x4 acc[2][MB] = {};
    stream_product<MB, GROUP, SETS>(xr, wr, wave, lane, p.kc, acc);

    // Accumulator element r of lane l: column (l / 16) * 4 + r of row l % 16.  The wavefronts' partial sums
    // lie one after another, so the sum reads are consecutive floats.
#pragma unroll
    for (int b = 0; b < MB; b++) {
        if (b) __syncthreads();
        part[wave][0][lane] = acc[0][b];
        part[wave][1][lane] = acc[1][b];
        __syncthreads();
        const int t = threadIdx.x & 255, half = threadIdx.x >> 8;
        const int row = row0 + b * 16 + ((t >> 2) & 15);
        const int col = (t >> 6) * 4 + (t & 3);
        const float *sums = reinterpret_cast<const float *>(part) + t;
        if (SWIGLU) {
            if (half) continue;
            float g = 0.0f, u = 0.0f;
#pragma unroll
            for (int w = 0; w < WAVES; w++) {
                g += sums[w * 512];
                u += sums[w * 512 + 256];
            }
            if (row < row_end && n0 + col < p.n_cols) {
                const int64_t o = static_cast<int64_t>(row) * p.n_cols + n0 + col;
                float h = (g * fast_sigmoid(g)) * u;
                if (p.row_scale) h *= p.row_scale[row];
                if (p.out[0]) {
                    p.out[0][o] = f32_to_bf16_bits(g);
                    p.out[1][o] = f32_to_bf16_bits(u);
                }
                p.out[2][o] = f32_to_bf16_bits(h);
            }
        } else {
            float y = 0.0f;
#pragma unroll
            for (int w = 0; w < WAVES; w++) y += sums[w * 512 + half * 256];
            const int n = n0 + half * 16 + col;
            if (row < row_end && n < p.n_cols) p.out[0][static_cast<int64_t>(row) * p.n_cols + n] = f32_to_bf16_bits(y);
        }
    }
}

// WIDE: registers for one block per CU, so that tiles of 32 and 64 rows have two groups in flight as well.
template <bool SWIGLU, bool WIDE> __global__ __launch_bounds__(WAVES * 64, WIDE ? 2 : 4) void stream_kernel(StreamParams p) {
    __shared__ f32x4 part[WAVES][2][64];
    const int lane = threadIdx.x & 63;
    int want = blockIdx.y, expert = -1, row0 = 0, row_end = 0;
    for (int e0 = 0; e0 < p.n_experts; e0 += 64) {
        const int e = e0 + lane;
        const int begin = p.cum[min(e, p.n_experts)], end = p.cum[min(e + 1, p.n_experts)];
        const int tiles = (end - begin + ROWS - 1) / ROWS;
        int upto = tiles;                                        // tiles of experts e0 .. e
        for (int o = 1; o < 64; o <<= 1) {
            const int below = __shfl_up(upto, o, 64);
            if (lane >= o) upto += below;
        }
        const int total = __shfl(upto, 63, 64);
        if (want < total) {
            const int l = __ffsll(__ballot(upto > want)) - 1;
            expert = e0 + l;
            row0 = __shfl(begin, l, 64) + (want - __shfl(upto - tiles, l, 64)) * ROWS;
            row_end = __shfl(end, l, 64);
            break;
        }
        want -= total;
    }
    if (expert < 0) return;                                      // (block-uniform: every wavefront scans the same)
    expert = __builtin_amdgcn_readfirstlane(expert);
    row0 = __builtin_amdgcn_readfirstlane(row0);
    row_end = __builtin_amdgcn_readfirstlane(min(row_end, row0 + ROWS));
    const int n0 = blockIdx.x * (SWIGLU ? 16 : 32);
    const int rows = row_end - row0;
    if (rows <= 16) stream_tile<SWIGLU, 1, WIDE ? 2 : 1, 2>(p, expert, row0, row_end, n0, part);
    else if (rows <= 32) stream_tile<SWIGLU, 2, WIDE ? 2 : 1, 2>(p, expert, row0, row_end, n0, part);
    else stream_tile<SWIGLU, 4, 1, WIDE ? 2 : 1>(p, expert, row0, row_end, n0, part);
}

template <bool SWIGLU> int launch(const StreamParams &p, int64_t rows, int64_t expected, hipStream_t st) {
    const int64_t hit = rows < p.n_experts ? rows : p.n_experts;
    const int64_t tiles = hit + rows / ROWS < rows ? hit + rows / ROWS : rows;   // >= sum of ceil(rows of an expert / ROWS)
    const int cols = SWIGLU ? 16 : 32;
    const dim3 grid((p.n_cols + cols - 1) / cols, static_cast<unsigned>(tiles)), block(WAVES * 64);
    if (expected > 16 * static_cast<int64_t>(p.n_experts)) stream_kernel<SWIGLU, true><<<grid, block, 0, st>>>(p);
    else stream_kernel<SWIGLU, false><<<grid, block, 0, st>>>(p);
    return om_launch_status();
}

}  // namespace

// The line between these kernels and the tiled ones (tiled -> here, us, gate+up + down):
//   fewer than two rows per expert on average: hidden 2048, ffn 1024, 64 experts, top-8: 1 token 22 + 12.3 -> 13.7 + 7.1,
//   2 tokens 24 + 14.1 -> 25 + 13.5, 3 tokens 35 + 20 -> 34 + 17, 8 tokens even, 16 tokens even + 40 -> 43; 37
//   tokens (4.6 rows) 111 + 43 -> 111 + 48, hidden 7168, ffn 2048 at 8 rows 321 + 165 -> 360 + 174: tiled from two on;
//   the same for a window of 32 experts of 7168 / 2048 whose rows are only expected (T tokens of top-8 of 256, six
//   draws of weights and tokens, whole pass): 40 tokens -3.5 to +3.6 %, 56 tokens -7 to +3 %, 9 tokens 241 -> 220;
//   fewer than half a row per expert where the tiled kernels load the weights past the caches (om_weights_pass_caches), which the
//   figures above are without: whole forward of 4 tokens 80 (here 95), 8 tokens 115 (132), 15 tokens 140 (160); the window of
//   32 experts, 20 tokens 246, 172, 178 (255, 179, 200), 60 tokens 275, 261, 244 (317, 266, 263); 2 and 9 tokens even; at half a row an expert
//   itself 64 experts of ffn 1024 are even on average (4 tokens, hidden 1024 51.8 (49.4), 1536 68.0 (63.7), 1792 74.6 (75.5), 2048 83.5
//   (91.4), 3072 111 (109)), at one row 2 to 9 % better;
//   more rows where the tiles cannot fill the chip (fewer tiles than CUs): one expert of hidden 7168, ffn 2048
//   with 64 rows 65 + 21 -> 40 + 14; 12 experts of hidden 1000, ffn 712 with 192 rows 19 + 11.6 -> 10.8 + 5.4;
//   beyond 64 rows of one expert the weights are streamed again per row tile: 128 rows 65 + 21 -> 43 + 25.
// `rows`: those to expect where only a bound is known.  (Going by the bound, eight times as many, the window of 32
// experts of 1024 / 256 ran its gate+up product on tiles at 4 rows per expert and on 256x256 ones at 62: forward of
// 128 tokens 82.3 -> 78.4 us, 256 86.5 -> 83.3, 1000 105.6 -> 102.3, 2000 112 -> 109; 512 91.6 -> 94.2.)
bool om_ggemm_streams(int64_t rows, int n_experts, int cols, bool past_caches) {
    if (rows > 64 + 16 * static_cast<int64_t>(n_experts)) return false;
    if (rows < (past_caches ? n_experts / 2 : 2 * static_cast<int64_t>(n_experts))) return true;
    const int64_t hit = rows < n_experts ? rows : n_experts;
    return (hit + rows / 128) * ((cols + 127) / 128) <= 256;
}

int om_ggemm_stream_gate_up(const void *x, const int32_t *x_rows, const void *w_gate, const void *w_up,
                            const float *row_weights, void *g, void *u, void *h, const int32_t *cum, int64_t rows, int64_t expected,
                            int G, int I, int H, int64_t w_stride, hipStream_t st) {
    StreamParams p = {};
    p.x = static_cast<const uint16_t *>(x);
    p.w[0] = static_cast<const uint16_t *>(w_gate);
    p.w[1] = static_cast<const uint16_t *>(w_up);
    p.out[0] = static_cast<uint16_t *>(g);
    p.out[1] = static_cast<uint16_t *>(u);
    p.out[2] = static_cast<uint16_t *>(h);
    p.cum = cum;
    p.row_index = x_rows;
    p.row_scale = row_weights;
    p.w_stride = w_stride;
    p.n_experts = G; p.n_cols = I; p.kc = H;
    return launch<true>(p, rows, expected, st);
}

int om_ggemm_stream_fwd(const void *x, const void *w, void *out, const int32_t *cum, int64_t rows, int64_t expected, int G,
                        int N, int K, int64_t w_stride, hipStream_t st) {
    StreamParams p = {};
    p.x = static_cast<const uint16_t *>(x);
    p.w[0] = p.w[1] = static_cast<const uint16_t *>(w);
    p.out[0] = static_cast<uint16_t *>(out);
    p.cum = cum;
    p.w_stride = w_stride;
    p.n_experts = G; p.n_cols = N; p.kc = K;
    return launch<false>(p, rows, expected, st);
}

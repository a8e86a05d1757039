// Grouped expert GEMMs in float32 (v_mfma_f32_32x32x2_f32, fp32 operands and accumulation), for
// modules kept in float32 like the reference's small CPU-runnable configuration
// (GroupedGemmFunction, optimus/models/common/moe.py:163-215, runs torch.matmul per expert in
// whatever dtype the module has).  Same products and the same variable-rows-per-expert contract as
// the bf16 kernels: forward, input gradient, weight gradient, and the merged MLP's forms of them (gate
// and up in one launch with the SwiGLU or its backward in the epilogue, the token gather in the loads).
//
// One 64x64 output tile per block of eight wavefronts: four of them (2x2 of 32x32) take the first half of
// each 64-deep contraction step and four the second, and the two sums are added through LDS at the end.
// Two LDS stages, one barrier per step; two further steps of both operands are on their way in registers.
// These launches are small (the tiny layer: 1.07 GFLOP a product, 256 to 288 tiles), so many CUs hold one
// tile and what bounds them is how much of the matrix core's time one block can use: a wavefront's chain of
// fragment read -> MFMA, the barrier, the misses.  Tiny layer (2048 tokens, hidden 256, ffn 512, 8
// experts, top-2), us per launch with four wavefronts, 32-deep steps and one step ahead -> now: gate+up
// 41 -> 39, down 24 -> 23, down input gradient 25 -> 27, gate/up input gradient 46 -> 44, down weight
// gradient 23 -> 17, gate/up weight gradients 33 -> 30; four steps ahead without the second group of
// wavefronts 39, 25, 29, 46, 20, 31.  The row products stay at 64 % of the matrix rate on the CUs that hold
// two of the 288 tiles.
//
// CONTIG operands ([row][c] in memory, c = contraction index) lie in LDS as [row][c] with a 68-float
// pitch: 16-byte writes and reads, 16 consecutive rows in 16 different 16-byte bank groups.  STRIDED
// operands ([c][row] in memory: the weight in dgrad, both operands in wgrad) lie as [c][row] with a
// 68-float pitch, read 4 bytes at a time (one read per 64-cycle MFMA: not what bounds).
#include "common.h"

namespace {

constexpr int TB = 64;      // tile rows and columns
constexpr int KS = 64;      // contraction step: 32 indices for each of the two groups of wavefronts
constexpr int THREADS = 512;
constexpr int PITCH_C = KS + 4, PITCH_S = TB + 4;
constexpr int STAGE = TB * PITCH_C > KS * PITCH_S ? TB * PITCH_C : KS * PITCH_S;   // floats per operand tile
typedef __attribute__((ext_vector_type(4))) float f4;

enum { F_CONTIG = 0, F_STRIDED = 1 };
enum { E_STORE = 0, E_SWIGLU = 1, E_SWIGLU_BWD = 2 };

struct F32Params {
    const float *A[2], *B[2];   // second pair: up matrix (E_SWIGLU), second phase, or second weight gradient
    float *C[3];                // output; E_SWIGLU: g, u, h; E_SWIGLU_BWD: dg, du; two weight gradients
    const float *G, *U;         // E_SWIGLU_BWD: saved g, u
    const int32_t *cum;
    const int32_t *row_index;   // row r of A (rows products) or contraction row r of B (wgrad) is row row_index[r]
    int64_t lda, ldb, ldc, strideB[2], strideC[2];
    int n_experts, n_cols, kc, phases;
    int accumulate;             // wgrad, bit w: C[w] += product instead of C[w] = product
};

// One thread's part of a tile and step: 8 floats along c (CONTIG) or along the rows (STRIDED).
struct Fetched { f4 v[2]; bool in; };
template <int KIND> __device__ __forceinline__ int slot_row(int tid) { return KIND == F_CONTIG ? tid >> 3 : (tid & 7) * 8; }
template <int KIND> __device__ __forceinline__ int slot_c(int tid) { return KIND == F_CONTIG ? (tid & 7) * 8 : tid >> 3; }
template <int KIND> __device__ __forceinline__ void stash(float *tile, const Fetched &q, int tid) {
    float *p = KIND == F_CONTIG ? tile + slot_row<KIND>(tid) * PITCH_C + slot_c<KIND>(tid)
                                : tile + slot_c<KIND>(tid) * PITCH_S + slot_row<KIND>(tid);
    const f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    reinterpret_cast<f4 *>(p)[0] = q.in ? q.v[0] : zero;
    reinterpret_cast<f4 *>(p)[1] = q.in ? q.v[1] : zero;
}
// 8 floats at p (always valid memory: callers clamp); `in` false: zeros take their place when they are
// stashed.  Extents are multiples of 8, so a slot is inside or outside as a whole.  No load is conditional:
// at the end of a branch around one the compiler would wait for every load in flight.
__device__ __forceinline__ Fetched fetch8(const float *p, bool in) {
    Fetched q;
    q.v[0] = reinterpret_cast<const f4 *>(p)[0];
    q.v[1] = reinterpret_cast<const f4 *>(p)[1];
    q.in = in;
    return q;
}
// Fragment of contraction indices 8s + 4*(lane/32) .. +3 of operand row `row`; element j goes to MFMA j.
template <int KIND> __device__ __forceinline__ f4 fragment(const float *tile, int row, int s, int half) {
    if (KIND == F_CONTIG) return *reinterpret_cast<const f4 *>(tile + row * PITCH_C + s * 8 + half * 4);
    f4 v;
#pragma unroll
    for (int j = 0; j < 4; j++) v[j] = tile[(s * 8 + half * 4 + j) * PITCH_S + row];
    return v;
}

// The main loop: `fetch_a(step)` / `fetch_b(step)` deliver this thread's part of a step, also past the last
// one (valid memory, not used).  AHEAD steps of both operands are on their way in registers, since a miss
// costs more than a step's 1024 cycles of MFMA.
constexpr int AHEAD = 2;    // (even: a register set always meets the same LDS stage)
template <int AKIND, int BKIND, typename FA, typename FB>
__device__ __forceinline__ void multiply(float *lds, int n_steps, int wm, int wn, FA &&fetch_a, FB &&fetch_b, f32x16 &acc) {
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, part = tid >> 8;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.0f;
    if (n_steps <= 0) return;
    Fetched a[AHEAD], b[AHEAD];
#pragma unroll
    for (int d = 0; d < AHEAD; d++) { a[d] = fetch_a(d); b[d] = fetch_b(d); }
    for (int s0 = 0;; s0 += AHEAD) {
#pragma unroll
        for (int d = 0; d < AHEAD; d++) {
            if (s0 + d >= n_steps) goto done;
            float *ta = lds + (d & 1) * 2 * STAGE, *tb = ta + STAGE;
            stash<AKIND>(ta, a[d], tid);
            stash<BKIND>(tb, b[d], tid);
            __syncthreads();   // (a stage is rewritten two steps later, behind the barrier of the step between)
            a[d] = fetch_a(s0 + d + AHEAD);
            b[d] = fetch_b(s0 + d + AHEAD);
#pragma unroll
            for (int h = 0; h < KS / 16; h++) {
                const int g = part * (KS / 16) + h;
                const f4 fa = fragment<AKIND>(ta, wm + (lane & 31), g, half);
                const f4 fb = fragment<BKIND>(tb, wn + (lane & 31), g, half);
#pragma unroll
                for (int j = 0; j < 4; j++)
                    // operands swapped: lane l then holds output row wm + l%32 and columns
                    // wn + 8*(r/4) + 4*(l/32) + r%4
                    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[j], fa[j], acc, 0, 0, 0);
            }
        }
    }
done:
    __syncthreads();
    float *ex = lds + (tid & 255);
    if (part) {
#pragma unroll
        for (int r = 0; r < 16; r++) ex[r * 256] = acc[r];
    }
    __syncthreads();
    if (!part) {
#pragma unroll
        for (int r = 0; r < 16; r++) acc[r] += ex[r * 256];
    }
}

// Which expert owns row tile `tile`: every wavefront scans the counts 64 experts at a time.
__device__ __forceinline__ bool find_row_tile(const int32_t *cum, int n_experts, int tile, int &expert, int &begin, int &end) {
    const int lane = threadIdx.x & 63;
    int base = 0;
    for (int e0 = 0; e0 < n_experts; e0 += 64) {
        const int e = e0 + lane;
        int s = 0, cnt = 0;
        if (e < n_experts) { s = cum[e]; cnt = cum[e + 1] - s; }
        const int tiles = (cnt + TB - 1) / TB;
        int incl = tiles;
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(incl, o, 64);
            if (lane >= o) incl += v;
        }
        const unsigned long long mine = __ballot(tile >= base + incl - tiles && tile < base + incl);
        if (mine) {
            const int src = __ffsll(static_cast<long long>(mine)) - 1;
            expert = e0 + src;
            begin = __shfl(s + (tile - base - (incl - tiles)) * TB, src, 64);
            end = __shfl(s + cnt, src, 64);
            return true;
        }
        base += __shfl(incl, 63, 64);
    }
    return false;
}

#pragma clang fp contract(off)

// blockIdx.x = row tile (cut per expert), blockIdx.y = column tile (E_SWIGLU: 32 columns of gate and the
// same 32 of up, side by side in the tile)
template <int BKIND, int EPI, bool GATHER>
__global__ __launch_bounds__(THREADS, 4) void ggemm_f32_rows_kernel(const F32Params p) {
    __shared__ __attribute__((aligned(16))) float lds[4 * STAGE];
    int expert, m0, m_end;
    if (!find_row_tile(p.cum, p.n_experts, blockIdx.x, expert, m0, m_end)) return;   // (the whole block: blockIdx only)
    constexpr int COLS = EPI == E_SWIGLU ? TB / 2 : TB;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = ((wave >> 1) & 1) * 32, wn = (wave & 1) * 32;
    const int n0 = blockIdx.y * COLS;
    const int steps = (p.kc + KS - 1) / KS;
    // A: [row][c]
    const int arow = m0 + slot_row<F_CONTIG>(tid), ac = slot_c<F_CONTIG>(tid);
    const bool a_in = arow < m_end;
    const int64_t a_src = !a_in ? 0 : GATHER ? p.row_index[arow] : arow;
    const int last = steps * p.phases - 1;
    auto fetch_a = [&](int s) {
        s = min(s, last);
        const int ph = s >= steps ? 1 : 0, c = (s - ph * steps) * KS + ac;
        return fetch8((ph ? p.A[1] : p.A[0]) + a_src * p.lda + min(c, p.kc - 8), a_in && c < p.kc);
    };
    // B: W[g] as [n][k] (forward) or [c][col] with c the contraction index (input gradient)
    const int brow = slot_row<BKIND>(tid), bc = slot_c<BKIND>(tid);
    const int64_t b0[2] = {expert * p.strideB[0], expert * p.strideB[1]};
    auto fetch_b = [&](int s) {
        s = min(s, last);
        const int ph = s >= steps ? 1 : 0, c = (s - ph * steps) * KS + bc;
        if (BKIND == F_CONTIG) {
            const int which = EPI == E_SWIGLU ? brow >> 5 : ph;
            const int n = n0 + (EPI == E_SWIGLU ? brow & 31 : brow);
            return fetch8((which ? p.B[1] + b0[1] : p.B[0] + b0[0]) + static_cast<int64_t>(min(n, p.n_cols - 1)) * p.ldb +
                              min(c, p.kc - 8), n < p.n_cols && c < p.kc);
        }
        const int n = n0 + brow;
        return fetch8((ph ? p.B[1] + b0[1] : p.B[0] + b0[0]) + static_cast<int64_t>(min(c, p.kc - 1)) * p.ldb +
                          min(n, p.n_cols - 8), c < p.kc && n < p.n_cols);
    };
    f32x16 acc;
    multiply<F_CONTIG, BKIND>(lds, steps * p.phases, wm, wn, fetch_a, fetch_b, acc);
    const int m = m0 + wm + (lane & 31);
    if (EPI == E_SWIGLU) {
        // the up half goes to the wavefront that holds the gate half of the same rows and columns
        __syncthreads();
        float *ex = lds + ((wave >> 1) & 1) * 16 * 64;
        if (wn && wave < 4) {
#pragma unroll
            for (int r = 0; r < 16; r++) ex[r * 64 + lane] = acc[r];
        }
        __syncthreads();
        if (m >= m_end || wave >= 4) return;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int n = n0 + q * 8 + (lane >> 5) * 4;
            if (n >= p.n_cols) continue;
            const int64_t o = static_cast<int64_t>(m) * p.ldc + n;
            f4 v = {acc[q * 4], acc[q * 4 + 1], acc[q * 4 + 2], acc[q * 4 + 3]};
            *reinterpret_cast<f4 *>(p.C[wn ? 1 : 0] + o) = v;
            if (wn) continue;
            f4 h;
#pragma unroll
            for (int j = 0; j < 4; j++) h[j] = (v[j] / (1.0f + expf(-v[j]))) * ex[(q * 4 + j) * 64 + lane];
            *reinterpret_cast<f4 *>(p.C[2] + o) = h;
        }
        return;
    }
    if (m >= m_end || wave >= 4) return;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int n = n0 + wn + q * 8 + (lane >> 5) * 4;
        if (n >= p.n_cols) continue;
        const int64_t o = static_cast<int64_t>(m) * p.ldc + n;
        f4 v = {acc[q * 4], acc[q * 4 + 1], acc[q * 4 + 2], acc[q * 4 + 3]};
        if (EPI == E_SWIGLU_BWD) {
            const f4 a = *reinterpret_cast<const f4 *>(p.G + o), b = *reinterpret_cast<const f4 *>(p.U + o);
            f4 og, ou;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float sg = 1.0f / (1.0f + expf(-a[j]));
                ou[j] = v[j] * (a[j] / (1.0f + expf(-a[j])));
                og[j] = (v[j] * b[j]) * (sg * (1.0f + a[j] * (1.0f - sg)));
            }
            *reinterpret_cast<f4 *>(p.C[0] + o) = og;
            *reinterpret_cast<f4 *>(p.C[1] + o) = ou;
        } else {
            *reinterpret_cast<f4 *>(p.C[0] + o) = v;
        }
    }
}

// blockIdx = (column tile of dW, row tile of dW, expert and which of up to two weight gradients):
// dW[g][n][k] = sum_r dout[r][n] * in[r][k]
template <bool GATHER>
__global__ __launch_bounds__(THREADS, 4) void ggemm_f32_wgrad_kernel(const F32Params p) {
    __shared__ __attribute__((aligned(16))) float lds[4 * STAGE];
    const int expert = blockIdx.z % p.n_experts, which = blockIdx.z / p.n_experts;
    const int r0 = p.cum[expert], r1 = p.cum[expert + 1];
    const int n0 = blockIdx.y * TB, k0 = blockIdx.x * TB;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = ((wave >> 1) & 1) * 32, wn = (wave & 1) * 32;
    const int row = slot_row<F_STRIDED>(tid), c = slot_c<F_STRIDED>(tid);
    // the loads past the segment (and past the extents) re-read its last row (the last 8 columns)
    const int a_col = min(n0 + row, p.kc - 8), b_col = min(k0 + row, p.n_cols - 8);
    const bool a_in = n0 + row < p.kc, b_in = k0 + row < p.n_cols;
    auto fetch_a = [&](int s) {
        const int r = r0 + s * KS + c;
        return fetch8(p.A[which] + static_cast<int64_t>(min(r, r1 - 1)) * p.lda + a_col, a_in && r < r1);
    };
    // GATHER: the source row of this thread's slot AHEAD steps on, looked up one step before it is needed
    int src = GATHER && r1 > r0 ? p.row_index[min(r0 + c, r1 - 1)] : 0;
    auto fetch_b = [&](int s) {
        const int r = r0 + s * KS + c;
        const int64_t from = GATHER ? src : min(r, r1 - 1);
        if (GATHER) src = p.row_index[min(r + KS, r1 - 1)];
        return fetch8(p.B[0] + from * p.ldb + b_col, b_in && r < r1);
    };
    f32x16 acc;
    multiply<F_STRIDED, F_STRIDED>(lds, (r1 - r0 + KS - 1) / KS, wm, wn, fetch_a, fetch_b, acc);
    float *C = p.C[which] + expert * p.strideC[which];
    const int n = n0 + wm + (lane & 31);
    if (n >= p.kc || wave >= 4) return;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int k = k0 + wn + q * 8 + (lane >> 5) * 4;
        if (k >= p.n_cols) continue;
        f4 v = {acc[q * 4], acc[q * 4 + 1], acc[q * 4 + 2], acc[q * 4 + 3]};
        f4 *dst = reinterpret_cast<f4 *>(C + static_cast<int64_t>(n) * p.ldc + k);
        if ((p.accumulate >> which) & 1) v += *dst;
        *dst = v;
    }
}

inline bool mult8(int64_t v) { return v > 0 && v % 8 == 0; }
inline unsigned tiles_of(int v, int tile = TB) { return static_cast<unsigned>((v + tile - 1) / tile); }
inline bool fits31(int64_t v) { return v >= 0 && v < (1LL << 31); }

template <int BKIND, int EPI> int rows_launch(const F32Params &p, int64_t rows, void *stream) {
    const int64_t m_tiles = (rows + TB - 1) / TB + p.n_experts;
    const unsigned n_tiles = tiles_of(p.n_cols, EPI == E_SWIGLU ? TB / 2 : TB);
    if (m_tiles > 0x7fffffffLL || n_tiles > 65535) return OM_ERR_SHAPE;
    const dim3 grid(static_cast<unsigned>(m_tiles), n_tiles);
    if (p.row_index) ggemm_f32_rows_kernel<BKIND, EPI, true><<<grid, dim3(THREADS), 0, om_stream(stream)>>>(p);
    else ggemm_f32_rows_kernel<BKIND, EPI, false><<<grid, dim3(THREADS), 0, om_stream(stream)>>>(p);
    return om_launch_status();
}

}  // namespace

extern "C" int om_grouped_gemm_fwd_f32(const float *input, const float *weight, float *output,
                                       const int32_t *cum_token_counts, int64_t rows, int G, int N, int K,
                                       int64_t w_stride, void *stream) {
    if (rows < 0 || G < 1 || !mult8(N) || !mult8(K)) return OM_ERR_SHAPE;
    if (rows == 0) return OM_OK;
    if (!input || !weight || !output || !cum_token_counts) return OM_ERR_NULL;
    if (!om_aligned16(input) || !om_aligned16(weight) || !om_aligned16(output)) return OM_ERR_ALIGN;
    F32Params p = {};
    p.A[0] = input; p.B[0] = weight; p.C[0] = output; p.cum = cum_token_counts;
    p.lda = K; p.ldb = K; p.ldc = N;
    p.strideB[0] = w_stride ? w_stride : static_cast<int64_t>(N) * K;
    if (p.strideB[0] % 4 != 0) return OM_ERR_ALIGN;
    if (!fits31(rows * K) || !fits31(rows * N) || !fits31(p.strideB[0] * G)) return OM_ERR_SHAPE;
    p.n_experts = G; p.n_cols = N; p.kc = K; p.phases = 1;
    return rows_launch<F_CONTIG, E_STORE>(p, rows, stream);
}

extern "C" int om_grouped_gemm_dgrad_f32(const float *output_grad, const float *weight, float *input_grad,
                                         const int32_t *cum_token_counts, int64_t rows, int G, int N, int K,
                                         int64_t w_stride, void *stream) {
    if (rows < 0 || G < 1 || !mult8(N) || !mult8(K)) return OM_ERR_SHAPE;
    if (rows == 0) return OM_OK;
    if (!output_grad || !weight || !input_grad || !cum_token_counts) return OM_ERR_NULL;
    if (!om_aligned16(output_grad) || !om_aligned16(weight) || !om_aligned16(input_grad)) return OM_ERR_ALIGN;
    F32Params p = {};
    p.A[0] = output_grad; p.B[0] = weight; p.C[0] = input_grad; p.cum = cum_token_counts;
    p.lda = N; p.ldb = K; p.ldc = K;   // din[r][k] = sum_n dout[r][n] * W[n][k]: B is [c = n][row = k]
    p.strideB[0] = w_stride ? w_stride : static_cast<int64_t>(N) * K;
    if (p.strideB[0] % 4 != 0) return OM_ERR_ALIGN;
    if (!fits31(rows * K) || !fits31(rows * N) || !fits31(p.strideB[0] * G)) return OM_ERR_SHAPE;
    p.n_experts = G; p.n_cols = K; p.kc = N; p.phases = 1;
    return rows_launch<F_STRIDED, E_STORE>(p, rows, stream);
}

// g = x Wg^T, u = x Wu^T, h = silu(g) * u in one launch; `x_rows` != null: row r of x is row x_rows[r] of
// a [src_rows, H] matrix
extern "C" int om_merged_mlp_gate_up_fwd_f32(const float *x, const int32_t *x_rows, int64_t src_rows, const float *w_gate,
                                             const float *w_up, float *g, float *u, float *h,
                                             const int32_t *cum_token_counts, int64_t rows, int G, int I, int H,
                                             int64_t gate_stride, int64_t up_stride, void *stream) {
    if (rows < 0 || G < 1 || !mult8(I) || !mult8(H)) return OM_ERR_SHAPE;
    if (rows == 0) return OM_OK;
    if (!x || !w_gate || !w_up || !g || !u || !h || !cum_token_counts) return OM_ERR_NULL;
    if (!om_aligned16(x) || !om_aligned16(w_gate) || !om_aligned16(w_up) || !om_aligned16(g) || !om_aligned16(u) ||
        !om_aligned16(h))
        return OM_ERR_ALIGN;
    if (x_rows && src_rows < 1) return OM_ERR_SHAPE;
    F32Params p = {};
    p.A[0] = x; p.B[0] = w_gate; p.B[1] = w_up; p.C[0] = g; p.C[1] = u; p.C[2] = h;
    p.cum = cum_token_counts; p.row_index = x_rows;
    p.lda = H; p.ldb = H; p.ldc = I;
    p.strideB[0] = gate_stride ? gate_stride : static_cast<int64_t>(I) * H;
    p.strideB[1] = up_stride ? up_stride : static_cast<int64_t>(I) * H;
    if (p.strideB[0] % 4 != 0 || p.strideB[1] % 4 != 0) return OM_ERR_ALIGN;
    if (!fits31((x_rows ? src_rows : rows) * H) || !fits31(rows * I) || !fits31(p.strideB[0] * G) || !fits31(p.strideB[1] * G)) return OM_ERR_SHAPE;
    p.n_experts = G; p.n_cols = I; p.kc = H; p.phases = 1;
    return rows_launch<F_CONTIG, E_SWIGLU>(p, rows, stream);
}

// dg, du = SwiGLU backward of dh = dy W_down, in one launch
extern "C" int om_merged_mlp_down_dgrad_f32(const float *dy, const float *w_down, const float *g, const float *u, float *dg,
                                            float *du, const int32_t *cum_token_counts, int64_t rows, int G, int I, int H,
                                            int64_t w_stride, void *stream) {
    if (rows < 0 || G < 1 || !mult8(I) || !mult8(H)) return OM_ERR_SHAPE;
    if (rows == 0) return OM_OK;
    if (!dy || !w_down || !g || !u || !dg || !du || !cum_token_counts) return OM_ERR_NULL;
    if (!om_aligned16(dy) || !om_aligned16(w_down) || !om_aligned16(g) || !om_aligned16(u) || !om_aligned16(dg) ||
        !om_aligned16(du))
        return OM_ERR_ALIGN;
    F32Params p = {};
    p.A[0] = dy; p.B[0] = w_down; p.C[0] = dg; p.C[1] = du; p.G = g; p.U = u; p.cum = cum_token_counts;
    p.lda = H; p.ldb = I; p.ldc = I;   // B = W_down[g] [c = h][row = i]
    p.strideB[0] = w_stride ? w_stride : static_cast<int64_t>(H) * I;
    if (p.strideB[0] % 4 != 0) return OM_ERR_ALIGN;
    if (!fits31(rows * H) || !fits31(rows * I) || !fits31(p.strideB[0] * G)) return OM_ERR_SHAPE;
    p.n_experts = G; p.n_cols = I; p.kc = H; p.phases = 1;
    return rows_launch<F_STRIDED, E_SWIGLU_BWD>(p, rows, stream);
}

// dx = dg W_gate + du W_up, one accumulation over both
extern "C" int om_merged_mlp_gate_up_dgrad_f32(const float *dg, const float *du, const float *w_gate, const float *w_up,
                                               float *dx, const int32_t *cum_token_counts, int64_t rows, int G, int I,
                                               int H, int64_t gate_stride, int64_t up_stride, void *stream) {
    if (rows < 0 || G < 1 || !mult8(I) || !mult8(H)) return OM_ERR_SHAPE;
    if (rows == 0) return OM_OK;
    if (!dg || !du || !w_gate || !w_up || !dx || !cum_token_counts) return OM_ERR_NULL;
    if (!om_aligned16(dg) || !om_aligned16(du) || !om_aligned16(w_gate) || !om_aligned16(w_up) || !om_aligned16(dx))
        return OM_ERR_ALIGN;
    F32Params p = {};
    p.A[0] = dg; p.A[1] = du; p.B[0] = w_gate; p.B[1] = w_up; p.C[0] = dx; p.cum = cum_token_counts;
    p.lda = I; p.ldb = H; p.ldc = H;
    p.strideB[0] = gate_stride ? gate_stride : static_cast<int64_t>(I) * H;
    p.strideB[1] = up_stride ? up_stride : static_cast<int64_t>(I) * H;
    if (p.strideB[0] % 4 != 0 || p.strideB[1] % 4 != 0) return OM_ERR_ALIGN;
    if (!fits31(rows * H) || !fits31(rows * I) || !fits31(p.strideB[0] * G) || !fits31(p.strideB[1] * G)) return OM_ERR_SHAPE;
    p.n_experts = G; p.n_cols = H; p.kc = I; p.phases = 2;
    return rows_launch<F_STRIDED, E_STORE>(p, rows, stream);
}

namespace {
// n_sets 1 or 2: dW[s] (+)= dout[s]^T in, over the same rows of `input` (through input_rows when given)
int wgrad_f32_launch(int n_sets, const float *const *output_grad, const float *input, const int32_t *input_rows,
                     int64_t src_rows, float *const *weight_grad, const int32_t *cum_token_counts, int64_t rows, int G,
                     int N, int K, const int64_t *w_stride, void *stream, int accumulate) {
    if (rows < 0 || G < 1 || n_sets * static_cast<int64_t>(G) > 65535 || !mult8(N) || !mult8(K)) return OM_ERR_SHAPE;
    if (!cum_token_counts || (rows > 0 && !input)) return OM_ERR_NULL;
    if (!om_aligned16(input)) return OM_ERR_ALIGN;
    F32Params p = {};
    for (int s = 0; s < n_sets; s++) {
        if (!weight_grad[s] || (rows > 0 && !output_grad[s])) return OM_ERR_NULL;
        if (!om_aligned16(output_grad[s]) || !om_aligned16(weight_grad[s])) return OM_ERR_ALIGN;
        p.A[s] = output_grad[s];
        p.C[s] = weight_grad[s];
        p.strideC[s] = w_stride[s] ? w_stride[s] : static_cast<int64_t>(N) * K;
        if (p.strideC[s] % 4 != 0) return OM_ERR_ALIGN;
        if (!fits31(p.strideC[s] * G)) return OM_ERR_SHAPE;
    }
    p.B[0] = input; p.cum = cum_token_counts; p.row_index = input_rows;
    p.lda = N; p.ldb = K; p.ldc = K;
    if (!fits31((input_rows ? src_rows : rows) * K) || !fits31(rows * N) || tiles_of(N) > 65535) return OM_ERR_SHAPE;
    p.n_experts = G; p.n_cols = K; p.kc = N;
    p.accumulate = accumulate;
    const dim3 grid(tiles_of(K), tiles_of(N), n_sets * G);
    if (input_rows) ggemm_f32_wgrad_kernel<true><<<grid, dim3(THREADS), 0, om_stream(stream)>>>(p);
    else ggemm_f32_wgrad_kernel<false><<<grid, dim3(THREADS), 0, om_stream(stream)>>>(p);
    return om_launch_status();
}
}  // namespace

extern "C" int om_grouped_gemm_wgrad_f32(const float *output_grad, const float *input, float *weight_grad,
                                         const int32_t *cum_token_counts, int64_t rows, int G, int N, int K,
                                         int64_t w_stride, void *stream) {
    return wgrad_f32_launch(1, &output_grad, input, nullptr, 0, &weight_grad, cum_token_counts, rows, G, N, K, &w_stride,
                            stream, 0);
}

extern "C" int om_grouped_gemm_wgrad_f32_accumulate(const float *output_grad, const float *input,
                                                    float *weight_grad, const int32_t *cum_token_counts,
                                                    int64_t rows, int G, int N, int K, int64_t w_stride,
                                                    void *stream) {
    return wgrad_f32_launch(1, &output_grad, input, nullptr, 0, &weight_grad, cum_token_counts, rows, G, N, K, &w_stride,
                            stream, 1);
}

// dW_gate (+)= dg^T x (bit 0 of accumulate) and dW_up (+)= du^T x (bit 1) in one launch, the rows of x
// through x_rows when given
extern "C" int om_merged_mlp_gate_up_wgrad_f32(const float *dg, const float *du, const float *x, const int32_t *x_rows,
                                               int64_t src_rows, float *dw_gate, float *dw_up,
                                               const int32_t *cum_token_counts, int64_t rows, int G, int I, int H,
                                               int64_t gate_stride, int64_t up_stride, int accumulate, void *stream) {
    if (x_rows && rows > 0 && src_rows < 1) return OM_ERR_SHAPE;
    const float *dout[2] = {dg, du};
    float *dw[2] = {dw_gate, dw_up};
    const int64_t strides[2] = {gate_stride, up_stride};
    return wgrad_f32_launch(2, dout, x, x_rows, src_rows, dw, cum_token_counts, rows, G, I, H, strides, stream,
                            accumulate);
}

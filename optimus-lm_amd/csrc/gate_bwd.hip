// Backward of the router's gate projection `router_logits = self.gate(hidden_states)` (reference
// optimus/models/common/moe.py:456, the gate nn.Linear of optimus/models/olmoe/modeling_olmoe.py):
// the weight gradient dW[n,h] = sum_t dlogits[t,n] * x[t,h] (first part of this file) and the input
// gradient dx[t,h] = sum_n dlogits[t,n] * W[n,h] (second part).
//
// The product is [N x T] x [T x H] with N = number of experts (tens to a few hundred), H the
// hidden size and T the tokens: a tiny output and a long contraction.  A library GEMM gives it a
// handful of tiles, i.e. a handful of CUs.  Here the token range is split over many blocks; every
// block contracts its tokens for one 128-column slice of H on bf16 MFMA with fp32 accumulation
// and writes an fp32 partial; a second kernel adds the partials in a fixed order (deterministic)
// and rounds once.  dlogits (fp32) is rounded to bf16 on the way into LDS, the precision a bf16
// gate's backward has anyway; bf16 x bf16 products are exact in fp32.
//
// Both operands are stored token-major ([t][n], [t][h]) while the MFMA wants, per lane, 8
// consecutive contraction indices (tokens) of one row.  The tiles are kept in LDS as they lie in
// memory and the fragments come from the transposing LDS read (ds_read_b64_tr_b16).  HBM-bound:
// x is read once (2 B per element), dlogits comes from L2 for all but the first column slice.
#include "common.h"

#include <algorithm>

namespace {

typedef __attribute__((address_space(3))) s16x4 *lds_s16x4_ptr;
typedef __attribute__((ext_vector_type(8))) short s16x8;

constexpr int HT = 128;   // columns of H per block
constexpr int TC = 64;    // tokens per LDS stage

// Tile [TC token rows][R operand rows] of bf16, R*2-byte token rows, 16-byte chunk `ch` of token row
// `crow` stored at chunk position ch ^ ((crow & 3) << 2): the four token rows one transposing read
// touches fall into four different 64-byte bank windows.  Needs R >= 128 (16 chunks per row).
template <int R> __device__ __forceinline__ int tile_off(int crow, int ch) {
    return crow * (R * 2) + ((ch ^ ((crow & 3) << 2)) << 4);
}

// MFMA 32x32x16 operand fragment: lane l gets operand row m0 + l%32, tokens c0 + 8*(l/32) .. +7.
template <int R>
__device__ __forceinline__ bf16x8 read_frag(const char *tile, int c0, int m0, int lane) {
    const int i = lane & 15;
    const int r = i >> 2, q = i & 3;
    const int mb = ((lane >> 4) & 1) * 16;
    const int g2 = lane >> 5;
    const int m = m0 + mb + 4 * q;
    const int cr = c0 + 8 * g2 + r;
    const char *p = tile + tile_off<R>(cr, m >> 3) + (m & 7) * 2;
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(p));
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(p + 4 * R * 2));
    return __builtin_bit_cast(bf16x8, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

__device__ __forceinline__ uint32_t pack2(float a, float b) {
    typedef __attribute__((ext_vector_type(2))) float f32x2;
    f32x2 f = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
}

// grid (H / 128, splits); 256 threads.  NB accumulators per wavefront cover N = 32 NB rows of dW, of
// which the first n_real exist (the rest are zero columns of the dlogits tile); wavefront w owns
// the 32 columns [h0 + 32 w, h0 + 32 w + 32) of the block's slice and all rows of dW.
// SHARED: the partials are stored at device scope, for the block of the launch that adds them up.
template <int NB> constexpr int WGRAD_LDS = TC * HT * 2 + TC * (NB * 32 < 128 ? 128 : NB * 32) * 2;
template <int NB, bool SHARED>
__device__ __forceinline__ void gate_wgrad_block(const uint16_t *__restrict__ x, const float *__restrict__ dlogits, int64_t T, int H,
                                                 int n_real, int64_t tokens_per_split, float *partial, int slice, int split, char *lds) {
    constexpr int N = NB * 32;
    constexpr int RD = N < 128 ? 128 : N;       // LDS row length of the dlogits tile (elements)
    constexpr int XL = TC * HT / 8 / 256;       // 16-byte x chunks per thread per stage
    constexpr int DL = TC * N / 4 / 256;        // float4 dlogits loads per thread per stage
    char *const xs = lds, *const ds = lds + TC * HT * 2;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int h0 = slice * HT;
    const int64_t t_begin = static_cast<int64_t>(split) * tokens_per_split;
    int64_t t_end = t_begin + tokens_per_split;
    if (t_end > T) t_end = T;

    f32x16 acc[NB];
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[b][r] = 0.0f;

    u32x4 xq[XL];
    f32x4 dq[DL];
    auto fetch = [&](int64_t t0) {   // tokens past t_end contribute zeros
#pragma unroll
        for (int j = 0; j < XL; j++) {
            const int q = j * 256 + tid;
            const int64_t t = t0 + q / (HT / 8);
            xq[j] = u32x4{0, 0, 0, 0};
            const int hc = h0 + (q % (HT / 8)) * 8;     // the last column slice may be partial
            if (t < t_end && hc < H) xq[j] = *reinterpret_cast<const u32x4 *>(x + t * H + hc);
        }
#pragma unroll
        for (int j = 0; j < DL; j++) {
            const int q = j * 256 + tid;
            const int64_t t = t0 + q / (N / 4);
            const int col = (q % (N / 4)) * 4;
            dq[j] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (t < t_end && col < n_real) {
                const float *src = dlogits + t * n_real + col;
                if ((n_real & 3) == 0) {
                    dq[j] = *reinterpret_cast<const f32x4 *>(src);
                } else {
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (col + i < n_real) dq[j][i] = src[i];
                }
            }
        }
    };
    auto stash = [&]() {
#pragma unroll
        for (int j = 0; j < XL; j++) {
            const int q = j * 256 + tid;
            *reinterpret_cast<u32x4 *>(xs + tile_off<HT>(q / (HT / 8), q % (HT / 8))) = xq[j];
        }
#pragma unroll
        for (int j = 0; j < DL; j++) {
            const int q = j * 256 + tid;
            const int crow = q / (N / 4), n = (q % (N / 4)) * 4;
            u32x2 v;
            v[0] = pack2(dq[j][0], dq[j][1]);
            v[1] = pack2(dq[j][2], dq[j][3]);
            *reinterpret_cast<u32x2 *>(ds + tile_off<RD>(crow, n >> 3) + (n & 7) * 2) = v;
        }
    };

    if (t_begin < t_end) fetch(t_begin);
    for (int64_t t0 = t_begin; t0 < t_end; t0 += TC) {
        __syncthreads();             // the previous stage has been read
        stash();
        __syncthreads();
        if (t0 + TC < t_end) fetch(t0 + TC);   // in flight under the MFMAs below
#pragma unroll
        for (int kk = 0; kk < TC / 16; kk++) {
            const bf16x8 fx = read_frag<HT>(xs, kk * 16, wave * 32, lane);
#pragma unroll
            for (int b = 0; b < NB; b++) {
                const bf16x8 fd = read_frag<RD>(ds, kk * 16, b * 32, lane);
                // lane l then holds column h = l % 32 and rows n = 8*(r/4) + 4*(l/32) + r%4
                acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fd, fx, acc[b], 0, 0, 0);
            }
        }
    }
    const int h = h0 + wave * 32 + (lane & 31);
    float *out = partial + (static_cast<int64_t>(split) * n_real) * H + h;
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int n = b * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
            if (n >= n_real || h >= H) continue;
            if (SHARED) __hip_atomic_store(out + static_cast<int64_t>(n) * H, acc[b][r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            else out[static_cast<int64_t>(n) * H] = acc[b][r];
        }
}
template <int NB>
__global__ __launch_bounds__(256) void gate_wgrad_kernel(const uint16_t *__restrict__ x, const float *__restrict__ dlogits, int64_t T, int H,
                                                         int n_real, int64_t tokens_per_split, float *__restrict__ partial) {
    __shared__ __attribute__((aligned(16))) char lds[WGRAD_LDS<NB>];
    gate_wgrad_block<NB, false>(x, dlogits, T, H, n_real, tokens_per_split, partial, blockIdx.x, blockIdx.y, lds);
}

// The same for more than 128 experts, a multiple of 4 of them: 256 rows and 256 columns of dW per block of eight wavefronts (64 x
// 128 each), so that the fp32 dlogits are read once per 256 columns, in steps of 32 tokens.  x comes by direct loads two steps
// ahead through a ring of three, the dlogits through registers, two steps ahead too, and a pair of buffers.  Every step loads,
// past the last one that one again, so that the number of loads in flight is known.  The dlogits' loads are among those that the
// wait counts: `dlogits` is not __restrict__, so that the compiler may not move them over the assembly's memory clobbers.
// (The compiler's own wait for the dlogits of the next step counts its loads alone, and so waits for x of that step too: of its
// two steps x has one and a part.)
// us with the launch that adds the ranges, x out of the caches, before (128 columns a block, both operands through registers
// one stage ahead) -> now, 256 experts: hidden 7168, 64 tokens 19.3 -> 16.4, 2048 tokens 57 -> 41, 8192 tokens 115 -> 72; hidden
// 1624, 8176 tokens 60 -> 42.  160 experts, hidden 5120, 4096 tokens 56 -> 37.  Without a way out between the two steps of the
// loop's body: 8192 tokens 77.1 -> 70.8, 160 experts 36.9 -> 34.4, 513 tokens of 4096, 200 experts 23.5 -> 22.0, 8000 tokens 69.0 -> 69.7.
constexpr int WW_HT = 256, WW_TC = 32;
__global__ __launch_bounds__(512) void gate_wgrad_wide_kernel(const uint16_t *__restrict__ x, const float *dlogits, int64_t T, int H,
                                                              int N, int64_t tokens_per_split, float *__restrict__ partial) {
    constexpr int SLOTS = 3, XS = WW_TC * WW_HT * 2, DS = WW_TC * 256 * 2, XL = XS / 1024 / 8, DL = WW_TC * 256 / 4 / 512;
    constexpr int TM = 2, TN = 4;
    __shared__ __attribute__((aligned(1024))) char lds[SLOTS * XS + 2 * DS];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int h0 = blockIdx.x * WW_HT;
    const int64_t t_begin = static_cast<int64_t>(blockIdx.y) * tokens_per_split;
    const int tokens = static_cast<int>(max(min(tokens_per_split, T - t_begin), static_cast<int64_t>(0)));
    const int steps = (tokens + WW_TC - 1) / WW_TC;
    float *out = partial + static_cast<int64_t>(blockIdx.y) * N * H;
    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;
    if (steps > 0) {
        const uint32_t lds0 = lds_address(lds);
        char *const ds = lds + SLOTS * XS;
        auto x_row = [&](int l) { return (wave * XL + l) * 2 + (lane >> 5); };
        auto issue_x = [&](int s, int slot) {     // rows and columns past the end: valid memory; the rows are zeroed, the columns unused
            const int step = min(s, steps - 1) * WW_TC;
#pragma unroll
            for (int l = 0; l < XL; l++) {
                const int row = x_row(l), col = h0 + ((lane & 31) ^ ((row & 3) << 2)) * 8;
                dma16_lane(reinterpret_cast<const char *>(x + (t_begin + min(step + row, tokens - 1)) * H + min(col, H - 8)),
                           lds0 + slot * XS + (wave * XL + l) * 1024);
            }
        };
        f32x4 dq[2][DL];
        auto fetch_d = [&](int s, int set) {
            const int step = min(s, steps - 1) * WW_TC;
#pragma unroll
            for (int j = 0; j < DL; j++) {
                const int q = j * 512 + tid;
                dq[set][j] = *reinterpret_cast<const f32x4 *>(dlogits + (t_begin + min(step + q / 64, tokens - 1)) * N + min(q % 64 * 4, N - 4));
            }
        };
        auto stash_d = [&](int s, int set) {      // tokens and experts past the end: zeros
#pragma unroll
            for (int j = 0; j < DL; j++) {
                const int q = j * 512 + tid, crow = q / 64, n = q % 64 * 4;
                const bool inside = s * WW_TC + crow < tokens && n < N;
                const f32x4 d = dq[set][j];
                const u32x2 v = {inside ? pack2(d[0], d[1]) : 0u, inside ? pack2(d[2], d[3]) : 0u};
                *reinterpret_cast<u32x2 *>(ds + (s & 1) * DS + tile_off<256>(crow, n >> 3) + (n & 7) * 2) = v;
            }
        };
        issue_x(0, 0);
        fetch_d(0, 0);
        stash_d(0, 0);
        fetch_d(1, 1);
        issue_x(1, 1);
        fetch_d(2, 0);
        int slot = 0, free_slot = 2;
        auto step = [&](int s, int set) {         // set: the dlogits of step s + 1
            // This wavefront's part of x of step s has landed: younger are at least the dlogits of step s + 1, which this step stores
            // to LDS, and x of s + 1 (the dlogits of s + 2 too, but behind the last steps the compiler may leave out what nothing reads).
            // Behind the barrier everyone's has, the dlogits of step s are there, and step s - 1 has been read.
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(XL + DL) : "memory");
            if ((s + 1) * WW_TC > tokens) {
#pragma unroll
                for (int l = 0; l < XL; l++)
                    if (s * WW_TC + x_row(l) >= tokens) *reinterpret_cast<u32x4 *>(lds + slot * XS + (wave * XL + l) * 1024 + lane * 16) = u32x4{0, 0, 0, 0};
            }
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            stash_d(s + 1, set);
            issue_x(s + 2, free_slot);
            fetch_d(s + 3, set);
            const char *xs = lds + slot * XS, *dd = ds + (s & 1) * DS;
#pragma unroll
            for (int kk = 0; kk < WW_TC / 16; kk++) {
                bf16x8 fd[TM], fx[TN];
#pragma unroll
                for (int i = 0; i < TM; i++) fd[i] = read_frag<256>(dd, kk * 16, wm * 64 + i * 32, lane);
#pragma unroll
                for (int j = 0; j < TN; j++) fx[j] = read_frag<256>(xs, kk * 16, wn * 128 + j * 32, lane);
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++)
                        // lane l then holds column h = l % 32 and rows n = 8*(r/4) + 4*(l/32) + r%4
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fd[i], fx[j], acc[i][j], 0, 0, 0);
            }
            free_slot = slot;
            slot = slot == SLOTS - 1 ? 0 : slot + 1;
        };
        int s = 0;
        for (; s + 1 < steps; s += 2) {   // (where paths join, the compiler waits for every load in flight)
            step(s, 1);
            step(s + 1, 0);
        }
        if (s < steps) step(s, 1);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no load into LDS outlives the block
    }
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int n = wm * 64 + i * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const int h = h0 + wn * 128 + j * 32 + (lane & 31);
                if (n < N && h < H) out[static_cast<int64_t>(n) * H + h] = acc[i][j][r];
            }
        }
}

// dW = sum over splits, in split order; 4 elements per thread.
template <typename T>
__global__ __launch_bounds__(256) void gate_wgrad_reduce_kernel(const float *__restrict__ partial,
                                                                int splits, int64_t nh, T *__restrict__ dw) {
    const int64_t i = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 4;
    if (i >= nh) return;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < splits; k0 += 8) {   // eight loads in flight, added in split order
        f32x4 v[8];
#pragma unroll
        for (int u = 0; u < 8; u++)
            v[u] = (k0 + u < splits) ? *reinterpret_cast<const f32x4 *>(partial + (k0 + u) * nh + i)
                                     : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < 8; u++) { s[0] += v[u][0]; s[1] += v[u][1]; s[2] += v[u][2]; s[3] += v[u][3]; }
    }
    if constexpr (sizeof(T) == 4) {
        *reinterpret_cast<f32x4 *>(dw + i) = s;
    } else {
        u32x2 v;
        v[0] = pack2(s[0], s[1]);
        v[1] = pack2(s[2], s[3]);
        *reinterpret_cast<u32x2 *>(dw + i) = v;
    }
}

void gate_wgrad_reduce_launch(const float *ws, int splits, int64_t nh, void *dweight, int dweight_dtype, hipStream_t st) {
    const dim3 grid(static_cast<unsigned>((nh / 4 + 255) / 256));
    if (dweight_dtype == OM_F32) gate_wgrad_reduce_kernel<float><<<grid, dim3(256), 0, st>>>(ws, splits, nh, static_cast<float *>(dweight));
    else gate_wgrad_reduce_kernel<uint16_t><<<grid, dim3(256), 0, st>>>(ws, splits, nh, static_cast<uint16_t *>(dweight));
}

inline bool gate_wgrad_wide(int N) { return N > 128 && N % 4 == 0; }

// Token ranges: the blocks that the chip holds at once (two per CU, one of the wide kernel's), at least two stages of tokens each.
inline int gate_wgrad_splits(int64_t T, int H, int N) {
    const int64_t stages = (T + TC - 1) / TC;
    const int ht = gate_wgrad_wide(N) ? WW_HT : HT, blocks = gate_wgrad_wide(N) ? 256 : 512;
    int64_t want = blocks / ((H + ht - 1) / ht);
    if (want > stages / 2) want = stages / 2;
    if (want < 1) want = 1;
    if (want > 256) want = 256;
    return static_cast<int>(want);
}

inline bool gate_wgrad_shape_ok(int64_t T, int H, int N) {
    return T >= 0 && H > 0 && H % 8 == 0 && N >= 1 && N <= 256;   // 16-byte chunks of x
}

// ---- input gradient of the gate projection ---------------------------------------------------
// dx[t,h] = sum_n bf16(dlogits[t,n]) * W[n,h], optionally added to another gradient of the same
// tensor (the experts' input gradient): out = bf16(float(base) + float(bf16(sum))), the two
// roundings autograd's "matmul, then accumulate" has.  [T x N] x [N x H] with a short contraction:
// a block owns 128 tokens x 128 columns; W's [N x 128] slice sits in LDS as it lies in memory and is
// read through the transposing LDS read; a lane's dlogits fragment (8 consecutive n of one token)
// comes straight from global memory.  The results leave through per-wavefront LDS strips so that
// every store (and the read of `base`) covers whole 256-byte row segments.
constexpr int DG_HT = 128, DG_TOK = 128;
constexpr int DG_PITCH = DG_HT * 2 + 8;             // strip row pitch: conflict-free 8-byte accesses
constexpr int DG_STRIPS = 4 * 32 * DG_PITCH;        // four wavefronts x 32 token rows

inline size_t gate_dgrad_lds(int N) {
    const size_t w = static_cast<size_t>((N + 15) & ~15) * DG_HT * 2;
    return w > DG_STRIPS ? w : DG_STRIPS;
}

// The dlogits of four 16-slices are fetched together, one batch ahead of their MFMAs, and `base` before the
// first of them, so that a block waits for one miss and not for one per slice: 8192 tokens, hidden 7168, 256
// experts 146 -> 113 us, 16384 x 2048, 64 experts 41 -> 36, 3001 x 1000, 12 experts 10.8 -> 6.4.
// BATCHES * 4 slices of 16 experts; ALIGNED: rows of dlogits are whole 16-byte vectors (N % 4 == 0)
template <int BATCHES, bool ALIGNED>
__device__ __forceinline__ void gate_dgrad_block(const float *__restrict__ dlogits, const uint16_t *__restrict__ weight,
                                                 const uint16_t *base, uint16_t *out, int64_t T, int H, int N, int slice,
                                                 int64_t token_block, char *lds) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int h0 = slice * DG_HT;
    const int64_t t0 = token_block * DG_TOK + wave * 32;
    const int n_pad = (N + 15) & ~15;
    for (int q = tid; q < n_pad * (DG_HT / 8); q += 256) {
        const int n = q / (DG_HT / 8), ch = q % (DG_HT / 8);
        u32x4 v = {0, 0, 0, 0};
        if (n < N && h0 + ch * 8 < H)
            v = *reinterpret_cast<const u32x4 *>(weight + static_cast<int64_t>(n) * H + h0 + ch * 8);
        *reinterpret_cast<u32x4 *>(lds + tile_off<DG_HT>(n, ch)) = v;
    }
    // tokens past the end: the last one's, results unused; experts past the end: zeros
    const float *drow = dlogits + min(t0 + (lane & 31), T - 1) * N;
    f32x4 raw[2][4][2];
    auto fetch = [&](int batch, int set) {
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int half = 0; half < 2; half++) {
                const int n = batch * 64 + k * 16 + 8 * (lane >> 5) + 4 * half;
                if (ALIGNED) {
                    raw[set][k][half] = *reinterpret_cast<const f32x4 *>(drow + min(n, N - 4));
                } else {
#pragma unroll
                    for (int i = 0; i < 4; i++) raw[set][k][half][i] = drow[min(n + i, N - 1)];
                }
            }
    };
    auto packed = [&](int batch, int set, int k) -> bf16x8 {
        u32x4 v;
#pragma unroll
        for (int half = 0; half < 2; half++) {
            const int n = batch * 64 + k * 16 + 8 * (lane >> 5) + 4 * half;
            float d[4];
#pragma unroll
            for (int i = 0; i < 4; i++) d[i] = n + i < N ? raw[set][k][half][i] : 0.0f;
            v[2 * half] = pack2(d[0], d[1]);
            v[2 * half + 1] = pack2(d[2], d[3]);
        }
        return __builtin_bit_cast(bf16x8, v);
    };
    fetch(0, 0);
    constexpr int ITS = 32 * (DG_HT / 8) / 64;
    u32x4 other[ITS];
    if (base) {
#pragma unroll
        for (int it = 0; it < ITS; it++) {
            const int q = it * 64 + lane;
            other[it] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(   // read once
                base + min(t0 + q / (DG_HT / 8), T - 1) * H + min(h0 + (q % (DG_HT / 8)) * 8, H - 8)));
        }
    }
    __syncthreads();
    f32x16 acc[DG_HT / 32];
#pragma unroll
    for (int b = 0; b < DG_HT / 32; b++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[b][r] = 0.0f;
#pragma unroll
    for (int batch = 0; batch < BATCHES; batch++) {
        if (batch + 1 < BATCHES) fetch(batch + 1, (batch + 1) & 1);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int kk = batch * 64 + k * 16;
            if (kk >= n_pad) continue;        // (uniform; the weight tile ends here)
            const bf16x8 fd = packed(batch, batch & 1, k);
#pragma unroll
            for (int b = 0; b < DG_HT / 32; b++) {
                const bf16x8 fw = read_frag<DG_HT>(lds, kk, b * 32, lane);
                // lane l then holds token l % 32 and columns 32 b + 8*(r/4) + 4*(l/32) + r%4
                acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fw, fd, acc[b], 0, 0, 0);
            }
        }
    }
    __syncthreads();   // the weight tile is dead; its memory becomes the strips
    char *strip = lds + wave * (32 * DG_PITCH);
#pragma unroll
    for (int b = 0; b < DG_HT / 32; b++)
#pragma unroll
        for (int rq = 0; rq < 4; rq++) {
            u32x2 v;
            v[0] = pack2(acc[b][rq * 4], acc[b][rq * 4 + 1]);
            v[1] = pack2(acc[b][rq * 4 + 2], acc[b][rq * 4 + 3]);
            const int col = b * 32 + rq * 8 + (lane >> 5) * 4;
            *reinterpret_cast<u32x2 *>(strip + (lane & 31) * DG_PITCH + col * 2) = v;
        }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int it = 0; it < ITS; it++) {
        const int q = it * 64 + lane;
        const int row = q / (DG_HT / 8), ch = q % (DG_HT / 8);
        const int64_t tt = t0 + row;
        const int h = h0 + ch * 8;
        if (tt < T && h < H) {
            const char *sp = strip + row * DG_PITCH + ch * 16;
            const u32x2 lo = *reinterpret_cast<const u32x2 *>(sp);
            const u32x2 hi = *reinterpret_cast<const u32x2 *>(sp + 8);
            u32x4 v = {lo[0], lo[1], hi[0], hi[1]};
            const int64_t o = tt * H + h;
            if (base) {
                float a[8], g[8];
                Elem<uint16_t>::unpack(other[it], a);
                Elem<uint16_t>::unpack(v, g);
#pragma unroll
                for (int i = 0; i < 8; i++) a[i] = a[i] + g[i];
                v = Elem<uint16_t>::pack(a);
            }
            __builtin_nontemporal_store(v, reinterpret_cast<u32x4 *>(out + o));
        }
    }
}

template <int BATCHES, bool ALIGNED>
__global__ __launch_bounds__(256, 2) void gate_dgrad_kernel(const float *__restrict__ dlogits, const uint16_t *__restrict__ weight,
                                                            const uint16_t *base, uint16_t *out, int64_t T, int H, int N) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    gate_dgrad_block<BATCHES, ALIGNED>(dlogits, weight, base, out, T, H, N, blockIdx.x, blockIdx.y, lds);
}

// Both gradients of the gate in one launch, up to 64 experts: either alone leaves most of the chip idle at small sizes and waits for one miss
// after the other.  us, two launches -> one: 2048 tokens, hidden 256, 8 experts 5.8 + 4.8 (and 2.9 for the sum of the ranges) -> 7.4 with that
// sum; 3001 of 1000, 12 experts 6.4 + 5.6 -> 7.6; 512 of 2048, 64 experts 7.2 + 5.9 -> 7.7; 16384 of 2048 34.8 + 22.6 -> 51.6.  Blocks 0 .. slices * splits - 1 are those of the weight gradient, the
// others those of the input gradient.  TOGETHER: the block that finishes a slice's last token range adds the ranges up (`done`: a count
// per slice, zero before the launch); else a launch behind this one does.
template <int NB, bool ALIGNED, bool TOGETHER, typename TD>
__global__ __launch_bounds__(256, 2) void gate_bwd_kernel(const uint16_t *__restrict__ x, const float *__restrict__ dlogits,
                                                          const uint16_t *__restrict__ weight, const uint16_t *base, uint16_t *dx,
                                                          int64_t T, int H, int N, int64_t tokens_per_split, int splits, float *partial,
                                                          unsigned *done, TD *dweight) {
    __shared__ __attribute__((aligned(16))) char lds[WGRAD_LDS<NB> > DG_STRIPS ? WGRAD_LDS<NB> : DG_STRIPS];
    static_assert(NB * 32 * DG_HT * 2 <= DG_STRIPS && HT == DG_HT, "the weight tile lies in the strips' place");
    const int slices = (H + HT - 1) / HT, b = blockIdx.x, slice = b % slices;
    if (b >= slices * splits) {
        gate_dgrad_block<1, ALIGNED>(dlogits, weight, base, dx, T, H, N, slice, b / slices - splits, lds);
        return;
    }
    gate_wgrad_block<NB, TOGETHER>(x, dlogits, T, H, N, tokens_per_split, partial, slice, b / slices, lds);
    if (!TOGETHER) return;
    // This block's partials are stored, and the others' read, at device scope, and the stores have completed before the block is
    // counted, so the last one sees them all (without writing back an L2: see grad_sumsq_kernel in gradnorm.hip).
    __shared__ bool last;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0)
        last = __hip_atomic_fetch_add(done + slice, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == static_cast<unsigned>(splits) - 1;
    __syncthreads();
    if (!last) return;
    const int h = slice * HT + threadIdx.x % HT;
    if (h >= H) return;
    const int64_t nh = static_cast<int64_t>(N) * H;
    constexpr int ROWS = 4, STEP = 256 / HT;     // rows of dW in flight per thread, and how far they are apart
    for (int n0 = threadIdx.x / HT; n0 < N; n0 += ROWS * STEP) {
        const float *from[ROWS];
        float s[ROWS] = {};
#pragma unroll
        for (int i = 0; i < ROWS; i++) from[i] = partial + static_cast<int64_t>(min(n0 + i * STEP, N - 1)) * H + h;
        for (int k0 = 0; k0 < splits; k0 += 8) {   // as gate_wgrad_reduce_kernel adds them
            float v[8][ROWS];
#pragma unroll
            for (int u = 0; u < 8; u++)
#pragma unroll
                for (int i = 0; i < ROWS; i++)
                    v[u][i] = __hip_atomic_load(from[i] + min(k0 + u, splits - 1) * nh, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int u = 0; u < 8; u++)
#pragma unroll
                for (int i = 0; i < ROWS; i++) s[i] += k0 + u < splits ? v[u][i] : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < ROWS; i++)
            if (n0 + i * STEP < N) Elem<TD>::store(dweight + static_cast<int64_t>(n0 + i * STEP) * H + h, s[i]);
    }
}

// The same for more than 64 experts, a multiple of 16 of them: with many experts a block's dlogits and weights are more
// than its results.  A block of eight wavefronts keeps the dlogits of its 256 tokens in registers (bf16, MFMA layout) and goes
// through a range of 64-column slices of the weight, which come by direct loads two slices ahead through a ring of three;
// `base` comes one slice ahead (not __restrict__: its loads are counted by a wait and must stay between the assembly
// statements around them).  What is left to bound it is `base` and dx.
// us, `base` and weights out of the caches, 256 experts, before (128 tokens x 128 columns a block, dlogits in fp32 once per 128
// columns) -> now: hidden 7168, 64 tokens 18.9 -> 11.3, 512 tokens 19.7 -> 16.4, 8192 tokens 113.9 -> 71.0 (4.0 TB/s of base,
// dx and dlogits); 128 experts, hidden 4096, 4096 tokens 29.3 -> 24.3.  Hidden sizes that are not a multiple of 64, `base` and
// dx past the caches / through them: 256 experts, hidden 7000, 8192 tokens (133 before) 135 / 98, 1624, 17000 tokens (69) 65 / 50;
// 128 experts, hidden 7000, 8192 tokens (91) 130 / 76.  With everything in the caches, as a repeated call alone finds it, the
// kernel before was the faster one from 200 tokens up to about 6 M elements (256 experts, hidden 2048, 1024 tokens 10.3 against
// 12.0); behind a layer's expert products, which leave the gate's weight to memory, 16.0 against 12.9.
constexpr int DW_HT = 64, DW_TOK = 256, DW_PITCH = DW_HT * 2 + 8;

// NK * 16 >= N experts; grid (column ranges of `tiles` slices, T / 256)
// LINES: the 128-byte pieces of `base` and dx that a slice takes are whole lines and pass the caches by; a line of two pieces would
// be moved twice.
template <int NK, bool BASE, bool LINES>
__global__ __launch_bounds__(512) void gate_dgrad_wide_kernel(const float *__restrict__ dlogits, const uint16_t *__restrict__ weight,
                                                              const uint16_t *base, uint16_t *out, int64_t T, int H, int N, int tiles) {
    constexpr int SLOTS = 3, SLOT = NK * 16 * DW_HT * 2, LOADS = SLOT / 1024 / 8, ITS = 32 * (DW_HT / 8) / 64;
    __shared__ __attribute__((aligned(1024))) char lds[SLOTS * SLOT + 8 * 32 * DW_PITCH];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int64_t t0 = static_cast<int64_t>(blockIdx.y) * DW_TOK + wave * 32;
    const int first = blockIdx.x * tiles, steps = min(tiles, (H + DW_HT - 1) / DW_HT - first);
    char *strip = lds + SLOTS * SLOT + wave * (32 * DW_PITCH);
    // chunk c (16 bytes) of weight row n at c ^ 4 * (n / 2 % 2): the four rows of a transposing read in different banks
    const uint32_t lds0 = lds_address(lds);
    const uint16_t *src[LOADS];
    int col[LOADS];
#pragma unroll
    for (int l = 0; l < LOADS; l++) {
        const int n = (wave * LOADS + l) * 8 + (lane >> 3);
        col[l] = first * DW_HT + ((lane & 7) ^ (((n >> 1) & 1) << 2)) * 8;
        src[l] = weight + static_cast<int64_t>(min(n, N - 1)) * H;     // (rows past the end are not multiplied)
    }
    auto issue = [&](int s, int slot) {          // columns past the end: the last chunk again, results unused
#pragma unroll
        for (int l = 0; l < LOADS; l++)
            dma16_lane(reinterpret_cast<const char *>(src[l] + min(col[l] + s * DW_HT, H - 8)), lds0 + slot * SLOT + (wave * LOADS + l) * 1024);
    };
    issue(0, 0);
    if (steps > 1) issue(1, 1);
    u32x4 other[2][ITS];
    auto fetch_base = [&](int s, int set) {
#pragma unroll
        for (int it = 0; it < ITS; it++) {
            const int q = it * 64 + lane;
            const u32x4 *from = reinterpret_cast<const u32x4 *>(
                base + min(t0 + q / (DW_HT / 8), T - 1) * H + min((first + s) * DW_HT + (q % (DW_HT / 8)) * 8, H - 8));
            other[set][it] = LINES ? __builtin_nontemporal_load(from) : *from;   // read once
        }
    };
    if (BASE) fetch_base(0, 0);
    bf16x8 fd[NK];                               // tokens past the end: the last one's, results unused
    const float *drow = dlogits + min(t0 + (lane & 31), T - 1) * N + 8 * (lane >> 5);
#pragma unroll
    for (int k = 0; k < NK; k++) {
        const f32x4 lo = *reinterpret_cast<const f32x4 *>(drow + min(k * 16, N - 16));
        const f32x4 hi = *reinterpret_cast<const f32x4 *>(drow + min(k * 16, N - 16) + 4);
        fd[k] = __builtin_bit_cast(bf16x8, u32x4{pack2(lo[0], lo[1]), pack2(lo[2], lo[3]), pack2(hi[0], hi[1]), pack2(hi[2], hi[3])});
    }
    const int r16 = (lane & 15) >> 2, cr = 8 * (lane >> 5) + r16, m = ((lane >> 4) & 1) * 16 + 4 * (lane & 3);
    int frag[2];
#pragma unroll
    for (int b = 0; b < 2; b++) frag[b] = cr * 128 + ((((b * 32 + m) >> 3) ^ (((cr >> 1) & 1) << 2)) << 4) + (m & 7) * 2;
    int slot = 0, free_slot = 2;
    auto step = [&](int s, int set) {
        // The wavefront's weights of step s have landed: younger are the next step's, and `base`'s loads of this one (stores
        // may be skipped and do not count).  Behind the barrier everyone's have, and everyone has read step s - 1.
        if (s + 1 < steps) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS + (BASE ? ITS : 0)) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (BASE && s + 1 < steps) fetch_base(s + 1, set ^ 1);
        f32x16 acc[2];
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[b][r] = 0.0f;
        const char *tile = lds + slot * SLOT;
#pragma unroll
        for (int k = 0; k < NK; k++) {
            if (k * 16 >= N) continue;           // (uniform)
#pragma unroll
            for (int b = 0; b < 2; b++) {
                const char *p = tile + frag[b] + k * 2048;
                const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(p));
                const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(p + 4 * 128));
                const bf16x8 fw = __builtin_bit_cast(bf16x8, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                // lane l then holds token l % 32 and columns 32 b + 8*(r/4) + 4*(l/32) + r%4
                acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fw, fd[k], acc[b], 0, 0, 0);
            }
        }
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int rq = 0; rq < 4; rq++) {
                const u32x2 v = {pack2(acc[b][rq * 4], acc[b][rq * 4 + 1]), pack2(acc[b][rq * 4 + 2], acc[b][rq * 4 + 3])};
                *reinterpret_cast<u32x2 *>(strip + (lane & 31) * DW_PITCH + (b * 32 + rq * 8 + (lane >> 5) * 4) * 2) = v;
            }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int it = 0; it < ITS; it++) {
            const int q = it * 64 + lane, row = q / (DW_HT / 8), ch = q % (DW_HT / 8);
            const int64_t tt = t0 + row;
            const int h = (first + s) * DW_HT + ch * 8;
            const char *sp = strip + row * DW_PITCH + ch * 16;
            const u32x2 lo = *reinterpret_cast<const u32x2 *>(sp), hi = *reinterpret_cast<const u32x2 *>(sp + 8);
            u32x4 v = {lo[0], lo[1], hi[0], hi[1]};
            if (BASE) {
                float a[8], g[8];
                Elem<uint16_t>::unpack(other[set][it], a);
                Elem<uint16_t>::unpack(v, g);
#pragma unroll
                for (int i = 0; i < 8; i++) a[i] = a[i] + g[i];
                v = Elem<uint16_t>::pack(a);
            }
            if (tt < T && h < H) {
                u32x4 *to = reinterpret_cast<u32x4 *>(out + tt * H + h);
                if (LINES) __builtin_nontemporal_store(v, to);
                else *to = v;
            }
        }
        if (s + 2 < steps) issue(s + 2, free_slot);
        free_slot = slot;
        slot = slot == SLOTS - 1 ? 0 : slot + 1;
    };
    for (int s = 0; s < steps; s += 2) {
        step(s, 0);
        if (s + 1 < steps) step(s + 1, 1);
    }
}

// Whether the last block of a slice adds its token ranges: where it has at most two rounds of loads to wait for.  It stores and loads
// past the L2s: 8 experts, 16 ranges 2 us for the launch of 3; with a round per eight rows and eight ranges 12 experts, 23 ranges
// took 10 us for 4, 64 experts, 4 ranges 17 for 5.
inline bool gate_bwd_together(int splits, int N) { return (N + 7) / 8 * ((splits + 7) / 8) <= 2; }

}  // namespace

extern "C" int om_router_gate_dgrad(const float *dlogits, const void *gate_weight, const void *base,
                                    void *dx, int64_t T, int H, int N, void *stream) {
    if (T < 0 || H < 8 || H % 8 != 0 || N < 1 || N > 256) return OM_ERR_SHAPE;
    if (T == 0) return OM_OK;
    if (!dlogits || !gate_weight || !dx) return OM_ERR_NULL;
    if (!om_aligned16(dlogits) || !om_aligned16(gate_weight) || !om_aligned16(dx) || !om_aligned16(base))
        return OM_ERR_ALIGN;
    hipStream_t st = om_stream(stream);
    const float *dl = dlogits;
    const uint16_t *w = static_cast<const uint16_t *>(gate_weight), *bp = static_cast<const uint16_t *>(base);
    uint16_t *dp = static_cast<uint16_t *>(dx);
    const int64_t wide_blocks = (T + DW_TOK - 1) / DW_TOK;
    if (N > 64 && N % 16 == 0 && wide_blocks <= 65535) {
        const int slices = (H + DW_HT - 1) / DW_HT, ranges = static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(slices, 256 / wide_blocks)));
        const int tiles = (slices + ranges - 1) / ranges;
        const dim3 grid((slices + tiles - 1) / tiles, static_cast<unsigned>(wide_blocks));
        const bool lines = H % 64 == 0 && reinterpret_cast<uintptr_t>(base) % 128 == 0 && reinterpret_cast<uintptr_t>(dx) % 128 == 0;
#define OM_WIDE(NK, BASE)                                                                                        \
    do {                                                                                                         \
        if (lines) gate_dgrad_wide_kernel<NK, BASE, true><<<grid, dim3(512), 0, st>>>(dl, w, bp, dp, T, H, N, tiles); \
        else gate_dgrad_wide_kernel<NK, BASE, false><<<grid, dim3(512), 0, st>>>(dl, w, bp, dp, T, H, N, tiles); \
    } while (0)
        if (N <= 128 && base) OM_WIDE(8, true);
        else if (N <= 128) OM_WIDE(8, false);
        else if (base) OM_WIDE(16, true);
        else OM_WIDE(16, false);
#undef OM_WIDE
        return om_launch_status();
    }
    const int64_t t_blocks = (T + DG_TOK - 1) / DG_TOK;
    if (t_blocks > 65535) {
        // the token blocks ride on the grid's second dimension: split long inputs into several launches
        const int64_t per = 65535LL * DG_TOK;
        for (int64_t done = 0; done < T; done += per) {
            const int64_t cnt = T - done < per ? T - done : per;
            const int rc = om_router_gate_dgrad(
                dlogits + done * N, gate_weight,
                base ? static_cast<const uint16_t *>(base) + done * H : nullptr,
                static_cast<uint16_t *>(dx) + done * H, cnt, H, N, stream);
            if (rc != OM_OK) return rc;
        }
        return OM_OK;
    }
    const dim3 grid((H + DG_HT - 1) / DG_HT, static_cast<unsigned>(t_blocks));
#define OM_DGRAD(BATCHES, ALIGNED)                                                                          \
    gate_dgrad_kernel<BATCHES, ALIGNED><<<grid, dim3(256), gate_dgrad_lds(N), st>>>(dl, w, bp, dp, T, H, N)
    if (N % 4 != 0) {
        if (N <= 64) OM_DGRAD(1, false);
        else OM_DGRAD(4, false);
    } else if (N <= 64) OM_DGRAD(1, true);
    else if (N <= 128) OM_DGRAD(2, true);
    else OM_DGRAD(4, true);
#undef OM_DGRAD
    return om_launch_status();
}

namespace {
// (with the weight gradient's blocks less than 2^32 threads)
bool gate_bwd_shape_ok(int64_t T, int H, int N) {
    return T >= 1 && H >= 8 && H % 8 == 0 && N >= 1 && N <= 64 && (T + DG_TOK - 1) / DG_TOK * ((H + DG_HT - 1) / DG_HT) <= (1 << 22);
}
int64_t gate_bwd_counts(int H) { return ((H + HT - 1) / HT + 3) / 4 * 4; }   // (16-byte aligned behind them)
}  // namespace

// workspace of om_router_softmax_bwd: counts, dlogits, partials
extern "C" int64_t om_router_softmax_bwd_workspace_bytes(int64_t T, int H, int N) {
    if (!gate_bwd_shape_ok(T, H, N)) return OM_ERR_SHAPE;
    return (gate_bwd_counts(H) + (T * N + 3) / 4 * 4 + static_cast<int64_t>(gate_wgrad_splits(T, H, N)) * N * H) * 4;
}

extern "C" int om_router_softmax_bwd(const void *x, const void *gate_weight, const void *logits, int logits_dtype, const int64_t *experts,
                                     const void *dweights, int dweights_dtype, const void *dlogits, const void *base, void *dx,
                                     void *dweight, int dweight_dtype, int64_t T, int H, int N, int K, int norm_topk_prob,
                                     void *workspace, int64_t workspace_bytes, void *stream) {
    for (int dtype : {logits_dtype, dweights_dtype, dweight_dtype})
        if (dtype != OM_BF16 && dtype != OM_F32) return OM_ERR_DTYPE;
    if (!gate_bwd_shape_ok(T, H, N) || K < 1 || K > N) return OM_ERR_SHAPE;
    if (!x || !gate_weight || !logits || !experts || !dweights || !dx || !dweight || !workspace) return OM_ERR_NULL;
    for (const void *p : {x, gate_weight, base, static_cast<const void *>(dx), static_cast<const void *>(dweight), static_cast<const void *>(workspace)})
        if (!om_aligned16(p)) return OM_ERR_ALIGN;
    if (workspace_bytes < om_router_softmax_bwd_workspace_bytes(T, H, N)) return OM_ERR_WORKSPACE;
    const int splits = gate_wgrad_splits(T, H, N), slices = (H + HT - 1) / HT;
    const int64_t nh = static_cast<int64_t>(N) * H;
    unsigned *done = static_cast<unsigned *>(workspace);
    float *dl = static_cast<float *>(workspace) + gate_bwd_counts(H), *ws = dl + (T * N + 3) / 4 * 4;
    hipStream_t st = om_stream(stream);
    om_launch_softmax_bwd(logits, logits_dtype, experts, dweights, dweights_dtype, dlogits, T, N, K, norm_topk_prob, dl, done, slices, st);
    const int64_t stages = (T + TC - 1) / TC, tokens_per_split = (stages + splits - 1) / splits * TC;
    const dim3 grid(slices * splits + static_cast<unsigned>((T + DG_TOK - 1) / DG_TOK) * slices);
    const bool together = gate_bwd_together(splits, N);
#define OM_BWD(NB, ALIGNED, TOGETHER, TD)                                                                                                         gate_bwd_kernel<NB, ALIGNED, TOGETHER, TD><<<grid, dim3(256), 0, st>>>(static_cast<const uint16_t *>(x), dl, static_cast<const uint16_t *>(gate_weight),                                                                  static_cast<const uint16_t *>(base), static_cast<uint16_t *>(dx), T, H, N,                                                                      tokens_per_split, splits, ws, done, static_cast<TD *>(dweight))
#define OM_BWD_N(TD)                                       \
    do {                                                   \
        if (together && N % 4 == 0) OM_BWD(1, true, true, TD);  \
        else if (together) OM_BWD(1, false, true, TD);     \
        else if (N <= 32 && N % 4 == 0) OM_BWD(1, true, false, TD); \
        else if (N <= 32) OM_BWD(1, false, false, TD);     \
        else if (N % 4 == 0) OM_BWD(2, true, false, TD);   \
        else OM_BWD(2, false, false, TD);                  \
    } while (0)
    if (dweight_dtype == OM_F32) OM_BWD_N(float);
    else OM_BWD_N(uint16_t);
#undef OM_BWD_N
#undef OM_BWD
    if (!together) gate_wgrad_reduce_launch(ws, splits, nh, dweight, dweight_dtype, st);
    return om_launch_status();
}

extern "C" int64_t om_router_gate_wgrad_workspace_bytes(int64_t T, int H, int N) {
    if (!gate_wgrad_shape_ok(T, H, N)) return OM_ERR_SHAPE;
    return static_cast<int64_t>(gate_wgrad_splits(T, H, N)) * N * H * 4;
}

extern "C" int om_router_gate_wgrad(const void *x, const float *dlogits, int64_t T, int H, int N,
                                    void *dweight, int dweight_dtype, void *workspace,
                                    int64_t workspace_bytes, void *stream) {
    if (dweight_dtype != OM_BF16 && dweight_dtype != OM_F32) return OM_ERR_DTYPE;
    if (!gate_wgrad_shape_ok(T, H, N)) return OM_ERR_SHAPE;
    if (!dweight || !workspace) return OM_ERR_NULL;
    if (T > 0 && (!x || !dlogits)) return OM_ERR_NULL;
    if (!om_aligned16(x) || !om_aligned16(dlogits) || !om_aligned16(dweight) || !om_aligned16(workspace))
        return OM_ERR_ALIGN;
    const int splits = gate_wgrad_splits(T, H, N);
    const int64_t nh = static_cast<int64_t>(N) * H;
    if (workspace_bytes < splits * nh * 4) return OM_ERR_WORKSPACE;
    hipStream_t st = om_stream(stream);
    const int64_t stages = (T + TC - 1) / TC;
    const int64_t tokens_per_split = (stages + splits - 1) / splits * TC;
    const dim3 grid((H + HT - 1) / HT, splits);
    const uint16_t *xp = static_cast<const uint16_t *>(x);
    float *ws = static_cast<float *>(workspace);
    if (gate_wgrad_wide(N))
        gate_wgrad_wide_kernel<<<dim3((H + WW_HT - 1) / WW_HT, splits), dim3(512), 0, st>>>(xp, dlogits, T, H, N, tokens_per_split, ws);
    else if (N <= 32)
        gate_wgrad_kernel<1><<<grid, dim3(256), 0, st>>>(xp, dlogits, T, H, N, tokens_per_split, ws);
    else if (N <= 64)
        gate_wgrad_kernel<2><<<grid, dim3(256), 0, st>>>(xp, dlogits, T, H, N, tokens_per_split, ws);
    else if (N <= 128)
        gate_wgrad_kernel<4><<<grid, dim3(256), 0, st>>>(xp, dlogits, T, H, N, tokens_per_split, ws);
    else
        gate_wgrad_kernel<8><<<grid, dim3(256), 0, st>>>(xp, dlogits, T, H, N, tokens_per_split, ws);
    gate_wgrad_reduce_launch(ws, splits, nh, dweight, dweight_dtype, st);
    return om_launch_status();
}

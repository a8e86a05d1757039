// Router gate projection split over slices of the hidden size, logits[t,n] = sum_h x[t,h] * W[n,h] in fp32 from bf16
// operands (the DeepSeek-V3 router: optimus/models/deepseek_v3/modeling_deepseek_v3.py:160 casts
// both operands to float32 and calls F.linear; bf16 x bf16 products are exact in fp32, so this is
// that value up to the order of the sum).
//
// With a few hundred experts the gate weight is megabytes (256 x 7168 bf16 = 3.7 MB).  A block that
// covers 32 tokens re-reads all of it from L2, and that traffic, not the read of x, bounds the
// launch.  Here a block covers 128 tokens and a slice of H; the weight tile of a 64-wide step is
// fetched once per block into LDS with direct loads and shared by its wavefronts, and the slices of
// H are added by a second kernel (or the routing's) in slice order (deterministic).  Weight traffic
// falls by 4x, the blocks still fill the chip through the split of H.
// Up to 64 experts: gate_logits_split_kernel, four wavefronts of 32 tokens whose token fragments come
// straight from global memory in MFMA layout, several blocks on a CU.  More: gate_logits_wide_kernel.
#include "common.h"

#include <algorithm>

namespace {

typedef const __attribute__((address_space(1))) void *glb_ptr;
typedef __attribute__((address_space(3))) void *lds_ptr;

constexpr int GT = 128;   // tokens per block
constexpr int GK = 64;    // columns of H per LDS stage

// W tile [rows][64 h] as 128-byte rows, 16-byte chunk c of row r stored at c ^ ((r >> 1) & 7):
// conflict-free for 16-byte fragment reads of 32 consecutive rows per half-wavefront.
__device__ __forceinline__ int w_off(int row, int ch) { return row * 128 + ((ch ^ ((row >> 1) & 7)) << 4); }

// grid (ceil(T / 128), splits); 256 threads; NB = ceil(N / 32) accumulators per wavefront
template <int NB>
__global__ __launch_bounds__(256) void gate_logits_split_kernel(const uint16_t *__restrict__ x,
                                                                const uint16_t *__restrict__ w,
                                                                int64_t T, int H, int N, int h_per_split,
                                                                float *__restrict__ partial) {
    constexpr int NP = NB * 32;                 // experts rounded up to MFMA blocks
    constexpr int W_LOADS = NP / 8 / 4;         // 1 KB direct loads per wavefront per stage
    __shared__ __attribute__((aligned(1024))) char ws[2][NP * 128];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t t0 = static_cast<int64_t>(blockIdx.x) * GT + wave * 32;
    const int h_begin = blockIdx.y * h_per_split;
    // H is any multiple of 8: the last slice may be shorter and its last step may hold fewer than 64 columns.  Its token
    // fragments past the end are zeros, its weight loads past the end re-read the last 8 columns.
    const int h_len = min(H - h_begin, h_per_split), steps = (h_len + GK - 1) / GK;
    // token fragment: lane l holds token t0 + l % 32, 8 consecutive h starting at 8 * (l / 32)
    int64_t ta = t0 + (lane & 31);
    if (ta >= T) ta = T - 1;                    // rows past the end: valid memory, result unused
    const uint16_t *xp = x + ta * H + h_begin + (lane >> 5) * 8;
    // weight loads: load i of this wavefront fills LDS rows (wave * W_LOADS + i) * 8 .. + 7; lane l
    // fetches row + l / 8, chunk (l % 8) ^ swizzle, so that the chunk lands at its swizzled place
    const uint16_t *wp[W_LOADS];
#pragma unroll
    for (int i = 0; i < W_LOADS; i++) {
        const int row = (wave * W_LOADS + i) * 8 + (lane >> 3);
        const int ch = (lane & 7) ^ ((row >> 1) & 7);
        const int src = row < N ? row : N - 1;  // padding rows repeat the last expert (never stored)
        wp[i] = w + static_cast<int64_t>(src) * H + h_begin + ch * 8;
    }
    auto issue_w = [&](int s, int stage) {
        const bool tail = (s + 1) * GK > h_len;          // block-uniform
        const int chunks = (h_len - s * GK) >> 3;         // 8-column chunks the step holds
#pragma unroll
        for (int i = 0; i < W_LOADS; i++) {
            const uint16_t *src = wp[i] + s * GK;
            if (tail) {
                const int row = (wave * W_LOADS + i) * 8 + (lane >> 3);
                const int ch = (lane & 7) ^ ((row >> 1) & 7);
                src -= max(ch - (chunks - 1), 0) * 8;
            }
            __builtin_amdgcn_global_load_lds((glb_ptr)src, (lds_ptr)(ws[stage] + (wave * W_LOADS + i) * 1024), 16, 0, 0);
        }
    };
    f32x16 acc[NB];
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[b][r] = 0.0f;
    u32x4 xa[2][GK / 16];
    auto fetch_x = [&](int s, int buf) {
        if ((s + 1) * GK > h_len) {                       // block-uniform
#pragma unroll
            for (int u = 0; u < GK / 16; u++) {
                const bool inside = s * GK + u * 16 + (lane >> 5) * 8 < h_len;
                xa[buf][u] = inside ? *reinterpret_cast<const u32x4 *>(xp + s * GK + u * 16) : u32x4{0, 0, 0, 0};
            }
            return;
        }
#pragma unroll
        for (int u = 0; u < GK / 16; u++) xa[buf][u] = *reinterpret_cast<const u32x4 *>(xp + s * GK + u * 16);
    };
    auto multiply = [&](int stage, int buf) {
#pragma unroll
        for (int u = 0; u < GK / 16; u++) {
#pragma unroll
            for (int b = 0; b < NB; b++) {
                const u32x4 wf = *reinterpret_cast<const u32x4 *>(ws[stage] + w_off(b * 32 + (lane & 31), u * 2 + (lane >> 5)));
                // lane l then holds token l % 32 and experts b*32 + 8*(r/4) + 4*(l/32) + r%4
                acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, wf),
                                                                 __builtin_bit_cast(bf16x8, xa[buf][u]),
                                                                 acc[b], 0, 0, 0);
            }
        }
    };
    if (steps > 0) {
        issue_w(0, 0);
        fetch_x(0, 0);
    }
    for (int s = 0; s < steps; s += 2) {
        // stage 0 holds step s; fetch step s+1 into stage 1 while step s is multiplied
        __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): this wavefront's part of step s has landed
        __syncthreads();                      // everyone's has; stage 1 is free (step s-1 was read)
        if (s + 1 < steps) { issue_w(s + 1, 1); fetch_x(s + 1, 1); }
        multiply(0, 0);
        if (s + 1 >= steps) break;
        __builtin_amdgcn_s_waitcnt(0x0F70);
        __syncthreads();
        if (s + 2 < steps) { issue_w(s + 2, 0); fetch_x(s + 2, 0); }
        multiply(1, 1);
    }
    const int64_t t = t0 + (lane & 31);
    if (t < T) {
        float *out = partial + (static_cast<int64_t>(blockIdx.y) * T + t) * N;
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int n = b * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
                if (n < N) out[n] = acc[b][r];
            }
    }
}

// The same for few tokens: a wavefront per 16 tokens, 16 experts and slice, all of a slice's 256 columns under way at once, straight into
// the fragments of v_mfma_f32_16x16x32_bf16 (the same sums).  What bounds it is one miss after another, above four of them at hidden
// 2048 (two stages of 64 columns), here one.  us, with the
// routing, weights out of the caches: hidden 2048, 64 experts, 1 token 12.5 -> 10.1, 64 13.7 -> 10.3, 512 15.8 -> 10.9; hidden 7168, 64 experts,
// 512 tokens 25.0 -> 16.3, 8 experts 20.5 -> 10.6.  Every 16 tokens read the weight again: hidden 3000, 60 experts, 1000 tokens 17.4 -> 19.8, 4000 21.3 ->
// 33.7, hidden 4040, 20 experts, 2000 tokens 14.8 -> 15.5.  Hence the line.
// More than 64 experts have more to read again, and it stays the sooner one up to about 100 tokens; the projection with the launch that adds the
// slices, weights out of the caches: 256 experts of 7168, 1 token 13.7 -> 9.6, 64 14.8 -> 12.4, 96 15.7 -> 15.2, 128 16.2 -> 16.3, 200 17.0 ->
// 21.5; of 2048, 64 tokens 11.8 -> 10.4, 96 12.5 -> 11.8; 160 of 1624, 64 tokens 11.7 -> 10.0.
// CH: chunks of 32 columns under way, no more than a slice has (64 columns asked for as 256: 64 tokens of 2048, 256 experts 12.8, 512 tokens of
// 1024, 64 experts 11.8 for 9.4, 300 of 2048 13.8 for 10.7).
constexpr int64_t GATE_FEW_TOKENS = 512, GATE_FEW_TOKENS_WIDE = 64;
template <int CH>
__global__ __launch_bounds__(64) void gate_logits_few_kernel(const uint16_t *__restrict__ x, const uint16_t *__restrict__ w, int64_t T, int H, int N,
                                                             int h_per_split, float *__restrict__ partial) {
    const int lane = threadIdx.x, l16 = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * 16, split = blockIdx.y;
    const int64_t t = static_cast<int64_t>(blockIdx.z) * 16 + l16;
    const int begin = split * h_per_split, len = min(H - begin, h_per_split);
    // rows past the end (tokens, experts): the last one, results unused; columns past the end: the last chunk again, as zeros (of both: zero
    // times an infinite weight is NaN)
    const uint16_t *xr = x + min(t, T - 1) * H + begin, *wr = w + static_cast<int64_t>(min(n0 + l16, N - 1)) * H + begin;
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int c = 0; c < len; c += CH * 32) {
        u32x4 wf[CH], xf[CH];
#pragma unroll
        for (int i = 0; i < CH; i++) {
            const int k = c + i * 32 + g * 8, at = min(k, len - 8);
            wf[i] = *reinterpret_cast<const u32x4 *>(wr + at);
            xf[i] = *reinterpret_cast<const u32x4 *>(xr + at);
            if (k >= len) xf[i] = u32x4{0, 0, 0, 0};
        }
        if (c + CH * 32 > len) {   // block-uniform: the selects in every round took a one-token decode of 35 us 0.2 us
#pragma unroll
            for (int i = 0; i < CH; i++)
                if (c + i * 32 + g * 8 >= len) wf[i] = u32x4{0, 0, 0, 0};
        }
#pragma unroll
        for (int i = 0; i < CH; i++)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wf[i]), __builtin_bit_cast(bf16x8, xf[i]), acc, 0, 0, 0);
    }
    // element r of lane l: expert 4 * (l / 16) + r of token l % 16
    if (t < T) {
        float *out = partial + (static_cast<int64_t>(split) * T + t) * N + n0 + g * 4;
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (n0 + g * 4 + r < N) out[r] = acc[r];
    }
}

// The same for more than 64 experts, where a step's weights (32 KB for 256) are most of what a CU takes in: 128 tokens and all
// experts per block of eight wavefronts (64 x 64 of the logits each, NB = 4: 32 x 64), tokens and weights both by direct loads of
// whole 128-byte rows, two steps ahead, through a ring of three.  Rows, chunks and the last step as above, but that the
// tokens' chunks past the end are zeroed in LDS.
// us with the launch that adds the slices, weights out of the caches, 256 experts (before: four wavefronts of 32 tokens x 256
// experts, tokens straight from global memory in MFMA layout one step ahead, twice as many slices where those had to divide the
// steps): hidden 7168, 64 tokens 23.0 -> 14.5, 512 tokens 32.3 -> 18.0, 8192 tokens 87.2 -> 59.4; hidden 1624, 8176 tokens
// 120.2 -> 34.2.  128 experts, hidden 4096, 4096 tokens 33.6 -> 25.1.
template <int NB>
__global__ __launch_bounds__(512) void gate_logits_wide_kernel(const uint16_t *__restrict__ x, const uint16_t *__restrict__ w, int64_t T,
                                                               int H, int N, int h_per_split, float *__restrict__ partial) {
    constexpr int NP = NB * 32, SLOTS = 3, WN = NP / 64, TM = GT / 32 / (8 / WN), TN = 2;
    constexpr int UNITS = (GT + NP) / 8, LOADS = UNITS / 8;   // 1 KB direct loads of a step, tokens first, and a wavefront's
    constexpr int STEP = (GT + NP) * 128;
    __shared__ __attribute__((aligned(1024))) char lds[SLOTS * STEP];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int wm = wave / WN, wn = wave % WN;
    const int64_t t0 = static_cast<int64_t>(blockIdx.x) * GT;
    const int h_begin = blockIdx.y * h_per_split, h_len = min(H - h_begin, h_per_split), steps = (h_len + GK - 1) / GK;
    const uint32_t lds0 = lds_address(lds);
    const char *src[LOADS];
    int chunk[LOADS];
#pragma unroll
    for (int l = 0; l < LOADS; l++) {
        const int unit = wave * LOADS + l, row = unit * 8 + (lane >> 3);
        chunk[l] = (lane & 7) ^ ((row >> 1) & 7);
        // rows past the end (tokens, experts): valid memory, results unused
        src[l] = reinterpret_cast<const char *>(row < GT ? x + min(t0 + row, T - 1) * H + h_begin
                                                         : w + static_cast<int64_t>(min(row - GT, N - 1)) * H + h_begin);
    }
    auto issue = [&](int s, int slot) {
        const int last = ((h_len - s * GK) >> 3) - 1;         // chunks past the end: the last one again
#pragma unroll
        for (int l = 0; l < LOADS; l++)
            dma16_lane(src[l] + s * (GK * 2) + min(chunk[l], last) * 16, lds0 + slot * STEP + (wave * LOADS + l) * 1024);
    };
    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;
    issue(0, 0);
    if (steps > 1) issue(1, 1);
    int slot = 0, free_slot = 2;
    for (int s = 0; s < steps; s++) {
        // This wavefront's part of step s has landed; behind the barrier everyone's has, and everyone has read step s - 1,
        // whose slot takes step s + 2.
        if (s + 1 < steps) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if ((s + 1) * GK > h_len) {
#pragma unroll
            for (int l = 0; l < LOADS; l++)
                if (wave * LOADS + l < GT / 8 && s * GK + chunk[l] * 8 >= h_len)
                    *reinterpret_cast<u32x4 *>(lds + slot * STEP + (wave * LOADS + l) * 1024 + lane * 16) = u32x4{0, 0, 0, 0};
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (s + 2 < steps) issue(s + 2, free_slot);
        const char *xs = lds + slot * STEP, *ws = xs + GT * 128;
#pragma unroll
        for (int u = 0; u < GK / 16; u++) {
            bf16x8 fx[TM], fw[TN];
#pragma unroll
            for (int i = 0; i < TM; i++)
                fx[i] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(xs + w_off((wm * TM + i) * 32 + (lane & 31), u * 2 + (lane >> 5))));
#pragma unroll
            for (int j = 0; j < TN; j++)
                fw[j] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(ws + w_off((wn * TN + j) * 32 + (lane & 31), u * 2 + (lane >> 5))));
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fx[i], fw[j], acc[i][j], 0, 0, 0);
        }
        free_slot = slot;
        slot = slot == SLOTS - 1 ? 0 : slot + 1;
    }
    // accumulator element r of lane l: token 8*(r/4) + 4*(l/32) + r%4, expert l%32
    float *out = partial + static_cast<int64_t>(blockIdx.y) * T * N;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int64_t t = t0 + (wm * TM + i) * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const int n = (wn * TN + j) * 32 + (lane & 31);
                if (t < T && n < N) out[t * N + n] = acc[i][j][r];
            }
        }
}

// logits = sum over the slices of H, in slice order
__global__ __launch_bounds__(256) void gate_logits_reduce_kernel(const float *__restrict__ partial,
                                                                 int splits, int64_t tn,
                                                                 float *__restrict__ logits) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= tn) return;
    float s = 0.0f;
    for (int k0 = 0; k0 < splits; k0 += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = (k0 + u < splits) ? partial[(k0 + u) * tn + i] : 0.0f;
#pragma unroll
        for (int u = 0; u < 8; u++) s += v[u];
    }
    logits[i] = s;
}

inline bool gate_split_shape_ok(int64_t T, int H, int N) {
    return T >= 0 && T <= 0x7fffffffLL && N >= 1 && N <= 256 && H >= 8 && H % 8 == 0;
}

// Slices of H: a block per CU, and no more (the fp32 partials cost 8 B per logit and slice).  At most 32: 64 tokens, hidden 7168,
// 256 experts 22 us with 16 slices, 19 with 28.  A slice is a whole number of 64-wide steps, the last one may be shorter and
// its last step partial.
// Up to 64 experts several blocks share a CU.  From 33 blocks of tokens on (below, more slices cost what they give) the
// count with the least time by this account is taken: a step of the busiest CU's k blocks takes 730 ns with one of them, 900 k -
// 700 with more, a slice's partials 3 ps per logit (fitted to 270 shapes of 8 to 61 experts, hidden 336 to 6440, 1 to 8 slices
// each).  us, a block per CU -> now: 8 experts, hidden 4104, 11000 tokens 28.8 -> 19.4, 18000 50.5 -> 28.5; 40 experts,
// hidden 4928, 6677 tokens 24.4 -> 21.5; 61 experts, hidden 6440, 18000 tokens 89.7 -> 59.1, 22000 133 -> 102; hidden 336, 22000
// tokens 15.5, one slice in both; at worst 8 experts, hidden 336, 5000 tokens 6.5 -> 7.1.
inline int gate_split_count(int64_t T, int H, int N) {
    const int64_t token_blocks = std::max<int64_t>((T + GT - 1) / GT, 1);
    const int steps = (H + GK - 1) / GK;
    auto steps_each = [&](int slices) { return (steps + slices - 1) / slices; };
    int want = static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(32, 256 / token_blocks)));
    if (N <= 64 && token_blocks > 32) {
        int64_t least = INT64_MAX;
        for (int s = 1; s <= std::min(8, steps); s++) {
            const int64_t k = (token_blocks * s + 255) / 256;
            const int64_t picoseconds = steps_each(s) * 1000 * (k == 1 ? 730 : 900 * k - 700) + s * 3 * T * N;
            if (picoseconds < least) { least = picoseconds; want = s; }
        }
    }
    const int each = steps_each(want);
    return (steps + each - 1) / each;
}

}  // namespace

// Behind a routing kernel that adds the slices itself: eight of them where the steps divide (the order of
// the sums is then that of om_router_gate_softmax_topk, bit for bit), else as above.
int om_gate_route_splits(int64_t T, int H, int N) {
    return N <= 64 && H % 512 == 0 ? 8 : gate_split_count(T, H, N);
}

void om_launch_gate_partials(const void *x, const void *gate_weight, int64_t T, int H, int N, int splits, float *ws,
                             hipStream_t st) {
    const dim3 grid(static_cast<unsigned>((T + GT - 1) / GT), splits);
    const uint16_t *xp = static_cast<const uint16_t *>(x), *wp = static_cast<const uint16_t *>(gate_weight);
    const int hps = ((H + GK - 1) / GK + splits - 1) / splits * GK;
    if (T <= (N <= 64 ? GATE_FEW_TOKENS : GATE_FEW_TOKENS_WIDE)) {
        const dim3 tiles((N + 15) / 16, splits, static_cast<unsigned>((T + 15) / 16));
        if (hps > 128) gate_logits_few_kernel<8><<<tiles, dim3(64), 0, st>>>(xp, wp, T, H, N, hps, ws);
        else if (hps > 64) gate_logits_few_kernel<4><<<tiles, dim3(64), 0, st>>>(xp, wp, T, H, N, hps, ws);
        else gate_logits_few_kernel<2><<<tiles, dim3(64), 0, st>>>(xp, wp, T, H, N, hps, ws);
    } else if (N <= 64) gate_logits_split_kernel<2><<<grid, dim3(256), 0, st>>>(xp, wp, T, H, N, hps, ws);
    else if (N <= 128) gate_logits_wide_kernel<4><<<grid, dim3(512), 0, st>>>(xp, wp, T, H, N, hps, ws);
    else gate_logits_wide_kernel<8><<<grid, dim3(512), 0, st>>>(xp, wp, T, H, N, hps, ws);
}

extern "C" int64_t om_router_gate_route_workspace_bytes(int64_t T, int H, int N) {
    if (!gate_split_shape_ok(T, H, N)) return OM_ERR_SHAPE;
    return static_cast<int64_t>(om_gate_route_splits(T, H, N)) * T * N * 4;
}

extern "C" int64_t om_router_gate_logits_split_workspace_bytes(int64_t T, int H, int N) {
    if (!gate_split_shape_ok(T, H, N)) return OM_ERR_SHAPE;
    return static_cast<int64_t>(gate_split_count(T, H, N)) * T * N * 4;
}

extern "C" int om_router_gate_logits_split(const void *x, const void *gate_weight, int64_t T, int H, int N,
                                           float *logits_out, void *workspace, int64_t workspace_bytes,
                                           void *stream) {
    if (!gate_split_shape_ok(T, H, N)) return OM_ERR_SHAPE;
    if (T == 0) return OM_OK;
    if (!x || !gate_weight || !logits_out || !workspace) return OM_ERR_NULL;
    if (!om_aligned16(x) || !om_aligned16(gate_weight) || !om_aligned16(workspace)) return OM_ERR_ALIGN;
    const int splits = gate_split_count(T, H, N);
    const int64_t tn = T * N;
    if (workspace_bytes < splits * tn * 4) return OM_ERR_WORKSPACE;
    hipStream_t st = om_stream(stream);
    float *ws = static_cast<float *>(workspace);
    om_launch_gate_partials(x, gate_weight, T, H, N, splits, ws, st);
    gate_logits_reduce_kernel<<<dim3(static_cast<unsigned>((tn + 255) / 256)), dim3(256), 0, st>>>(ws, splits, tn, logits_out);
    return om_launch_status();
}

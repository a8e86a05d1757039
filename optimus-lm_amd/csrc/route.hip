// Routers: one wavefront per token.
//  * softmax -> top-K (-> renormalise) of the OLMoE block, forward and backward;
//  * sigmoid -> bias-corrected group-limited top-K of the DeepSeek-V3 block, forward and backward.
// Selection order is total: (score descending, expert index ascending), so the result does not
// depend on lane scheduling.  Scores live in registers, expert i = lane + 64*j.
#include "sort_block.h"

#include <algorithm>
#include <type_traits>

namespace {

#pragma clang fp contract(off)

constexpr int TOKENS_PER_BLOCK = 4;

template <typename T> __device__ __forceinline__ float load_logit(const T *p);
template <> __device__ __forceinline__ float load_logit<float>(const float *p) { return *p; }
template <> __device__ __forceinline__ float load_logit<uint16_t>(const uint16_t *p) { return bf16_bits_to_f32(*p); }

// (value, index) arg-max across the wavefront by an xor butterfly of lane permutes; ties go to
// the lower index.  Twelve dependent permutes: the slow path of wave_argmax below.
__device__ __forceinline__ void wave_argmax_butterfly(float &v, int &i) {
    for (int o = 32; o > 0; o >>= 1) {
        const float ov = __shfl_xor(v, o, 64);
        const int oi = __shfl_xor(i, o, 64);
        if (ov > v || (ov == v && oi < i)) { v = ov; i = oi; }
    }
}

// Maximum over the wavefront with data-parallel-primitive moves (no LDS traffic): within each row
// of 16 lanes by quad permutes and mirrors, then row 0 -> 1 and 2 -> 3, then rows 0-1 -> 2-3; lane
// 63 ends with the maximum and hands it to everyone through a scalar register.  A maximum does not
// depend on the order of the comparisons, so this is exact.
__device__ __forceinline__ float wave_max_dpp(float v) {
    int x = __float_as_int(v);
#define OM_DPP_MAX(ctrl, row_mask)                                                                   \
    x = __float_as_int(fmaxf(__int_as_float(x), __int_as_float(__builtin_amdgcn_update_dpp(         \
            x, x, ctrl, row_mask, 0xf, false))))
    OM_DPP_MAX(0xB1, 0xf);    // quad_perm [1,0,3,2]
    OM_DPP_MAX(0x4E, 0xf);    // quad_perm [2,3,0,1]
    OM_DPP_MAX(0x141, 0xf);   // row_half_mirror
    OM_DPP_MAX(0x140, 0xf);   // row_mirror: every lane of a row holds the row's maximum
    OM_DPP_MAX(0x142, 0xa);   // row_bcast15 into rows 1 and 3
    OM_DPP_MAX(0x143, 0xc);   // row_bcast31 into rows 2 and 3
#undef OM_DPP_MAX
    return __int_as_float(__builtin_amdgcn_readlane(x, 63));
}

// (value, index) arg-max across the wavefront; ties go to the lower index.  Fast path: the maximum
// by wave_max_dpp, a ballot of the lanes that hold it, and when exactly one lane does (no tie, no
// NaN) its index through a scalar lane read.  Everything else takes the butterfly, so the result
// is the butterfly's in every case.
__device__ __forceinline__ void wave_argmax(float &v, int &i) {
    const float m = wave_max_dpp(v);
    const unsigned long long vote = __ballot(v == m);
    if (__popcll(vote) == 1) {
        const int src = __ffsll(static_cast<long long>(vote)) - 1;
        i = __builtin_amdgcn_readlane(i, src);
        v = m;
    } else {
        wave_argmax_butterfly(v, i);
    }
}

// value of `x[e / 64]` held by lane e % 64, for a per-lane e (e < 0: undefined, caller masks)
template <int PER>
__device__ __forceinline__ float fetch_expert_value(const float (&x)[PER], int e) {
    float out = 0.0f;
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const float v = __shfl(x[j], e & 63, 64);
        if ((e >> 6) == j) out = v;
    }
    return out;
}

// The logits of token t of a gate projection that was split over H: the slices' partial sums
// [splits][Tn][N] added in slice order; lanes past N get -inf.
template <int PER>
__device__ __forceinline__ void partial_logits(const float *partial, int splits, int64_t Tn, int64_t t, int N, int lane,
                                               float (&x)[PER]) {
    // eight slices of all the lane's experts in flight, added in slice order; past the end the last valid one again
    float s[PER];
#pragma unroll
    for (int j = 0; j < PER; j++) s[j] = 0.0f;
    for (int k0 = 0; k0 < splits; k0 += 8) {
        float v[8][PER];
#pragma unroll
        for (int u = 0; u < 8; u++)
#pragma unroll
            for (int j = 0; j < PER; j++)
                v[u][j] = partial[(min(k0 + u, splits - 1) * Tn + t) * N + min(lane + 64 * j, N - 1)];
#pragma unroll
        for (int u = 0; u < 8; u++)
#pragma unroll
            for (int j = 0; j < PER; j++) s[j] += k0 + u < splits ? v[u][j] : 0.0f;
    }
#pragma unroll
    for (int j = 0; j < PER; j++) x[j] = lane + 64 * j < N ? s[j] : -INFINITY;
}

// logits (lanes past N: -inf) -> softmax probabilities, in place
template <int PER> __device__ __forceinline__ void softmax_in_place(int N, int lane, float (&p)[PER]) {
    float mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < PER; j++) mx = fmaxf(mx, p[j]);
    mx = wave_max_dpp(mx);
    float sum = 0.0f;
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int i = lane + 64 * j;
        p[j] = (i < N) ? expf(p[j] - mx) : 0.0f;
        sum += p[j];
    }
    sum = wave_sum(sum);
#pragma unroll
    for (int j = 0; j < PER; j++) p[j] = p[j] / sum;
}

// softmax probabilities of this token's row into p[PER]; returns nothing else.
template <int PER, typename T>
__device__ __forceinline__ void row_softmax(const T *row, int N, int lane, float (&p)[PER]) {
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int i = lane + 64 * j;
        p[j] = (i < N) ? load_logit<T>(row + i) : -INFINITY;
    }
    softmax_in_place<PER>(N, lane, p);
}

// The lowest expert that is not among the first r selections, of which lane q holds the q-th: what a group-limited router selects where no
// score is left that compares (NaN, or biases of -inf).
__device__ __forceinline__ int lowest_free(int e, int r, int lane) {
    int i = 0;
    while (__ballot(lane < r && e == i) != 0) i++;
    return i;
}

// K rounds of wave arg-max over s[PER] (entries with index >= N must be < every real score).
// Lane r keeps the r-th winner in (my_v, my_i).  Scores that are NaN or -inf never win; where no other is left the index is
// 0x7fffffff, or with FREE the lowest that was not selected.
template <int PER, bool FREE = false>
__device__ __forceinline__ void select_topk(float (&s)[PER], int N, int K, int lane, float &my_v,
                                            int &my_i) {
    my_v = 0.0f;
    my_i = 0;
    for (int r = 0; r < K; r++) {
        float bv = -INFINITY;
        int bi = 0x7fffffff;
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const int i = lane + 64 * j;
            if (i < N && (s[j] > bv)) { bv = s[j]; bi = i; }  // ascending i: first max wins
        }
        wave_argmax(bv, bi);
        if (FREE && bi == 0x7fffffff) bi = lowest_free(my_i, r, lane);
        if (lane == r) { my_v = bv; my_i = bi; }
#pragma unroll
        for (int j = 0; j < PER; j++)
            if (lane + 64 * j == bi) s[j] = -INFINITY;  // taken
    }
}

template <int PER, typename T, typename TW>
__global__ __launch_bounds__(256) void softmax_topk_kernel(const T *__restrict__ logits, int64_t Tn,
                                                           int N, int K, int renorm,
                                                           TW *__restrict__ weights_out,
                                                           int64_t *__restrict__ experts_out) {
    const int lane = threadIdx.x & 63;
    const int64_t t = static_cast<int64_t>(blockIdx.x) * TOKENS_PER_BLOCK + (threadIdx.x >> 6);
    if (t >= Tn) return;
    float p[PER];
    row_softmax<PER, T>(logits + t * N, N, lane, p);
    float w; int e;
    select_topk<PER>(p, N, K, lane, w, e);
    if (renorm) {
        const float s = wave_sum(lane < K ? w : 0.0f);
        w = w / s;
    }
    if (lane < K) {
        Elem<TW>::store(weights_out + t * K + lane, w);
        experts_out[t * K + lane] = e;
    }
}

// The same behind a gate projection that was split over H: adds the slices, writes the logits (rounded to
// TL first, which is what the softmax then sees) and routes.  One launch instead of a reduction, a
// conversion and a routing launch, each of which is a few microseconds of latency for a small batch.
template <int PER, typename TL, typename TW>
__global__ __launch_bounds__(256) void partial_softmax_topk_kernel(const float *__restrict__ partial, int splits, int64_t Tn,
                                                                   int N, int K, int renorm, TL *__restrict__ logits_out,
                                                                   TW *__restrict__ weights_out,
                                                                   int64_t *__restrict__ experts_out) {
    const int lane = threadIdx.x & 63;
    const int64_t t = static_cast<int64_t>(blockIdx.x) * TOKENS_PER_BLOCK + (threadIdx.x >> 6);
    if (t >= Tn) return;
    float p[PER];
    partial_logits<PER>(partial, splits, Tn, t, N, lane, p);
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int i = lane + 64 * j;
        if (i >= N) continue;
        Elem<TL>::store(logits_out + t * N + i, p[j]);
        if (sizeof(TL) == 2) p[j] = bf16_bits_to_f32(f32_to_bf16_bits(p[j]));
    }
    softmax_in_place<PER>(N, lane, p);
    float w; int e;
    select_topk<PER>(p, N, K, lane, w, e);
    if (renorm) {
        const float s = wave_sum(lane < K ? w : 0.0f);
        w = w / s;
    }
    if (lane < K) {
        Elem<TW>::store(weights_out + t * K + lane, w);
        experts_out[t * K + lane] = e;
    }
}

// The gate projection of a float32 module, logits[t,n] = sum_h x[t,h] W[n,h]: one wavefront per token, lanes over h, the 64 partial sums
// added by a butterfly, eight experts at a time (one at a time, each waited for its loads and its butterfly).  ROUTE (up to 64
// experts): the softmax router in the same launch, as softmax_topk_kernel.  2048 tokens of 256, 8 experts: 8.2 + 3.4 -> 6.4 us.
template <bool ROUTE, typename TW>
__global__ __launch_bounds__(256) void gate_f32_kernel(const float *__restrict__ x, const float *__restrict__ w, int64_t Tn, int H, int N,
                                                       int K, int renorm, float *__restrict__ logits, TW *__restrict__ weights_out,
                                                       int64_t *__restrict__ experts_out) {
#pragma clang fp contract(fast)
    const int lane = threadIdx.x & 63;
    const int64_t t = static_cast<int64_t>(blockIdx.x) * TOKENS_PER_BLOCK + (threadIdx.x >> 6);
    if (t >= Tn) return;
    const float *xr = x + t * H;
    float p[1] = {-INFINITY};
    for (int n0 = 0; n0 < N; n0 += 8) {
        float s[8] = {};
        for (int h = lane; h < H; h += 64) {
            const float xv = xr[h];
#pragma unroll
            for (int j = 0; j < 8; j++) s[j] += xv * w[static_cast<int64_t>(min(n0 + j, N - 1)) * H + h];
        }
#pragma unroll
        for (int j = 0; j < 8; j++) {
            s[j] = wave_sum(s[j]);
            if (n0 + j >= N) continue;
            if (ROUTE && lane == n0 + j) p[0] = s[j];
            if (!ROUTE && lane == 0) logits[t * N + n0 + j] = s[j];
        }
    }
    if (!ROUTE) return;
    if (lane < N) logits[t * N + lane] = p[0];
    softmax_in_place<1>(N, lane, p);
    float wt; int e;
    select_topk<1>(p, N, K, lane, wt, e);
    if (renorm) wt = wt / wave_sum(lane < K ? wt : 0.0f);
    if (lane < K) {
        Elem<TW>::store(weights_out + t * K + lane, wt);
        experts_out[t * K + lane] = e;
    }
}

// dlogits_i = p_i * (dp_i - sum_j dp_j p_j), dp = scatter of dw over the selected experts, and
// with renormalisation dw_k = (dw'_k - sum_j dw'_j w_j / S) / S, S = sum_k w_k, w_k = p[e_k].
// TO: T, or float for the gate's gradients (om_launch_softmax_bwd, which says what the last three arguments are).
template <int PER, typename T, typename TW, typename TO>
__global__ __launch_bounds__(256) void softmax_topk_bwd_kernel(const T *__restrict__ logits,
                                                               const int64_t *__restrict__ experts,
                                                               const TW *__restrict__ dweights,
                                                               int64_t Tn, int N, int K, int renorm,
                                                               TO *__restrict__ dlogits, const T *__restrict__ more, unsigned *zero, int n_zero) {
    if (n_zero > 0 && blockIdx.x == 0)
        for (int i = threadIdx.x; i < n_zero; i += 256) zero[i] = 0;
    const int lane = threadIdx.x & 63;
    const int64_t t = static_cast<int64_t>(blockIdx.x) * TOKENS_PER_BLOCK + (threadIdx.x >> 6);
    if (t >= Tn) return;
    float p[PER];
    row_softmax<PER, T>(logits + t * N, N, lane, p);
    // lane k < K: its expert, the probability there and the incoming gradient
    const int e = (lane < K) ? static_cast<int>(experts[t * K + lane]) : -1;
    float dwk = (lane < K) ? Elem<TW>::load(dweights + t * K + lane) : 0.0f;
    float wk = fetch_expert_value<PER>(p, e);   // lane k < K: the probability of its expert
    if (lane >= K) wk = 0.0f;
    if (renorm) {
        const float S = wave_sum(wk);
        const float dot = wave_sum(dwk * wk);
        dwk = (dwk - dot / S) / S;
    }
    const float inner = wave_sum(dwk * wk);  // sum_j dp_j p_j
    float dp[PER];
#pragma unroll
    for (int j = 0; j < PER; j++) dp[j] = 0.0f;
    for (int k = 0; k < K; k++) {
        const int ek = __shfl(e, k, 64);
        const float dk = __shfl(dwk, k, 64);
#pragma unroll
        for (int j = 0; j < PER; j++)
            if (lane + 64 * j == ek) dp[j] = dk;
    }
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int i = lane + 64 * j;
        if (i >= N) continue;
        float d = p[j] * (dp[j] - inner);
        if (sizeof(T) == 2) d = bf16_bits_to_f32(f32_to_bf16_bits(d));
        if (more) {
            d += load_logit<T>(more + t * N + i);
            if (sizeof(T) == 2) d = bf16_bits_to_f32(f32_to_bf16_bits(d));
        }
        Elem<TO>::store(dlogits + t * N + i, d);
    }
}

// DeepSeek-V3 group-limited routing.  LDS holds the choice scores of the 4 tokens of the block
// so a lane can scan "its" group; everything else stays in registers.
// PARTIAL: the logits are the sum of a split gate projection's slices and are written out.
template <int PER, bool PARTIAL, typename TB>
__global__ __launch_bounds__(256) void sigmoid_group_topk_kernel(
    const float *__restrict__ logits, int splits, float *__restrict__ logits_out, const TB *__restrict__ bias, int64_t Tn, int N, int n_group,
    int topk_group, int K, int renorm, float scale, int64_t *__restrict__ experts_out,
    float *__restrict__ weights_out) {
    __shared__ float choice_lds[TOKENS_PER_BLOCK][PER * 64];
    const int lane = threadIdx.x & 63;
    const int wv = threadIdx.x >> 6;
    const int64_t t = static_cast<int64_t>(blockIdx.x) * TOKENS_PER_BLOCK + wv;
    if (t >= Tn) return;  // whole wavefront leaves together; no block-wide barrier below
    float score[PER], choice[PER], row[PER];
    if (PARTIAL) partial_logits<PER>(logits, splits, Tn, t, N, lane, row);
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int i = lane + 64 * j;
        if (i < N) {
            const float x = PARTIAL ? row[j] : logits[t * N + i];
            if (PARTIAL) logits_out[t * N + i] = x;
            score[j] = 1.0f / (1.0f + expf(-x));
            choice[j] = score[j] + Elem<TB>::load(bias + i);
            choice_lds[wv][i] = choice[j];
        } else {
            score[j] = 0.0f;
            choice[j] = -INFINITY;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // lane g < n_group: sum of the two largest choice values of group g
    const int gs = N / n_group;
    float gscore = -INFINITY;
    if (lane < n_group) {
        float a = -INFINITY, b = -INFINITY;
        for (int i = 0; i < gs; i++) {
            const float v = choice_lds[wv][lane * gs + i];
            if (v > a) { b = a; a = v; } else if (v > b) { b = v; }
        }
        gscore = (gs >= 2) ? (a + b) : a;
        if (gscore != gscore) gscore = -INFINITY;   // (+inf and nothing beside it)
    }
    // keep the topk_group best groups (score desc, group index asc)
    unsigned long long keep = 0ull;
    for (int r = 0; r < topk_group; r++) {
        float bv = gscore; int bi = (lane < n_group) ? lane : 0x7fffffff;
        wave_argmax(bv, bi);
        keep |= (1ull << bi);
        if (lane == bi) gscore = -INFINITY;
    }
    // masked_fill(~mask, 0.0): dropped groups compete with the value 0.0
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int i = lane + 64 * j;
        if (i < N && !((keep >> (i / gs)) & 1ull)) choice[j] = 0.0f;
    }
    float cv; int e;
    select_topk<PER, true>(choice, N, K, lane, cv, e);
    // weight = sigmoid score (no bias) at the selected expert
    float w = fetch_expert_value<PER>(score, e);
    if (lane >= K) w = 0.0f;
    if (renorm) {
        const float S = wave_sum(lane < K ? w : 0.0f) + 1e-20f;
        w = w / S;
    }
    w = w * scale;
    if (lane < K) {
        experts_out[t * K + lane] = e;
        weights_out[t * K + lane] = w;
    }
}

// The same behind a split gate projection, up to 256 experts in groups of a power of two, four at least: a lane holds four neighbouring
// experts, so a slice's partial sums are one load a lane, of sixteen slices under way at once, and a group's two best meet by exchanges
// between its lanes (above, one lane scans a group's scores in LDS).  A token waits for its loads and for chains of a few
// instructions; with few tokens a wavefront per block.  Same sums, same order of selection.  us, 256 experts, 64 tokens of 28
// slices 13.6 -> 8.0, 8192 of 4 slices 22.4 -> 17.2 (and 5 less for a bias in bf16, which was widened by a launch of its own); 0.2 of it
// for scores that are not finite.
constexpr int QUADS = 4;
template <typename TB>
__global__ __launch_bounds__(256) void sigmoid_group_quads_kernel(const float *__restrict__ partial, int splits, float *__restrict__ logits_out,
                                                                  const TB *__restrict__ bias, int64_t Tn, int N, int n_group, int topk_group,
                                                                  int K, int renorm, float scale, int64_t *__restrict__ experts_out,
                                                                  float *__restrict__ weights_out) {
    const int lane = threadIdx.x & 63;
    const int64_t t = static_cast<int64_t>(blockIdx.x) * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (t >= Tn) return;
    const int i0 = lane * QUADS, from = min(i0, N - QUADS);
    const bool inside = i0 < N;
    float b[QUADS];
#pragma unroll
    for (int j = 0; j < QUADS; j++) b[j] = Elem<TB>::load(bias + from + j);
    f32x4 x = {0.0f, 0.0f, 0.0f, 0.0f};
    const float *row = partial + t * N + from;
    for (int k0 = 0; k0 < splits; k0 += 16) {
        f32x4 v[16];
#pragma unroll
        for (int u = 0; u < 16; u++) v[u] = *reinterpret_cast<const f32x4 *>(row + min(k0 + u, splits - 1) * Tn * N);
#pragma unroll
        for (int u = 0; u < 16; u++)
#pragma unroll
            for (int j = 0; j < QUADS; j++) x[j] += k0 + u < splits ? v[u][j] : 0.0f;
    }
    if (inside) *reinterpret_cast<f32x4 *>(logits_out + t * N + i0) = x;
    float score[QUADS], choice[QUADS];
#pragma unroll
    for (int j = 0; j < QUADS; j++) {
        score[j] = inside ? 1.0f / (1.0f + expf(-x[j])) : 0.0f;
        choice[j] = inside ? score[j] + b[j] : -INFINITY;
    }
    // the two largest of the lane's, then of its group's lanes; NaN is none of them, as in the scan
    const int lanes = N / n_group / QUADS;
    float best = -INFINITY, next = -INFINITY;
#pragma unroll
    for (int j = 0; j < QUADS; j++) {
        const float v = choice[j] == choice[j] ? choice[j] : -INFINITY;
        next = fmaxf(next, fminf(best, v));
        best = fmaxf(best, v);
    }
    for (int o = 1; o < lanes; o <<= 1) {
        const float other = __shfl_xor(best, o, 64), other_next = __shfl_xor(next, o, 64);
        next = fmaxf(fmaxf(next, other_next), fminf(best, other));
        best = fmaxf(best, other);
    }
    // kept: the groups that fewer than topk_group others precede (score descending, group ascending).  A group with less than two
    // scores that compare has -inf and is not kept, but where such groups are reached at all the first group is.
    const float sum = best + next, mine = sum == sum ? sum : -INFINITY;
    const int group = i0 / (lanes * QUADS);
    int before = 0, above = 0;
    for (int q = 0; q < n_group; q++) {
        const float other = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(mine), q * lanes));
        before += other > mine || (other == mine && q < group) ? 1 : 0;
        above += other > -INFINITY ? 1 : 0;
    }
    const bool kept = mine > -INFINITY ? before < topk_group : group == 0 && above < topk_group;
    // masked_fill(~mask, 0.0): dropped groups compete with the value 0.0
    if (inside && !kept) {
#pragma unroll
        for (int j = 0; j < QUADS; j++) choice[j] = 0.0f;
    }
    float w = 0.0f;
    int e = 0;
    for (int r = 0; r < K; r++) {
        float bv = -INFINITY;
        int bi = 0x7fffffff;
#pragma unroll
        for (int j = 0; j < QUADS; j++)
            if (inside && choice[j] > bv) { bv = choice[j]; bi = i0 + j; }   // ascending experts: the first maximum wins
        wave_argmax(bv, bi);
        if (bi == 0x7fffffff) bi = lowest_free(e, r, lane);
        if (lane == r) e = bi;
#pragma unroll
        for (int j = 0; j < QUADS; j++)
            if (i0 + j == bi) choice[j] = -INFINITY;                         // taken
    }
    // weight = sigmoid score (no bias) at the selected expert
#pragma unroll
    for (int j = 0; j < QUADS; j++) {
        const float v = __shfl(score[j], (e >> 2) & 63, 64);
        if ((e & 3) == j) w = v;
    }
    if (lane >= K) w = 0.0f;
    if (renorm) w = w / (wave_sum(w) + 1e-20f);
    w = w * scale;
    if (lane < K) {
        experts_out[t * K + lane] = e;
        weights_out[t * K + lane] = w;
    }
}

// w'_k = scale * s_k / (S + 1e-20) (or scale * s_k); ds_k -> dlogit = ds * s * (1 - s).
template <int PER>
__global__ __launch_bounds__(256) void sigmoid_topk_bwd_kernel(const float *__restrict__ logits,
                                                               const int64_t *__restrict__ experts,
                                                               const float *__restrict__ dweights,
                                                               int64_t Tn, int N, int K, int renorm,
                                                               float scale, float *__restrict__ dlogits) {
    const int lane = threadIdx.x & 63;
    const int64_t t = static_cast<int64_t>(blockIdx.x) * TOKENS_PER_BLOCK + (threadIdx.x >> 6);
    if (t >= Tn) return;
    const int64_t selected = (lane < K) ? experts[t * K + lane] : -1;
    const int e = selected >= 0 && selected < N ? static_cast<int>(selected) : -1;   // (a number that is no expert's: no weight, no gradient)
    float sk = 0.0f;
    if (e >= 0) sk = 1.0f / (1.0f + expf(-logits[t * N + e]));
    float d = (lane < K) ? dweights[t * K + lane] * scale : 0.0f;  // through "* scale"
    if (renorm) {
        const float S = wave_sum(sk) + 1e-20f;
        const float dot = wave_sum(d * sk);
        d = (d - dot / S) / S;
    }
    const float dl = d * (sk * (1.0f - sk));
    float out[PER];
#pragma unroll
    for (int j = 0; j < PER; j++) out[j] = 0.0f;
    for (int k = 0; k < K; k++) {
        const int ek = __shfl(e, k, 64);
        const float dk = __shfl(dl, k, 64);
#pragma unroll
        for (int j = 0; j < PER; j++)
            if (lane + 64 * j == ek) out[j] += dk;
    }
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int i = lane + 64 * j;
        if (i < N) dlogits[t * N + i] = out[j];
    }
}

// Router gate fused with the routing: logits = x @ Wg^T for 32 tokens per block on the matrix
// cores (bf16 operands whose products are exact in fp32, fp32 accumulation: the value of
// x.float() @ Wg.float().T up to the order of the sum), the contraction split over the block's
// wavefronts and reduced through LDS in a fixed order, then softmax / top-K of those tokens
// straight from LDS.  x is read from HBM exactly once (the pass is HBM-bound on it); Wg stays in L2.
// Operand fragments come straight from global memory in MFMA layout (lane = row, 8 consecutive
// h): the four loads that share a 128-byte line are issued together.
template <int NB, int WAVES, int UNR, int PER, typename TW, bool ROUTE>
__global__ __launch_bounds__(WAVES * 64) void gate_route_kernel(
    const uint16_t *__restrict__ x, const uint16_t *__restrict__ wg, int64_t Tn, int H, int N, int K,
    int renorm, float *__restrict__ logits_out, TW *__restrict__ weights_out,
    int64_t *__restrict__ experts_out) {
    constexpr int NP = NB * 32;  // expert count rounded up to the MFMA block
    __shared__ float part[WAVES][32][NP];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t t0 = static_cast<int64_t>(blockIdx.x) * 32;
    const int hw = H / WAVES;
    const int r32 = lane & 31, kofs = (lane >> 5) * 8;
    int64_t ta = t0 + r32;
    if (ta >= Tn) ta = Tn - 1;  // rows past the end: valid memory, result unused
    const uint16_t *ap = x + ta * H + wave * hw + kofs;
    const uint16_t *bp[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) {
        int e = j * 32 + r32;
        if (e >= N) e = N - 1;
        bp[j] = wg + static_cast<int64_t>(e) * H + wave * hw + kofs;
    }
    f32x16 acc[NB];
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[j][r] = 0.0f;
    for (int h = 0; h < hw; h += 16 * UNR) {
        u32x4 a[UNR], b[NB][UNR];
#pragma unroll
        for (int u = 0; u < UNR; u++) {
            a[u] = *reinterpret_cast<const u32x4 *>(ap + h + u * 16);
#pragma unroll
            for (int j = 0; j < NB; j++) b[j][u] = *reinterpret_cast<const u32x4 *>(bp[j] + h + u * 16);
        }
#pragma unroll
        for (int u = 0; u < UNR; u++)
#pragma unroll
            for (int j = 0; j < NB; j++)
                acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[u]),
                                                                 __builtin_bit_cast(bf16x8, b[j][u]),
                                                                 acc[j], 0, 0, 0);
    }
    // accumulator element r of lane l: token (r/4)*8 + (l/32)*4 + r%4, expert j*32 + l%32
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
        for (int r = 0; r < 16; r++)
            part[wave][(r >> 2) * 8 + (lane >> 5) * 4 + (r & 3)][j * 32 + r32] = acc[j][r];
    __syncthreads();
    for (int idx = threadIdx.x; idx < 32 * NP; idx += WAVES * 64) {
        const int row = idx / NP, col = idx % NP;
        float sum = part[0][row][col];
#pragma unroll
        for (int w = 1; w < WAVES; w++) sum += part[w][row][col];
        part[0][row][col] = sum;
        if (logits_out && t0 + row < Tn && col < N) logits_out[(t0 + row) * N + col] = sum;
    }
    if (!ROUTE) return;
    __syncthreads();
    for (int tk = wave; tk < 32; tk += WAVES) {
        const int64_t t = t0 + tk;
        if (t >= Tn) break;
        float p[PER];
        row_softmax<PER, float>(&part[0][tk][0], N, lane, p);
        float w; int e;
        select_topk<PER>(p, N, K, lane, w, e);
        if (renorm) {
            const float sk = wave_sum(lane < K ? w : 0.0f);
            w = w / sk;
        }
        if (lane < K) {
            Elem<TW>::store(weights_out + t * K + lane, w);
            experts_out[t * K + lane] = e;
        }
    }
}

// Within each row of 16 lanes.  The sum adds lanes 8 apart first, then 4, 2 and 1, as the last steps of wave_sum do.
#define OM_ROW_STEP(x, ctrl) __builtin_amdgcn_update_dpp(0, x, ctrl, 0xf, 0xf, true)
__device__ __forceinline__ float row_max(float v) {
    v = fmaxf(v, __int_as_float(OM_ROW_STEP(__float_as_int(v), 0x128)));    // row_ror:8
    v = fmaxf(v, __int_as_float(OM_ROW_STEP(__float_as_int(v), 0x124)));    // row_ror:4
    v = fmaxf(v, __int_as_float(OM_ROW_STEP(__float_as_int(v), 0x4E)));     // quad_perm [2,3,0,1]
    return fmaxf(v, __int_as_float(OM_ROW_STEP(__float_as_int(v), 0xB1)));  // quad_perm [1,0,3,2]
}
__device__ __forceinline__ int row_min(int v) {
    v = min(v, OM_ROW_STEP(v, 0x128));
    v = min(v, OM_ROW_STEP(v, 0x124));
    v = min(v, OM_ROW_STEP(v, 0x4E));
    return min(v, OM_ROW_STEP(v, 0xB1));
}
__device__ __forceinline__ float row_sum(float v) {
    v += __int_as_float(OM_ROW_STEP(__float_as_int(v), 0x128));
    v += __int_as_float(OM_ROW_STEP(__float_as_int(v), 0x124));
    v += __int_as_float(OM_ROW_STEP(__float_as_int(v), 0x4E));
    return v + __int_as_float(OM_ROW_STEP(__float_as_int(v), 0xB1));
}
#undef OM_ROW_STEP

// softmax_in_place and select_topk for four tokens in a wavefront, a row of 16 lanes each: lane l of a row holds
// the logits of experts l + 16 * j in p[j] (past N: -inf), the lane of rank r < K <= 16 gets the r-th winner.  The same
// bits as with a wavefront per token: the sum pairs the same experts, the selection order is total.
// One CU routes the 32 tokens of a block, so it is vector-instruction issue that counts: a round of selection is
// about as many instructions here for four tokens as there for one.
template <int Q>
__device__ __forceinline__ void row_softmax_topk(float (&p)[Q], int N, int K, int l16, float &my_v, int &my_i) {
    float mx = p[0];
#pragma unroll
    for (int j = 1; j < Q; j++) mx = fmaxf(mx, p[j]);
    mx = row_max(mx);
#pragma unroll
    for (int j = 0; j < Q; j++) p[j] = l16 + 16 * j < N ? expf(p[j] - mx) : 0.0f;
    const float sum = row_sum(Q == 4 ? (p[0] + p[2]) + (p[1] + p[3]) : p[0] + p[1]);
#pragma unroll
    for (int j = 0; j < Q; j++) p[j] = l16 + 16 * j < N ? p[j] / sum : -INFINITY;
    my_v = 0.0f;
    my_i = 0;
    for (int r = 0; r < K; r++) {
        float bv = -INFINITY;
        int bi = 0x7fffffff;
#pragma unroll
        for (int j = 0; j < Q; j++)
            if (p[j] > bv) { bv = p[j]; bi = l16 + 16 * j; }   // ascending experts: the first maximum wins
        const float m = row_max(bv);
        const int i = row_min(bv == m ? bi : 0x7fffffff);
        if (l16 == r) { my_v = m; my_i = i; }
#pragma unroll
        for (int j = 0; j < Q; j++)
            if (l16 + 16 * j == i) p[j] = -INFINITY;           // taken
    }
}

// The same for at most 64 experts and hidden sizes that are multiples of 512.  What bounds it is how fast a CU takes in
// 32 rows of x and the whole gate weight (256 KB for 64 experts at hidden 2048), so everything comes by direct loads of
// whole 64-byte row pieces, two steps ahead, through a ring of three steps in LDS: a step is 32 columns of each of eight
// slices of H, a slice has a wavefront for each 32 experts (NB), and those share the slice's rows of x.  Slices are added
// in their order, whatever the number of tokens.  TL: the logits' type; bf16 logits are rounded before the softmax, as a
// bf16 linear layer returns them.
// us with the routing (before: eight wavefronts over eight slices with fragments straight from global memory, 32-byte
// pieces of 64 rows at a time): 64 experts, hidden 2048: 4096 tokens 10.7 (22.0), 16384 tokens 23.6 (38.0: 2.8 TB/s of x
// now); 32 experts, hidden 1024: 512 tokens 4.9 (9.0), 16384 tokens 11.0 (20.6).
template <int NB, typename TL, typename TW, bool ROUTE>
__global__ __launch_bounds__(NB * 512) void gate_route_slices_kernel(const uint16_t *__restrict__ x, const uint16_t *__restrict__ wg,
                                                                     int64_t Tn, int H, int N, int K, int renorm,
                                                                     TL *__restrict__ logits_out, TW *__restrict__ weights_out,
                                                                     int64_t *__restrict__ experts_out) {
    constexpr int NP = NB * 32, SLICES = 8, WAVES = NB * SLICES, SLOTS = 3;
    constexpr int UNITS = 2 + 2 * NB;                       // 1 KB loads (16 rows of 64 bytes) of a slice's step: x, then weight
    constexpr int LOADS = UNITS / NB;                       // of which each wavefront issues
    constexpr int SLICE_BYTES = UNITS * 1024, STEP_BYTES = SLICES * SLICE_BYTES;
    constexpr int LD = NP + 8;                              // (the two halves of a wavefront store to different banks)
    static_assert(SLOTS * STEP_BYTES >= SLICES * 32 * LD * 4, "the partial sums take the ring's place");
    __shared__ __attribute__((aligned(1024))) char lds[SLOTS * STEP_BYTES];
    float (*part)[32][LD] = reinterpret_cast<float (*)[32][LD]>(lds);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int slice = wave / NB, nb = wave % NB;
    const int64_t t0 = static_cast<int64_t>(blockIdx.x) * 32;
    const int steps = H / (SLICES * 32);                    // at least two
    const int r32 = lane & 31;
    // Chunk c (16 bytes) of a 64-byte row r is stored at c ^ (r / 4 % 4): fragment reads of 16 rows use every bank once.
    const char *src[LOADS];
    uint32_t dst[LOADS];
    const uint32_t lds0 = lds_address(lds);
#pragma unroll
    for (int l = 0; l < LOADS; l++) {
        const int unit = nb * LOADS + l, row = (unit < 2 ? unit : unit - 2) * 16 + (lane >> 2);
        const int column = slice * (H / SLICES) + ((lane & 3) ^ (lane >> 4)) * 8;
        // rows past the end (tokens, experts): valid memory, results unused
        src[l] = reinterpret_cast<const char *>(unit < 2 ? x + min(t0 + row, Tn - 1) * H + column
                                                         : wg + static_cast<int64_t>(min(row, N - 1)) * H + column);
        dst[l] = lds0 + slice * SLICE_BYTES + unit * 1024;
    }
    auto issue = [&](int step, int slot) {
#pragma unroll
        for (int l = 0; l < LOADS; l++) dma16_lane(src[l] + step * 64, dst[l] + slot * STEP_BYTES);
    };
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.0f;
    issue(0, 0);
    issue(1, 1);
    int slot = 0, free_slot = 2;
    for (int s = 0; s < steps; s++) {
        // This wavefront's part of step s has landed (step s + 1 may be outstanding); behind the barrier everyone's has, and
        // everyone has read step s - 1, whose slot takes step s + 2.
        if (s + 1 < steps) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (s + 2 < steps) issue(s + 2, free_slot);
        const char *at = lds + slot * STEP_BYTES + slice * SLICE_BYTES + r32 * 64;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int o = ((u * 2 + (lane >> 5)) ^ (r32 >> 2 & 3)) << 4;
            const u32x4 a = *reinterpret_cast<const u32x4 *>(at + o);
            const u32x4 b = *reinterpret_cast<const u32x4 *>(at + 2048 + nb * 2048 + o);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
        }
        free_slot = slot;
        slot = slot == SLOTS - 1 ? 0 : slot + 1;
    }
    __syncthreads();                                        // every step has been read
    // accumulator element r of lane l: token (r/4)*8 + (l/32)*4 + r%4, expert nb*32 + l%32
#pragma unroll
    for (int r = 0; r < 16; r++) part[slice][(r >> 2) * 8 + (lane >> 5) * 4 + (r & 3)][nb * 32 + r32] = acc[r];
    __syncthreads();
    if (!ROUTE || K <= 16) {                                // a row of 16 lanes per token
        constexpr int Q = NP / 16;
        const int l16 = lane & 15, tk = wave * 4 + (lane >> 4);
        if (wave >= 8) return;
        float p[Q];
#pragma unroll
        for (int j = 0; j < Q; j++) p[j] = part[0][tk][l16 + 16 * j];
#pragma unroll
        for (int s = 1; s < SLICES; s++)
#pragma unroll
            for (int j = 0; j < Q; j++) p[j] += part[s][tk][l16 + 16 * j];
        const bool inside = t0 + tk < Tn;
#pragma unroll
        for (int j = 0; j < Q; j++) {
            const int n = l16 + 16 * j;
            if (logits_out && inside && n < N) Elem<TL>::store(logits_out + (t0 + tk) * N + n, p[j]);
            if (sizeof(TL) == 2) p[j] = bf16_bits_to_f32(f32_to_bf16_bits(p[j]));
            if (n >= N) p[j] = -INFINITY;
        }
        if (!ROUTE) return;
        float w; int e;
        row_softmax_topk<Q>(p, N, K, l16, w, e);
        if (renorm) w = w / row_sum(l16 < K ? w : 0.0f);
        if (inside && l16 < K) {
            Elem<TW>::store(weights_out + (t0 + tk) * K + l16, w);
            experts_out[(t0 + tk) * K + l16] = e;
        }
        return;
    }
    for (int tk = wave; tk < 32 && t0 + tk < Tn; tk += WAVES) {   // a wavefront per token
        float p[1] = {-INFINITY};
        if (lane < N) {
            p[0] = part[0][tk][lane];
#pragma unroll
            for (int s = 1; s < SLICES; s++) p[0] += part[s][tk][lane];
            if (logits_out) Elem<TL>::store(logits_out + (t0 + tk) * N + lane, p[0]);
            if (sizeof(TL) == 2) p[0] = bf16_bits_to_f32(f32_to_bf16_bits(p[0]));
        }
        softmax_in_place<1>(N, lane, p);
        float w; int e;
        select_topk<1>(p, N, K, lane, w, e);
        if (renorm) w = w / wave_sum(lane < K ? w : 0.0f);
        if (lane < K) {
            Elem<TW>::store(weights_out + (t0 + tk) * K + lane, w);
            experts_out[(t0 + tk) * K + lane] = e;
        }
    }
}

// partial_softmax_topk_kernel and the sort of its selections (om_moe_sort_weighted) by one block, for up to 64 tokens: a row of 16 lanes per
// token, then a thread per pair.  Either alone is a launch and one chain of waits: one token of 64 experts, top-8, 3.2 + 3.4 -> 5.2 us, 37
// tokens 4.9 + 4.8 -> 8.2 (traced; whole passes 1.7 and 1.4 less).
constexpr int ROUTE_SORT_TOKENS = 64;
struct SortOut {
    int start, end, nbits;
    int32_t *cum_token_counts, *cum_expert_counts_ep, *input_indices, *output_indices, *selected_experts_indices;
    float *row_weights;
};
template <int Q, typename TL, typename TW>
__global__ __launch_bounds__(1024) void partial_softmax_topk_sort_kernel(const float *__restrict__ partial, int splits, int Tn, int N, int K,
                                                                         int renorm, TL *__restrict__ logits_out, TW *__restrict__ weights_out,
                                                                         int64_t *__restrict__ experts_out, const SortOut out) {
    __shared__ int pair_expert[ROUTE_SORT_TOKENS * 16];
    __shared__ float pair_weight[ROUTE_SORT_TOKENS * 16];
    const int l16 = threadIdx.x & 15, t = threadIdx.x >> 4;
    const bool there = t < Tn;
    if ((t & ~3) < Tn) {                                    // (the whole wavefront)
        const float *row = partial + min(t, Tn - 1) * N;
        float p[Q] = {};
        for (int k0 = 0; k0 < splits; k0 += 8) {            // as partial_logits adds them
            float v[8][Q];
#pragma unroll
            for (int u = 0; u < 8; u++)
#pragma unroll
                for (int j = 0; j < Q; j++) v[u][j] = row[static_cast<int64_t>(min(k0 + u, splits - 1)) * Tn * N + min(l16 + 16 * j, N - 1)];
#pragma unroll
            for (int u = 0; u < 8; u++)
#pragma unroll
                for (int j = 0; j < Q; j++) p[j] += k0 + u < splits ? v[u][j] : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < Q; j++) {
            const int n = l16 + 16 * j;
            if (there && n < N) Elem<TL>::store(logits_out + t * N + n, p[j]);
            if (sizeof(TL) == 2) p[j] = bf16_bits_to_f32(f32_to_bf16_bits(p[j]));
            if (n >= N) p[j] = -INFINITY;
        }
        float w; int e;
        row_softmax_topk<Q>(p, N, K, l16, w, e);
        if (renorm) w = w / row_sum(l16 < K ? w : 0.0f);
        if (there && l16 < K) {
            Elem<TW>::store(weights_out + t * K + l16, w);
            experts_out[t * K + l16] = e;
            pair_expert[t * K + l16] = e;
            pair_weight[t * K + l16] = sizeof(TW) == 2 ? bf16_bits_to_f32(f32_to_bf16_bits(w)) : w;   // (as stored)
        }
    }
    __syncthreads();
    const int n_pairs = Tn * K, pair = min(static_cast<int>(threadIdx.x), n_pairs - 1);
    sort_block(pair_expert[pair], pair_weight[pair], n_pairs, K, out.start, out.end, out.end - out.start, out.nbits, out.cum_token_counts,
               out.cum_expert_counts_ep, out.input_indices, out.output_indices, out.selected_experts_indices, out.row_weights);
}

// Projection and routing of up to 64 experts in one launch, 16 tokens at a time, for gates of a small weight: what bounds those is a chain of
// waits and launches.  So a block has eight wavefronts for every 32 experts, each with a slice of H or two, and a wavefront asks for
// 128 columns at a time before it waits: straight into the fragments of v_mfma_f32_16x16x32_bf16, a weight is used by one wavefront only.
// Slices of 64 columns (WHOLE): the weight stays in registers for the block's further tokens, whose x is on its way while the last
// ones are routed (hidden 256: 64 experts, 2048 tokens 9.4 -> 7.6 us, 16384 20.2 -> 16.8).  The slices are added in their order: the sums, and so
// the logits, are those of the split projection, bit for bit.
constexpr int ROWS_TOKENS = 16;

// CH: pieces of 32 columns that are loaded at once; SL: slices at most; WHOLE: a wavefront has at most one slice, of CH pieces.
template <int NH, int CH, int SL, bool WHOLE, typename TL, typename TW>
__global__ __launch_bounds__(NH * 512) void gate_route_rows_kernel(const uint16_t *__restrict__ x, const uint16_t *__restrict__ wg, int64_t Tn, int H,
                                                                   int N, int K, int renorm, int slices, int slice_len,
                                                                   TL *__restrict__ logits_out, TW *__restrict__ weights_out,
                                                                   int64_t *__restrict__ experts_out) {
    constexpr int NP = NH * 32, LD = NP + 4, Q = NP / 16, BUFS = SL > 8 ? 1 : 2;
    __shared__ __attribute__((aligned(16))) float part[BUFS][SL][ROWS_TOKENS][LD];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int half = wave % NH, first_slice = wave / NH;
    const int l16 = lane & 15, g = lane >> 4;
    uint32_t w_row[2];                                      // bytes; rows past the last expert: it again, results unused
#pragma unroll
    for (int m = 0; m < 2; m++) w_row[m] = static_cast<uint32_t>(min(half * 32 + m * 16 + l16, N - 1)) * static_cast<uint32_t>(H) * 2;
    u32x4 wf[CH][2], xf[CH];
    auto at = [](const uint16_t *base, uint32_t bytes) { return *reinterpret_cast<const u32x4 *>(reinterpret_cast<const char *>(base) + bytes); };
    // byte of the lane's chunk in piece i of CH that `columns` are left of: past them the last chunk again, as zeros (of both: zero times an
    // infinite weight is NaN)
    auto chunk = [&](int i, int columns) { return static_cast<uint32_t>(WHOLE ? i * 32 + g * 8 : min(i * 32 + g * 8, columns - 8)) * 2; };
    auto load_w = [&](int begin, int columns) {
#pragma unroll
        for (int i = 0; i < CH; i++)
#pragma unroll
            for (int m = 0; m < 2; m++) {
                wf[i][m] = at(wg + begin, w_row[m] + chunk(i, columns));
                if (!WHOLE && i * 32 + g * 8 >= columns) wf[i][m] = u32x4{0, 0, 0, 0};
            }
    };
    auto load_x = [&](int64_t tile, int begin, int columns) {
        const uint32_t row = static_cast<uint32_t>(min(static_cast<int64_t>(l16), Tn - 1 - tile * ROWS_TOKENS)) * static_cast<uint32_t>(H) * 2;
#pragma unroll
        for (int i = 0; i < CH; i++) {
            xf[i] = at(x + tile * ROWS_TOKENS * H + begin, row + chunk(i, columns));
            if (!WHOLE && i * 32 + g * 8 >= columns) xf[i] = u32x4{0, 0, 0, 0};
        }
    };
    const int64_t tiles = (Tn + ROWS_TOKENS - 1) / ROWS_TOKENS;
    const bool mine = first_slice < slices;
    if (WHOLE && mine) {
        load_w(first_slice * slice_len, 0);
        load_x(blockIdx.x, first_slice * slice_len, 0);
    }
    int buf = 0;
    for (int64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        for (int s = first_slice; s < slices; s += 8) {
            f32x4 acc[2] = {};
            const int begin = s * slice_len, len = min(H - begin, slice_len);
            for (int c = 0; c < (WHOLE ? 1 : len); c += CH * 32) {
                if (!WHOLE) {
                    load_w(begin + c, len - c);
                    load_x(tile, begin + c, len - c);
                }
#pragma unroll
                for (int i = 0; i < CH; i++)
#pragma unroll
                    for (int m = 0; m < 2; m++)
                        acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wf[i][m]), __builtin_bit_cast(bf16x8, xf[i]), acc[m], 0, 0, 0);
            }
            // element r of lane l: expert 4 * (l / 16) + r of token l % 16
#pragma unroll
            for (int m = 0; m < 2; m++) *reinterpret_cast<f32x4 *>(&part[buf][s][l16][half * 32 + m * 16 + g * 4]) = acc[m];
            if (WHOLE) break;
        }
        // (with two buffers the wavefronts that route a tile are at the next tile's barrier before theirs is written again)
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (wave < ROWS_TOKENS / 4) {                       // a row of 16 lanes per token
            const int tk = wave * 4 + g;
            const int64_t t = tile * ROWS_TOKENS + tk;
            float p[Q];
#pragma unroll
            for (int j = 0; j < Q; j++) p[j] = part[buf][0][tk][l16 + 16 * j];
#pragma unroll 2
            for (int s = 1; s < slices; s++)
#pragma unroll
                for (int j = 0; j < Q; j++) p[j] += part[buf][s][tk][l16 + 16 * j];
            const bool there = t < Tn;
#pragma unroll
            for (int j = 0; j < Q; j++) {
                const int n = l16 + 16 * j;
                if (logits_out && there && n < N) Elem<TL>::store(logits_out + t * N + n, p[j]);
                if (sizeof(TL) == 2) p[j] = bf16_bits_to_f32(f32_to_bf16_bits(p[j]));
                if (n >= N) p[j] = -INFINITY;
            }
            float w; int e;
            row_softmax_topk<Q>(p, N, K, l16, w, e);
            if (renorm) w = w / row_sum(l16 < K ? w : 0.0f);
            if (there && l16 < K) {
                Elem<TW>::store(weights_out + t * K + l16, w);
                experts_out[t * K + l16] = e;
            }
        }
        // (the wavefronts that route ask later than the others: beside the weight they have no registers for both)
        if (WHOLE && mine && tile + gridDim.x < tiles) load_x(tile + gridDim.x, first_slice * slice_len, 0);
        if (BUFS == 2) buf ^= 1;
        else asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
}

// Hidden sizes that gate_route_slices_kernel does not take, up to 64 K weights: a block takes in all of them, from memory behind a layer's
// expert products.  Two launches -> one, us, the router alone: 8 experts, hidden 256, 2048 tokens 9.6 -> 6.2, 16384 16.2 -> 9.6; 12 of 1000, 3001
// 10.9 -> 7.1, 16000 21.2 -> 18.0; 64 of 256, 2048 13.9 -> 7.6; 40 of 776, 512 12.1 -> 10.7, 4096 15.5 -> 9.2; 61 of 1000, 512 13.2 -> 13.0, 4096
// 20.8 -> 10.9, 16384 32.4 -> 31.4; but 12 of 4040, 9000 27.2 -> 29.6, 60 of 3000, 9000 34.4 -> 46.5, 64 of 6000, 9000 48.8 -> 84.9.  Hidden sizes that are multiples of
// 512 as fast here as by slices, or up to 15 % slower; with 64 experts of 2048 in a layer, 512 tokens 15.6 against 13.9 in two launches.
inline bool gate_rows_fit(int64_t T, int H, int N, int K) {
    return N <= 64 && K <= 16 && H % 512 != 0 && N * H <= (64 << 10) && om_gate_route_splits(T, H, N) <= 16;
}

template <typename TL, typename TW>
int launch_gate_rows(const void *x, const void *wg, int64_t T, int H, int N, int K, int renorm, void *logits_out, void *weights_out,
                     int64_t *experts_out, hipStream_t st) {
    const int slices = om_gate_route_splits(T, H, N), slice_len = ((H + 63) / 64 + slices - 1) / slices * 64;
    const dim3 grid(static_cast<unsigned>(std::min<int64_t>((T + ROWS_TOKENS - 1) / ROWS_TOKENS, 256)));
    const uint16_t *xp = static_cast<const uint16_t *>(x), *wp = static_cast<const uint16_t *>(wg);
    TL *lo = static_cast<TL *>(logits_out);
    TW *wo = static_cast<TW *>(weights_out);
#define OM_ROWS(NH, CH, SL, WHOLE)                                                                                                        \
    gate_route_rows_kernel<NH, CH, SL, WHOLE, TL, TW><<<grid, NH * 512, 0, st>>>(xp, wp, T, H, N, K, renorm, slices, slice_len, lo, wo, experts_out)
    const bool whole = slices <= 8 && slice_len == 64 && slices * 64 == H;
    if (N <= 32 && whole) OM_ROWS(1, 2, 8, true);
    else if (N <= 32) OM_ROWS(1, 4, 16, false);
    else if (whole) OM_ROWS(2, 2, 8, true);
    else OM_ROWS(2, 4, 16, false);
#undef OM_ROWS
    return om_launch_status();
}

// shapes of gate_route_slices_kernel
inline bool gate_slices_fit(int H, int N) { return N <= 64 && H % 512 == 0; }

template <typename TL, typename TW, bool ROUTE>
int launch_gate_slices(const void *x, const void *wg, int64_t T, int H, int N, int K, int renorm, void *logits_out,
                       void *weights_out, int64_t *experts_out, hipStream_t st) {
    const unsigned nb = static_cast<unsigned>((T + 31) / 32);
    const uint16_t *xp = static_cast<const uint16_t *>(x), *wp = static_cast<const uint16_t *>(wg);
    TL *lo = static_cast<TL *>(logits_out);
    TW *wo = static_cast<TW *>(weights_out);
    if (N <= 32) gate_route_slices_kernel<1, TL, TW, ROUTE><<<nb, 512, 0, st>>>(xp, wp, T, H, N, K, renorm, lo, wo, experts_out);
    else gate_route_slices_kernel<2, TL, TW, ROUTE><<<nb, 1024, 0, st>>>(xp, wp, T, H, N, K, renorm, lo, wo, experts_out);
    return om_launch_status();
}

template <bool ROUTE, typename TW>
int launch_gate(const void *x, const void *wg, int64_t T, int H, int N, int K, int renorm,
                float *logits_out, void *weights_out, int64_t *experts_out, hipStream_t st) {
    const unsigned nb = static_cast<unsigned>((T + 31) / 32);
    const uint16_t *xp = static_cast<const uint16_t *>(x), *wp = static_cast<const uint16_t *>(wg);
    TW *wo = static_cast<TW *>(weights_out);
#define OM_GATE(NB, WAVES, UNR, PER)                                                              \
    do {                                                                                          \
        if (H % (WAVES * 16 * UNR) != 0) return OM_ERR_SHAPE;                                     \
        gate_route_kernel<NB, WAVES, UNR, PER, TW, ROUTE><<<nb, WAVES * 64, 0, st>>>(             \
            xp, wp, T, H, N, K, renorm, logits_out, wo, experts_out);                             \
    } while (0)
    if (N <= 64) {
        if (!gate_slices_fit(H, N)) return OM_ERR_SHAPE;
        return launch_gate_slices<float, TW, ROUTE>(x, wg, T, H, N, K, renorm, logits_out, weights_out, experts_out, st);
    }
    if (N <= 128) OM_GATE(4, 8, 2, 2);
    else OM_GATE(8, 4, 1, 4);
#undef OM_GATE
    return om_launch_status();
}

// Load-balancing statistics of one layer's router logits: for every expert the sum over tokens
// of its softmax probability and the number of tokens whose top-K contains it (the two factors of
// the auxiliary loss, reference optimus/models/olmoe/modeling_olmoe.py:29-85).  A block walks
// BAL_TOKENS tokens, one wavefront per token at a time, and leaves one partial row; a second
// kernel adds the rows in block order, so the result does not depend on scheduling.
// What bounds both is a chain of latencies, not the 4 MB of logits: with four wavefronts a block took 16
// softmax and top-K selections one after another (46 us at 16384 tokens, 64 experts), and one thread per
// expert then added 256 rows with one load in flight (66 us).  Sixteen wavefronts per block and 16 loads in
// flight: 17.5 us and balance_sums'.
constexpr int BAL_TOKENS = 64, BAL_WAVES = 16;
template <int PER, typename T>
__global__ __launch_bounds__(BAL_WAVES * 64) void balance_stats_kernel(const T *__restrict__ logits,
                                                                       const float *__restrict__ token_weight,
                                                                       int64_t Tn, int N, int K,
                                                                       float *__restrict__ part_prob,
                                                                       float *__restrict__ part_count) {
    __shared__ float lds[BAL_WAVES][PER * 64];   // the probabilities first, then the counts
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float psum[PER];
    float cnt[PER];   // sums of token weights; whole numbers (exact) for 0/1 weights and without weights
#pragma unroll
    for (int j = 0; j < PER; j++) { psum[j] = 0.0f; cnt[j] = 0.0f; }
    const int64_t t_first = static_cast<int64_t>(blockIdx.x) * BAL_TOKENS;
    for (int i = wave; i < BAL_TOKENS; i += BAL_WAVES) {
        const int64_t t = t_first + i;
        if (t >= Tn) break;
        const float tw = token_weight ? token_weight[t] : 1.0f;   // the token's attention-mask entry
        float p[PER], s[PER];
        row_softmax<PER, T>(logits + t * N, N, lane, p);
#pragma unroll
        for (int j = 0; j < PER; j++) { psum[j] += token_weight ? tw * p[j] : p[j]; s[j] = p[j]; }
        float w; int e;
        select_topk<PER>(s, N, K, lane, w, e);
        for (int k = 0; k < K; k++) {
            const int ek = __shfl(e, k, 64);
#pragma unroll
            for (int j = 0; j < PER; j++)
                if (lane + 64 * j == ek) cnt[j] += tw;
        }
    }
#pragma unroll
    for (int q = 0; q < 2; q++) {
        if (q) __syncthreads();
#pragma unroll
        for (int j = 0; j < PER; j++) lds[wave][lane + 64 * j] = q ? cnt[j] : psum[j];
        __syncthreads();
        for (int i = threadIdx.x; i < N; i += BAL_WAVES * 64) {
            float v[BAL_WAVES];
#pragma unroll
            for (int w = 0; w < BAL_WAVES; w++) v[w] = lds[w][i];
#pragma unroll
            for (int n = BAL_WAVES / 2; n > 0; n /= 2)
#pragma unroll
                for (int w = 0; w < n; w++) v[w] += v[w + n];
            (q ? part_count : part_prob)[static_cast<int64_t>(blockIdx.x) * N + i] = v[0];
        }
    }
}

// The partial rows of 64 experts: a sixteenth of them to each wavefront, 16 loads in flight, then the wavefronts' sums in a fixed
// order; lane i of wavefront 0 has expert i's.  (One wavefront for all: 256 rows 8.6 us -> 4.3.)
__device__ __forceinline__ void balance_sums(const float *part_prob, const float *part_count, int n_blocks, int N, int i, float &prob, float &count) {
    __shared__ float lds_p[BAL_WAVES][64];
    __shared__ double lds_c[BAL_WAVES][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float ps = 0.0f;
    // a block's partial is a sum of at most BAL_TOKENS token weights (whole numbers for 0/1 weights
    // and without weights); adding the partials in double keeps whole-number counts exact at any
    // token count (a hot expert can exceed 2^24 tokens), one rounding to float at the end
    double c = 0.0;
    if (i < N) {
        int b = static_cast<int>(static_cast<int64_t>(n_blocks) * wave / BAL_WAVES);
        const int end = static_cast<int>(static_cast<int64_t>(n_blocks) * (wave + 1) / BAL_WAVES);
        for (; b + 16 <= end; b += 16) {
            float p[16], q[16];
#pragma unroll
            for (int u = 0; u < 16; u++) {
                p[u] = part_prob[static_cast<int64_t>(b + u) * N + i];
                q[u] = part_count[static_cast<int64_t>(b + u) * N + i];
            }
#pragma unroll
            for (int u = 0; u < 16; u++) {
                ps += p[u];
                c += static_cast<double>(q[u]);
            }
        }
        for (; b < end; b++) {
            ps += part_prob[static_cast<int64_t>(b) * N + i];
            c += static_cast<double>(part_count[static_cast<int64_t>(b) * N + i]);
        }
    }
    __syncthreads();   // (a group of experts before this one has been read)
    lds_p[wave][lane] = ps;
    lds_c[wave][lane] = c;
    __syncthreads();
    if (wave == 0) {
        for (int w = 1; w < BAL_WAVES; w++) {
            ps += lds_p[w][lane];
            c += lds_c[w][lane];
        }
    }
    prob = ps;
    count = static_cast<float>(c);
}
__global__ __launch_bounds__(BAL_WAVES * 64) void balance_reduce_kernel(const float *__restrict__ part_prob, const float *__restrict__ part_count,
                                                                        int n_blocks, int N, float *__restrict__ prob_sum,
                                                                        float *__restrict__ count) {
    const int i = blockIdx.x * 64 + (threadIdx.x & 63);
    float p, c;
    balance_sums(part_prob, part_count, n_blocks, N, i, p, c);
    if (threadIdx.x < 64 && i < N) {
        prob_sum[i] = p;
        count[i] = c;
    }
}
// The same, and loss = scale * sum over the experts of (count / T) * (prob_sum / T): one block.
__global__ __launch_bounds__(BAL_WAVES * 64) void balance_loss_kernel(const float *__restrict__ part_prob, const float *__restrict__ part_count,
                                                                      int n_blocks, int64_t Tn, int N, float scale, float *__restrict__ count,
                                                                      float *__restrict__ loss) {
    const float t = static_cast<float>(Tn);
    float sum = 0.0f;
    for (int e0 = 0; e0 < N; e0 += 64) {
        const int i = e0 + (threadIdx.x & 63);
        float p, c;
        balance_sums(part_prob, part_count, n_blocks, N, i, p, c);
        if (i < N) sum += (c / t) * (p / t);
        if (threadIdx.x < 64 && i < N) count[i] = c;
    }
    sum = wave_sum(sum);
    if (threadIdx.x == 0) *loss = sum * scale;
}

// dlogits[t,i] = p_i * (g_i - sum_j p_j g_j): the softmax backward of sum_i g_i * p[t,i].
// LOSS: g holds the counts, and the gradient of the probabilities' sums is that of the loss: grad * scale * (count / T) / T.
template <int PER, typename T, bool LOSS = false>
__global__ __launch_bounds__(256) void balance_bwd_kernel(const T *__restrict__ logits,
                                                          const float *__restrict__ g,
                                                          const float *__restrict__ token_weight,
                                                          int64_t Tn, int N, T *__restrict__ dlogits,
                                                          const float *__restrict__ grad = nullptr, float scale = 0.0f) {
    const int lane = threadIdx.x & 63;
    const int64_t t = static_cast<int64_t>(blockIdx.x) * TOKENS_PER_BLOCK + (threadIdx.x >> 6);
    if (t >= Tn) return;
    float p[PER];
    row_softmax<PER, T>(logits + t * N, N, lane, p);
    float gv[PER], dot = 0.0f;
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int i = lane + 64 * j;
        gv[j] = (i < N) ? g[i] : 0.0f;
        if (LOSS) gv[j] = ((*grad * scale) * (gv[j] / static_cast<float>(Tn))) / static_cast<float>(Tn);
        dot += p[j] * gv[j];
    }
    dot = wave_sum(dot);
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int i = lane + 64 * j;
        if (i < N) Elem<T>::store(dlogits + t * N + i, (token_weight ? token_weight[t] : 1.0f) * (p[j] * (gv[j] - dot)));
    }
}

inline unsigned token_blocks(int64_t T) {
    return static_cast<unsigned>((T + TOKENS_PER_BLOCK - 1) / TOKENS_PER_BLOCK);
}
inline int per_lane(int N) { return N <= 64 ? 1 : N <= 128 ? 2 : N <= 256 ? 4 : 8; }

}  // namespace

#define OM_DISPATCH_PER(N, CALL)              \
    switch (per_lane(N)) {                    \
        case 1: { constexpr int PER = 1; CALL; } break; \
        case 2: { constexpr int PER = 2; CALL; } break; \
        case 4: { constexpr int PER = 4; CALL; } break; \
        default: { constexpr int PER = 8; CALL; } break; \
    }

extern "C" int om_router_gate_logits_f32(const float *x, const float *gate_weight, int64_t T, int H, int N,
                                         float *logits_out, void *stream) {
    if (T < 0 || T > 0x7fffffffLL || H < 1 || N < 1 || N > 65535) return OM_ERR_SHAPE;
    if (T == 0) return OM_OK;
    if (!x || !gate_weight || !logits_out) return OM_ERR_NULL;
    gate_f32_kernel<false, float><<<token_blocks(T), 256, 0, om_stream(stream)>>>(x, gate_weight, T, H, N, 0, 0, logits_out, nullptr, nullptr);
    return om_launch_status();
}

extern "C" int om_router_gate_softmax_topk_f32(const float *x, const float *gate_weight, int64_t T, int H, int N, int K, int norm_topk_prob,
                                               float *logits_out, void *weights_out, int weights_dtype, int64_t *experts_out, void *stream) {
    if (weights_dtype != OM_F32 && weights_dtype != OM_BF16) return OM_ERR_DTYPE;
    if (T < 0 || T > 0x7fffffffLL || H < 1 || N < 1 || N > 64 || K < 1 || K > N) return OM_ERR_SHAPE;
    if (T == 0) return OM_OK;
    if (!x || !gate_weight || !logits_out || !weights_out || !experts_out) return OM_ERR_NULL;
    if (weights_dtype == OM_F32)
        gate_f32_kernel<true, float><<<token_blocks(T), 256, 0, om_stream(stream)>>>(x, gate_weight, T, H, N, K, norm_topk_prob, logits_out,
                                                                                  static_cast<float *>(weights_out), experts_out);
    else
        gate_f32_kernel<true, uint16_t><<<token_blocks(T), 256, 0, om_stream(stream)>>>(x, gate_weight, T, H, N, K, norm_topk_prob, logits_out,
                                                                                     static_cast<uint16_t *>(weights_out), experts_out);
    return om_launch_status();
}

extern "C" int om_route_softmax_topk(const void *logits, int logits_dtype, int64_t T, int N, int K,
                                     int norm_topk_prob, void *weights_out, int weights_dtype,
                                     int64_t *experts_out, void *stream) {
    if ((logits_dtype != OM_F32 && logits_dtype != OM_BF16) ||
        (weights_dtype != OM_F32 && weights_dtype != OM_BF16))
        return OM_ERR_DTYPE;
    if (T < 0 || N < 1 || N > 512 || K < 1 || K > N || K > 64 || T > 0x7fffffffLL) return OM_ERR_SHAPE;
    if (T == 0) return OM_OK;
    if (!logits || !weights_out || !experts_out) return OM_ERR_NULL;
    hipStream_t st = om_stream(stream);
    const unsigned nb = token_blocks(T);
#define OM_RT(TL, TW)                                                                          \
    OM_DISPATCH_PER(N, (softmax_topk_kernel<PER, TL, TW><<<nb, 256, 0, st>>>(                  \
                           static_cast<const TL *>(logits), T, N, K, norm_topk_prob,           \
                           static_cast<TW *>(weights_out), experts_out)))
    if (logits_dtype == OM_F32 && weights_dtype == OM_F32) { OM_RT(float, float); }
    else if (logits_dtype == OM_F32) { OM_RT(float, uint16_t); }
    else if (weights_dtype == OM_F32) { OM_RT(uint16_t, float); }
    else { OM_RT(uint16_t, uint16_t); }
#undef OM_RT
    return om_launch_status();
}

extern "C" int om_route_softmax_topk_bwd(const void *logits, int logits_dtype, const int64_t *experts,
                                         const void *dweights, int weights_dtype, int64_t T, int N,
                                         int K, int norm_topk_prob, void *dlogits, void *stream) {
    if ((logits_dtype != OM_F32 && logits_dtype != OM_BF16) ||
        (weights_dtype != OM_F32 && weights_dtype != OM_BF16))
        return OM_ERR_DTYPE;
    if (T < 0 || N < 1 || N > 512 || K < 1 || K > N || K > 64 || T > 0x7fffffffLL) return OM_ERR_SHAPE;
    if (T == 0) return OM_OK;
    if (!logits || !experts || !dweights || !dlogits) return OM_ERR_NULL;
    hipStream_t st = om_stream(stream);
    const unsigned nb = token_blocks(T);
#define OM_RB(TL, TW)                                                                          \
    OM_DISPATCH_PER(N, (softmax_topk_bwd_kernel<PER, TL, TW, TL><<<nb, 256, 0, st>>>(          \
                           static_cast<const TL *>(logits), experts,                           \
                           static_cast<const TW *>(dweights), T, N, K, norm_topk_prob,         \
                           static_cast<TL *>(dlogits), nullptr, nullptr, 0)))
    if (logits_dtype == OM_F32 && weights_dtype == OM_F32) { OM_RB(float, float); }
    else if (logits_dtype == OM_F32) { OM_RB(float, uint16_t); }
    else if (weights_dtype == OM_F32) { OM_RB(uint16_t, float); }
    else { OM_RB(uint16_t, uint16_t); }
#undef OM_RB
    return om_launch_status();
}

// (up to 64 experts)
void om_launch_softmax_bwd(const void *logits, int logits_dtype, const int64_t *experts, const void *dweights, int dweights_dtype,
                           const void *more, int64_t T, int N, int K, int renorm, float *dlogits, unsigned *zero, int n_zero,
                           hipStream_t stream) {
#define OM_RB(TL, TW)                                                                                                               \
    softmax_topk_bwd_kernel<1, TL, TW, float><<<token_blocks(T), 256, 0, stream>>>(static_cast<const TL *>(logits), experts,            \
                                                                                  static_cast<const TW *>(dweights), T, N, K, renorm, \
                                                                                  dlogits, static_cast<const TL *>(more), zero, n_zero)
    if (logits_dtype == OM_F32 && dweights_dtype == OM_F32) OM_RB(float, float);
    else if (logits_dtype == OM_F32) OM_RB(float, uint16_t);
    else if (dweights_dtype == OM_F32) OM_RB(uint16_t, float);
    else OM_RB(uint16_t, uint16_t);
#undef OM_RB
}

extern "C" int om_route_sigmoid_group_topk(const float *logits, const float *bias, int64_t T, int N,
                                           int n_group, int topk_group, int K, int norm_topk_prob,
                                           double routed_scaling_factor, int64_t *experts_out,
                                           float *weights_out, void *stream) {
    if (T < 0 || N < 1 || N > 512 || K < 1 || K > N || K > 64 || n_group < 1 || n_group > 64 ||
        N % n_group != 0 || topk_group < 1 || topk_group > n_group || T > 0x7fffffffLL)
        return OM_ERR_SHAPE;
    if (T == 0) return OM_OK;
    if (!logits || !bias || !experts_out || !weights_out) return OM_ERR_NULL;
    hipStream_t st = om_stream(stream);
    const unsigned nb = token_blocks(T);
    const float scale = static_cast<float>(routed_scaling_factor);
    OM_DISPATCH_PER(N, (sigmoid_group_topk_kernel<PER, false, float><<<nb, 256, 0, st>>>(
                           logits, 0, nullptr, bias, T, N, n_group, topk_group, K, norm_topk_prob, scale,
                           experts_out, weights_out)));
    return om_launch_status();
}

extern "C" int om_route_sigmoid_topk_bwd(const float *logits, const int64_t *experts,
                                         const float *dweights, int64_t T, int N, int K,
                                         int norm_topk_prob, double routed_scaling_factor,
                                         float *dlogits, void *stream) {
    if (T < 0 || N < 1 || N > 512 || K < 1 || K > N || K > 64 || T > 0x7fffffffLL) return OM_ERR_SHAPE;
    if (T == 0) return OM_OK;
    if (!logits || !experts || !dweights || !dlogits) return OM_ERR_NULL;
    hipStream_t st = om_stream(stream);
    const unsigned nb = token_blocks(T);
    const float scale = static_cast<float>(routed_scaling_factor);
    OM_DISPATCH_PER(N, (sigmoid_topk_bwd_kernel<PER><<<nb, 256, 0, st>>>(
                           logits, experts, dweights, T, N, K, norm_topk_prob, scale, dlogits)));
    return om_launch_status();
}

extern "C" int om_router_gate_softmax_topk(const void *x, const void *gate_weight, int64_t T, int H,
                                           int N, int K, int norm_topk_prob, float *logits_out,
                                           void *weights_out, int weights_dtype, int64_t *experts_out,
                                           void *stream) {
    if (weights_dtype != OM_F32 && weights_dtype != OM_BF16) return OM_ERR_DTYPE;
    if (T < 0 || H < 1 || H % 8 != 0 || N < 1 || N > 256 || K < 1 || K > N || K > 64 ||
        T > 0x7fffffffLL)
        return OM_ERR_SHAPE;
    if (T == 0) return OM_OK;
    if (!x || !gate_weight || !weights_out || !experts_out) return OM_ERR_NULL;
    if (!om_aligned16(x) || !om_aligned16(gate_weight)) return OM_ERR_ALIGN;
    hipStream_t st = om_stream(stream);
    if (weights_dtype == OM_F32)
        return launch_gate<true, float>(x, gate_weight, T, H, N, K, norm_topk_prob, logits_out,
                                        weights_out, experts_out, st);
    return launch_gate<true, uint16_t>(x, gate_weight, T, H, N, K, norm_topk_prob, logits_out,
                                       weights_out, experts_out, st);
}

namespace {
// What the two entry points below have in common: the projection's slices into the workspace.
int gate_operands(const void *x, const void *gate_weight, int64_t T, int H, int N, const void *workspace,
                  int64_t workspace_bytes) {
    const int64_t need = om_router_gate_route_workspace_bytes(T, H, N);
    if (need < 0) return static_cast<int>(need);
    if (!x || !gate_weight || !workspace) return OM_ERR_NULL;
    if (!om_aligned16(x) || !om_aligned16(gate_weight) || !om_aligned16(workspace)) return OM_ERR_ALIGN;
    return workspace_bytes < need ? OM_ERR_WORKSPACE : OM_OK;
}

int gate_partials(const void *x, const void *gate_weight, int64_t T, int H, int N, void *workspace, void *stream) {
    const int splits = om_gate_route_splits(T, H, N);
    om_launch_gate_partials(x, gate_weight, T, H, N, splits, static_cast<float *>(workspace), om_stream(stream));
    return splits;
}
}  // namespace

// Whether the router of these sizes is the split projection and a routing launch that can sort as well.
extern "C" int om_router_gate_softmax_topk_sort_fits(int64_t T, int H, int N, int K) {
    if (T < 1 || T > ROUTE_SORT_TOKENS || H < 8 || H % 8 != 0 || N < 1 || N > 64 || K < 1 || K > N || K > 16) return 0;
    return gate_rows_fit(T, H, N, K) || (gate_slices_fit(H, N) && H < 1024) ? 0 : 1;
}

extern "C" int om_router_gate_softmax_topk_sort(const void *x, const void *gate_weight, int64_t T, int H, int N, int K, int norm_topk_prob,
                                                void *logits_out, int logits_dtype, void *weights_out, int weights_dtype,
                                                int64_t *experts_out, int expert_start_idx, int expert_end_idx,
                                                int32_t *cum_token_counts, int32_t *cum_expert_counts_ep, int32_t *input_indices,
                                                int32_t *output_indices, int32_t *selected_experts_indices, float *row_weights,
                                                void *workspace, int64_t workspace_bytes, void *stream) {
    if ((weights_dtype != OM_F32 && weights_dtype != OM_BF16) || (logits_dtype != OM_F32 && logits_dtype != OM_BF16))
        return OM_ERR_DTYPE;
    if (!om_router_gate_softmax_topk_sort_fits(T, H, N, K) || expert_start_idx < 0 || expert_end_idx <= expert_start_idx || expert_end_idx > N)
        return OM_ERR_SHAPE;
    for (const void *p : {static_cast<const void *>(logits_out), static_cast<const void *>(weights_out), static_cast<const void *>(experts_out),
                          static_cast<const void *>(cum_token_counts), static_cast<const void *>(cum_expert_counts_ep),
                          static_cast<const void *>(input_indices), static_cast<const void *>(output_indices),
                          static_cast<const void *>(selected_experts_indices)})
        if (!p) return OM_ERR_NULL;
    const int rc = gate_operands(x, gate_weight, T, H, N, workspace, workspace_bytes);
    if (rc != OM_OK) return rc;
    const int splits = gate_partials(x, gate_weight, T, H, N, workspace, stream);
    const SortOut out = {expert_start_idx, expert_end_idx, key_bits(expert_end_idx - expert_start_idx), cum_token_counts, cum_expert_counts_ep,
                         input_indices, output_indices, selected_experts_indices, row_weights};
#define OM_PS(Q, TL, TW)                                                                                                            \
    partial_softmax_topk_sort_kernel<Q, TL, TW><<<1, 1024, 0, om_stream(stream)>>>(static_cast<const float *>(workspace), splits,      \
        static_cast<int>(T), N, K, norm_topk_prob, static_cast<TL *>(logits_out), static_cast<TW *>(weights_out), experts_out, out)
#define OM_PS_Q(TL, TW)                       \
    do {                                      \
        if (N <= 32) OM_PS(2, TL, TW);        \
        else OM_PS(4, TL, TW);                \
    } while (0)
    if (logits_dtype == OM_F32 && weights_dtype == OM_F32) OM_PS_Q(float, float);
    else if (logits_dtype == OM_F32) OM_PS_Q(float, uint16_t);
    else if (weights_dtype == OM_F32) OM_PS_Q(uint16_t, float);
    else OM_PS_Q(uint16_t, uint16_t);
#undef OM_PS_Q
#undef OM_PS
    return om_launch_status();
}

extern "C" int om_router_gate_split_softmax_topk(const void *x, const void *gate_weight, int64_t T, int H, int N, int K,
                                                 int norm_topk_prob, void *logits_out, int logits_dtype,
                                                 void *weights_out, int weights_dtype, int64_t *experts_out,
                                                 void *workspace, int64_t workspace_bytes, void *stream) {
    if ((weights_dtype != OM_F32 && weights_dtype != OM_BF16) || (logits_dtype != OM_F32 && logits_dtype != OM_BF16))
        return OM_ERR_DTYPE;
    if (T < 0 || N < 1 || K < 1 || K > N || K > 64) return OM_ERR_SHAPE;
    if (T == 0) return OM_OK;
    if (!logits_out || !weights_out || !experts_out) return OM_ERR_NULL;
    const int rc = gate_operands(x, gate_weight, T, H, N, workspace, workspace_bytes);
    if (rc != OM_OK) return rc;
    hipStream_t st = om_stream(stream);
    // One launch or two: with the gate weight out of the caches (after a forward's expert weights) one CU waits for it longer
    // than many do.  A whole MoE forward of 64 experts, hidden 2048, us, one launch -> two: 1 token 43.7 -> 41.8, 37 tokens
    // 173.7 -> 171.8; 512 tokens (with the backward) 700 -> 701; 4096 tokens 520.7 -> 524.2.  In the caches, the router alone:
    // 1 token 7.7 -> 7.8, 512 tokens 8.1 -> 12.2, 4096 tokens 10.7 -> 19.0, and at hidden 7168 15.5 -> 11.5, 16.2 -> 18.5 and
    // 25.8 -> 26.7.  Below hidden 1024 the weight is small: 512, 32 experts, 512 tokens 4.4 -> 9.2.
    // More than 16 selections take a wavefront per token, of a block's 32 tokens two or four to each of its wavefronts: one launch
    // only where its blocks (256 at a time) fill their last round by three quarters and there are 16 wavefronts, or for a few
    // tokens of a small weight.  One -> two, 64 experts, hidden 2048, 32 selections: 600 tokens 24.3 -> 16.2, 4500 27.2 -> 31.2, 8192 28.8 ->
    // 37.9, 12000 53.9 -> 51.4, 16384 56.5 -> 66.7; 60 selections, hidden 4096: 6000 49.1 -> 46.3, 8192 52.2 -> 57.0; 32 experts, 24
    // selections, hidden 2048: 600 24.8 -> 13.0, 8192 28.0 -> 27.4, 12000 53.2 -> 38.9; hidden 512, 40 of 62: 4 tokens 10.1 -> 12.4, 20 of
    // 40: 52 tokens 15.4 -> 9.5.
    const bool one_launch = K <= 16 ? T > 512 || H < 1024 : H < 1024 && T <= 16 ? true : N > 32 && (T - 1) % 8192 >= 6144;
    if (gate_rows_fit(T, H, N, K)) {
#define OM_GR(TL, TW) launch_gate_rows<TL, TW>(x, gate_weight, T, H, N, K, norm_topk_prob, logits_out, weights_out, experts_out, st)
        if (logits_dtype == OM_F32) return weights_dtype == OM_F32 ? OM_GR(float, float) : OM_GR(float, uint16_t);
        return weights_dtype == OM_F32 ? OM_GR(uint16_t, float) : OM_GR(uint16_t, uint16_t);
#undef OM_GR
    }
    if (gate_slices_fit(H, N) && one_launch) {
#define OM_GS(TL, TW) \
    launch_gate_slices<TL, TW, true>(x, gate_weight, T, H, N, K, norm_topk_prob, logits_out, weights_out, experts_out, st)
        if (logits_dtype == OM_F32) return weights_dtype == OM_F32 ? OM_GS(float, float) : OM_GS(float, uint16_t);
        return weights_dtype == OM_F32 ? OM_GS(uint16_t, float) : OM_GS(uint16_t, uint16_t);
#undef OM_GS
    }
    const int splits = gate_partials(x, gate_weight, T, H, N, workspace, stream);
    const unsigned nb = token_blocks(T);
    const float *part = static_cast<const float *>(workspace);
#define OM_PR(TL, TW)                                                                                     \
    OM_DISPATCH_PER(N, (partial_softmax_topk_kernel<PER, TL, TW><<<nb, 256, 0, st>>>(                     \
                           part, splits, T, N, K, norm_topk_prob, static_cast<TL *>(logits_out),          \
                           static_cast<TW *>(weights_out), experts_out)))
    if (logits_dtype == OM_F32 && weights_dtype == OM_F32) { OM_PR(float, float); }
    else if (logits_dtype == OM_F32) { OM_PR(float, uint16_t); }
    else if (weights_dtype == OM_F32) { OM_PR(uint16_t, float); }
    else { OM_PR(uint16_t, uint16_t); }
#undef OM_PR
    return om_launch_status();
}

extern "C" int om_router_gate_split_sigmoid_group_topk_bias(const void *x, const void *gate_weight, const void *bias, int bias_dtype,
                                                            int64_t T, int H, int N, int n_group, int topk_group, int K,
                                                            int norm_topk_prob, double routed_scaling_factor, float *logits_out,
                                                            int64_t *experts_out, float *weights_out, void *workspace,
                                                            int64_t workspace_bytes, void *stream) {
    if (bias_dtype != OM_F32 && bias_dtype != OM_BF16) return OM_ERR_DTYPE;
    if (T < 0 || N < 1 || K < 1 || K > N || K > 64 || n_group < 1 || n_group > 64 || N % n_group != 0 ||
        topk_group < 1 || topk_group > n_group)
        return OM_ERR_SHAPE;
    if (T == 0) return OM_OK;
    if (!bias || !logits_out || !experts_out || !weights_out) return OM_ERR_NULL;
    const int rc = gate_operands(x, gate_weight, T, H, N, workspace, workspace_bytes);
    if (rc != OM_OK) return rc;
    const int splits = gate_partials(x, gate_weight, T, H, N, workspace, stream);
    hipStream_t st = om_stream(stream);
    const float *part = static_cast<const float *>(workspace);
    const float scale = static_cast<float>(routed_scaling_factor);
    const int lanes = N / n_group / QUADS;
    const bool quads = N / n_group % QUADS == 0 && (lanes & (lanes - 1)) == 0 && om_aligned16(logits_out);
#define OM_SG(TB)                                                                                                              \
    do {                                                                                                                       \
        const TB *bp = static_cast<const TB *>(bias);                                                                          \
        if (quads) {                                                                                                           \
            const int waves = T <= 1024 ? 1 : TOKENS_PER_BLOCK;                                                                \
            sigmoid_group_quads_kernel<TB><<<static_cast<unsigned>((T + waves - 1) / waves), waves * 64, 0, st>>>(             \
                part, splits, logits_out, bp, T, N, n_group, topk_group, K, norm_topk_prob, scale, experts_out, weights_out);  \
        } else {                                                                                                               \
            OM_DISPATCH_PER(N, (sigmoid_group_topk_kernel<PER, true, TB><<<token_blocks(T), 256, 0, st>>>(                     \
                                   part, splits, logits_out, bp, T, N, n_group, topk_group, K, norm_topk_prob, scale,          \
                                   experts_out, weights_out)));                                                                \
        }                                                                                                                      \
    } while (0)
    if (bias_dtype == OM_F32) OM_SG(float);
    else OM_SG(uint16_t);
#undef OM_SG
    return om_launch_status();
}

extern "C" int om_router_gate_split_sigmoid_group_topk(const void *x, const void *gate_weight, const float *bias, int64_t T,
                                                       int H, int N, int n_group, int topk_group, int K,
                                                       int norm_topk_prob, double routed_scaling_factor,
                                                       float *logits_out, int64_t *experts_out, float *weights_out,
                                                       void *workspace, int64_t workspace_bytes, void *stream) {
    return om_router_gate_split_sigmoid_group_topk_bias(x, gate_weight, bias, OM_F32, T, H, N, n_group, topk_group, K, norm_topk_prob,
                                                        routed_scaling_factor, logits_out, experts_out, weights_out, workspace,
                                                        workspace_bytes, stream);
}

extern "C" int om_router_gate_logits(const void *x, const void *gate_weight, int64_t T, int H, int N,
                                     float *logits_out, void *stream) {
    if (T < 0 || H < 1 || H % 8 != 0 || N < 1 || N > 256 || T > 0x7fffffffLL) return OM_ERR_SHAPE;
    if (T == 0) return OM_OK;
    if (!x || !gate_weight || !logits_out) return OM_ERR_NULL;
    if (!om_aligned16(x) || !om_aligned16(gate_weight)) return OM_ERR_ALIGN;
    return launch_gate<false, float>(x, gate_weight, T, H, N, 1, 0, logits_out, nullptr, nullptr,
                                     om_stream(stream));
}

extern "C" int64_t om_router_balance_workspace_bytes(int64_t T, int N) {
    if (T < 0 || N < 1) return 0;
    const int64_t blocks = (T + BAL_TOKENS - 1) / BAL_TOKENS;
    return blocks * N * 8;   // one float and one int per (block, expert)
}

namespace {
struct BalancePartials { const float *prob, *count; int blocks; };
BalancePartials balance_partials(const void *logits, int logits_dtype, const float *token_weight, int64_t T, int N, int K, void *workspace,
                                 hipStream_t st) {
    const int nb = static_cast<int>((T + BAL_TOKENS - 1) / BAL_TOKENS);
    float *pp = static_cast<float *>(workspace);
    float *pc = pp + static_cast<int64_t>(nb) * N;
    if (logits_dtype == OM_F32) {
        OM_DISPATCH_PER(N, (balance_stats_kernel<PER, float><<<nb, BAL_WAVES * 64, 0, st>>>(
                               static_cast<const float *>(logits), token_weight, T, N, K, pp, pc)));
    } else {
        OM_DISPATCH_PER(N, (balance_stats_kernel<PER, uint16_t><<<nb, BAL_WAVES * 64, 0, st>>>(
                               static_cast<const uint16_t *>(logits), token_weight, T, N, K, pp, pc)));
    }
    return {pp, pc, nb};
}
}  // namespace

extern "C" int om_router_balance_stats_masked(const void *logits, int logits_dtype,
                                              const float *token_weight, int64_t T, int N, int K,
                                              float *prob_sum, float *count, void *workspace,
                                              int64_t workspace_bytes, void *stream) {
    if (logits_dtype != OM_F32 && logits_dtype != OM_BF16) return OM_ERR_DTYPE;
    if (T < 1 || N < 1 || N > 512 || K < 1 || K > N || K > 64 || T > 0x7fffffffLL) return OM_ERR_SHAPE;
    if (!logits || !prob_sum || !count || !workspace) return OM_ERR_NULL;
    if (workspace_bytes < om_router_balance_workspace_bytes(T, N)) return OM_ERR_WORKSPACE;
    hipStream_t st = om_stream(stream);
    const BalancePartials p = balance_partials(logits, logits_dtype, token_weight, T, N, K, workspace, st);
    balance_reduce_kernel<<<(N + 63) / 64, BAL_WAVES * 64, 0, st>>>(p.prob, p.count, p.blocks, N, prob_sum, count);
    return om_launch_status();
}

extern "C" int om_router_balance_stats(const void *logits, int logits_dtype, int64_t T, int N, int K,
                                       float *prob_sum, float *count, void *workspace,
                                       int64_t workspace_bytes, void *stream) {
    return om_router_balance_stats_masked(logits, logits_dtype, nullptr, T, N, K, prob_sum, count,
                                          workspace, workspace_bytes, stream);
}

extern "C" int om_router_balance_bwd_masked(const void *logits, int logits_dtype, const float *prob_grad,
                                            const float *token_weight, int64_t T, int N, void *dlogits,
                                            void *stream) {
    if (logits_dtype != OM_F32 && logits_dtype != OM_BF16) return OM_ERR_DTYPE;
    if (T < 0 || N < 1 || N > 512 || T > 0x7fffffffLL) return OM_ERR_SHAPE;
    if (T == 0) return OM_OK;
    if (!logits || !prob_grad || !dlogits) return OM_ERR_NULL;
    hipStream_t st = om_stream(stream);
    const unsigned nb = token_blocks(T);
    if (logits_dtype == OM_F32) {
        OM_DISPATCH_PER(N, (balance_bwd_kernel<PER, float><<<nb, 256, 0, st>>>(
                               static_cast<const float *>(logits), prob_grad, token_weight, T, N,
                               static_cast<float *>(dlogits))));
    } else {
        OM_DISPATCH_PER(N, (balance_bwd_kernel<PER, uint16_t><<<nb, 256, 0, st>>>(
                               static_cast<const uint16_t *>(logits), prob_grad, token_weight, T, N,
                               static_cast<uint16_t *>(dlogits))));
    }
    return om_launch_status();
}

extern "C" int om_router_balance_loss(const void *logits, int logits_dtype, int64_t T, int N, int K, double scale, float *count, float *loss,
                                      void *workspace, int64_t workspace_bytes, void *stream) {
    if (logits_dtype != OM_F32 && logits_dtype != OM_BF16) return OM_ERR_DTYPE;
    if (T < 1 || N < 1 || N > 512 || K < 1 || K > N || K > 64 || T > 0x7fffffffLL) return OM_ERR_SHAPE;
    if (!logits || !count || !loss || !workspace) return OM_ERR_NULL;
    if (workspace_bytes < om_router_balance_workspace_bytes(T, N)) return OM_ERR_WORKSPACE;
    hipStream_t st = om_stream(stream);
    const BalancePartials p = balance_partials(logits, logits_dtype, nullptr, T, N, K, workspace, st);
    balance_loss_kernel<<<1, BAL_WAVES * 64, 0, st>>>(p.prob, p.count, p.blocks, T, N, static_cast<float>(scale), count, loss);
    return om_launch_status();
}

extern "C" int om_router_balance_loss_bwd(const void *logits, int logits_dtype, const float *count, const float *loss_grad, double scale,
                                          int64_t T, int N, void *dlogits, void *stream) {
    if (logits_dtype != OM_F32 && logits_dtype != OM_BF16) return OM_ERR_DTYPE;
    if (T < 1 || N < 1 || N > 512 || T > 0x7fffffffLL) return OM_ERR_SHAPE;
    if (!logits || !count || !loss_grad || !dlogits) return OM_ERR_NULL;
    hipStream_t st = om_stream(stream);
    const float s = static_cast<float>(scale);
    if (logits_dtype == OM_F32) {
        OM_DISPATCH_PER(N, (balance_bwd_kernel<PER, float, true><<<token_blocks(T), 256, 0, st>>>(
                               static_cast<const float *>(logits), count, nullptr, T, N, static_cast<float *>(dlogits), loss_grad, s)));
    } else {
        OM_DISPATCH_PER(N, (balance_bwd_kernel<PER, uint16_t, true><<<token_blocks(T), 256, 0, st>>>(
                               static_cast<const uint16_t *>(logits), count, nullptr, T, N, static_cast<uint16_t *>(dlogits), loss_grad, s)));
    }
    return om_launch_status();
}

extern "C" int om_router_balance_bwd(const void *logits, int logits_dtype, const float *prob_grad,
                                     int64_t T, int N, void *dlogits, void *stream) {
    return om_router_balance_bwd_masked(logits, logits_dtype, prob_grad, nullptr, T, N, dlogits, stream);
}

// Flat-buffer mixed-precision AdamW: one coalesced, vectorised pass (HBM-bound).
// Algorithmic traffic per element: read grad 2 + master 4 + m 4 + v 4, write master 4 + m 4 +
// v 4 + param 2 = 28 bytes (bf16 mode).  Each fp32 operation is rounded on its own (no FMA
// contraction) so the result is reproducible bit for bit by a scalar CPU loop.
#include "common.h"
#include <type_traits>

namespace {

struct AdamScalars {
    float b1, b2, omb1, omb2, bc1, bc2, eps, neg_lr, neg_lr_wd;
    int use_wd;
};

#pragma clang fp contract(off)
__device__ __forceinline__ void adam_update(float g, float &m, float &v, float &w,
                                            const AdamScalars &s) {
    float mm = m * s.b1;
    mm = mm + s.omb1 * g;
    float vv = v * s.b2;
    vv = vv + (s.omb2 * g) * g;
    float mh = mm / s.bc1;
    float vh = vv / s.bc2;
    float d = sqrtf(vh) + s.eps;
    float ww = w + s.neg_lr * (mh / d);
    if (s.use_wd) ww = ww + s.neg_lr_wd * ww;
    m = mm; v = vv; w = ww;
}

// Streaming policy (both modes), from measurements at 6.9e9 elements on MI355X (same box, same run):
//   * one wavefront per block and one 16-byte vector per lane and stream: 64-thread blocks that own
//     1 KB of every fp32 stream reach 76 % of 8 TB/s where 256-thread blocks owning 16 KB reach 69 %
//     (a pure write stream: 87 % with 4 KB per block, 75 % with 16 KB; grid-stride and span-per-block
//     persistent grids: 65-66 %);
//   * nontemporal loads AND stores: each buffer is touched once per step and is far larger than any
//     cache; either hint alone gains nothing, both together 5-8 %.  Stores that do not stay in the L2s either
//     (store_past_caches), whole steps of 2.3e9 bf16 parameters: 11.33 -> 11.12 ms; with them ordinary loads 11.66.
//   * at most 12 such wavefronts resident per CU: with the 32 that fit by registers the same kernel
//     reaches 76.5 %, with 20 / 16 / 14 / 12 / 11 / 10: 79.2 / 79.8 / 81.0 / 82.0 / 81.8 / 79.6 % (fewer
//     requests queued at the memory controllers at once); with the stores as they are now, 2.3e9 parameters, ms: all
//     11.91, 20 / 16 / 14 / 12 / 11 / 10 11.50 / 11.46 / 11.24 / 11.25 / 11.18 / 11.32, two runs apart by 0.1.  The launch asks for an LDS allocation it
//     never touches, sized so that 12 blocks fill a CU's 160 KB; nothing else in HIP bounds the
//     number of resident blocks.
// Every wavefront access is one contiguous span (512 B of the bf16 streams, 1 KB of the fp32 ones).
constexpr int ADAMW_THREADS = 64;
constexpr size_t ADAMW_OCCUPANCY_LDS = 13600;   // bytes of dynamic LDS per block: 12 blocks per CU
// More elements than this are stored past the caches: their 128 MB of states are several times what the L2s hold (32 MB), and what lies there
// does not serve the next step.  us, through them (nt alone) -> past them, steps in a row / caches filled by others: bf16, 1.3e6 6.9 -> 8.8
// / 11.1 -> 11.2, 3e6 15.8 -> 17.5 / 20.8 -> 20.4, 6e6 29.0 -> 29.6 / 33.0 -> 32.0, 1e7 48.7 -> 48.5 / 52.8 -> 51.3, 2e7 91.7 -> 90.1 / 94.7 ->
// 92.7; float32 6.4 -> 9.3 / 11.7 -> 11.7, 15.9 -> 18.2 / 20.4 -> 20.6, 30.0 -> 31.2 / 35.2 -> 34.1, 51.3 -> 51.1 / 55.4 -> 53.6, 99.9 -> 96.8 /
// 103.9 -> 99.8.
constexpr int64_t PAST_CACHES = 8 << 20;

template <typename T> __device__ __forceinline__ T stream_load(const T *p) { return __builtin_nontemporal_load(p); }
// vector c of this thread; PAST: see PAST_CACHES
template <bool PAST, typename T, typename P> __device__ __forceinline__ void stream_store(P *p, T v) {
    T *block = reinterpret_cast<T *>(p) + static_cast<int64_t>(blockIdx.x) * ADAMW_THREADS;
    if constexpr (PAST) store_past_caches(block, threadIdx.x * sizeof(T), v);
    else __builtin_nontemporal_store(v, block + threadIdx.x);
}
// Keeps a value that is only copied from being recognised as "the value just loaded from there"
// (the traffic probe writes back what it read and must keep its stores).
__device__ __forceinline__ void opaque(f32x4 &v) { asm volatile("" : "+v"(v)); }

// Elements past the last full vector of 4 (at most 3), taken by the lane that would own that vector.
__device__ __forceinline__ void adam_tail(uint16_t *param, const uint16_t *grad, uint16_t *grad_store, float coef, bool clip,
                                          float *master, float *exp_avg, float *exp_avg_sq, int64_t start, int64_t n,
                                          const AdamScalars &s) {
    for (int64_t i = start; i < n; i++) {
        float m = exp_avg[i], v = exp_avg_sq[i], w = master[i];
        float g = bf16_bits_to_f32(grad[i]);
        if (clip) {
            const uint16_t gb = f32_to_bf16_bits(g * coef);
            g = bf16_bits_to_f32(gb);
            if (grad_store) grad_store[i] = gb;
        }
        adam_update(g, m, v, w, s);
        exp_avg[i] = m; exp_avg_sq[i] = v; master[i] = w;
        param[i] = f32_to_bf16_bits(w);
    }
}
__device__ __forceinline__ void adam_tail(float *master, const float *grad, float *grad_store, float coef, bool clip,
                                          float *exp_avg, float *exp_avg_sq, int64_t start, int64_t n,
                                          const AdamScalars &s) {
    for (int64_t i = start; i < n; i++) {
        float m = exp_avg[i], v = exp_avg_sq[i], w = master[i];
        float g = grad[i];
        if (clip) {
            g = g * coef;
            if (grad_store) grad_store[i] = g;
        }
        adam_update(g, m, v, w, s);
        exp_avg[i] = m; exp_avg_sq[i] = v; master[i] = w;
    }
}

// Whether the scaled gradients of this wavefront are other bits than those that it read.  Where they are not (a norm within the limit:
// the coefficient is 1; experts that no token reached: zeros) they need not be written: 2 of 30 bytes an element in bf16, 4 of 32 in
// float32, of a pass bound by bytes.  A whole wavefront's or none, since parts of lines are slower to write than lines; and behind the
// other stores: ahead of them the branch held those back, and scaled gradients took 10435 -> 10579 us.  2.3e9 elements, us, always
// written -> where changed: coefficient 1, bf16 10430 -> 9567, float32 11063 -> 9537; 0.75, 10420 -> 10425 and 11048 -> 11088
// (runs 70 apart); 4e8 elements, coefficient 1, 1827 -> 1675 and 2004 -> 1723.
template <typename V> __device__ __forceinline__ bool changed(const V &scaled, const V &read) {
    uint32_t differ = 0;
#pragma unroll
    for (unsigned i = 0; i < sizeof(V) / 4; i++) differ |= scaled[i] ^ read[i];
    return __ballot(differ != 0) != 0;
}

// CLIP selects what happens to the gradient before the update (reference optimizers.py:136-152,
// torch.nn.utils.clip_grads_with_norm_): 0 = used as is; 1 = multiplied by *grad_scale and rounded
// back to the gradient dtype, as the in-place multiply of the bf16 gradient views does; 2 = the
// same, and the scaled gradient is also stored (then `grad` is null and `grad_rw` is both the
// source and the destination).
// MATH = false is the traffic probe: the same loads and stores with the arithmetic left out (the
// fp32 states are written back as read, param = bf16(master)).
// TAIL: the lane after the last full vector takes the elements behind it (a branch that the large launches
// do without: it costs them 1-2 %).
template <int CLIP, bool MATH, bool TAIL, bool PAST>
__global__ __launch_bounds__(ADAMW_THREADS) void adamw_bf16_kernel(uint16_t *__restrict__ param,
                                                                      const uint16_t *__restrict__ grad,
                                                                      uint16_t *grad_rw,
                                                                      const float *__restrict__ grad_scale,
                                                                      float *__restrict__ master,
                                                                      float *__restrict__ exp_avg,
                                                                      float *__restrict__ exp_avg_sq,
                                                                      int64_t n_vec4, int64_t n, AdamScalars s) {
    const int64_t c = static_cast<int64_t>(blockIdx.x) * ADAMW_THREADS + threadIdx.x;
    const uint16_t *gsrc = CLIP == 2 ? grad_rw : grad;
    float coef = 1.0f;
    if (CLIP) coef = *grad_scale;
    if (c >= n_vec4) {
        if (TAIL && c == n_vec4)
            adam_tail(param, gsrc, CLIP == 2 ? grad_rw : nullptr, coef, CLIP != 0, master, exp_avg, exp_avg_sq, c * 4, n, s);
        return;
    }
    const u32x2 gq = stream_load(reinterpret_cast<const u32x2 *>(gsrc) + c);
    f32x4 m0 = stream_load(reinterpret_cast<const f32x4 *>(exp_avg) + c);
    f32x4 v0 = stream_load(reinterpret_cast<const f32x4 *>(exp_avg_sq) + c);
    f32x4 w0 = stream_load(reinterpret_cast<const f32x4 *>(master) + c);
    float g[4];
    g[0] = __uint_as_float(gq[0] << 16);
    g[1] = __uint_as_float(gq[0] & 0xffff0000u);
    g[2] = __uint_as_float(gq[1] << 16);
    g[3] = __uint_as_float(gq[1] & 0xffff0000u);
    u32x2 gs = gq;
    if (CLIP) {
        uint16_t gb[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            gb[i] = f32_to_bf16_bits(g[i] * coef);
            g[i] = bf16_bits_to_f32(gb[i]);
        }
        if (CLIP == 2) {
            gs[0] = static_cast<uint32_t>(gb[0]) | (static_cast<uint32_t>(gb[1]) << 16);
            gs[1] = static_cast<uint32_t>(gb[2]) | (static_cast<uint32_t>(gb[3]) << 16);
        }
    }
    if (MATH) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float ma = m0[i], va = v0[i], wa = w0[i];
            adam_update(g[i], ma, va, wa, s);
            m0[i] = ma; v0[i] = va; w0[i] = wa;
        }
    } else {
        asm volatile("" : : "v"(g[0]), "v"(g[1]), "v"(g[2]), "v"(g[3]));   // the gradient load stays
        opaque(m0); opaque(v0); opaque(w0);
    }
    stream_store<PAST>(exp_avg, m0);
    stream_store<PAST>(exp_avg_sq, v0);
    stream_store<PAST>(master, w0);
    u32x2 pk;
    pk[0] = static_cast<uint32_t>(f32_to_bf16_bits(w0[0])) | (static_cast<uint32_t>(f32_to_bf16_bits(w0[1])) << 16);
    pk[1] = static_cast<uint32_t>(f32_to_bf16_bits(w0[2])) | (static_cast<uint32_t>(f32_to_bf16_bits(w0[3])) << 16);
    stream_store<PAST>(param, pk);
    if (CLIP == 2 && changed(gs, gq)) stream_store<PAST>(grad_rw, gs);
}

// fp32 mode: the parameter buffer is the master buffer (16 B read, 12 B written per element).
template <int CLIP, bool TAIL, bool PAST>
__global__ __launch_bounds__(ADAMW_THREADS) void adamw_f32_kernel(float *__restrict__ master,
                                                                  const float *__restrict__ grad,
                                                                  float *grad_rw,
                                                                  const float *__restrict__ grad_scale,
                                                                  float *__restrict__ exp_avg,
                                                                  float *__restrict__ exp_avg_sq,
                                                                  int64_t n_vec4, int64_t n, AdamScalars s) {
    const int64_t c = static_cast<int64_t>(blockIdx.x) * ADAMW_THREADS + threadIdx.x;
    const float *gsrc = CLIP == 2 ? grad_rw : grad;
    float coef = 1.0f;
    if (CLIP) coef = *grad_scale;
    if (c >= n_vec4) {
        if (TAIL && c == n_vec4)
            adam_tail(master, gsrc, CLIP == 2 ? grad_rw : nullptr, coef, CLIP != 0, exp_avg, exp_avg_sq, c * 4, n, s);
        return;
    }
    f32x4 g = stream_load(reinterpret_cast<const f32x4 *>(gsrc) + c);
    f32x4 m = stream_load(reinterpret_cast<const f32x4 *>(exp_avg) + c);
    f32x4 v = stream_load(reinterpret_cast<const f32x4 *>(exp_avg_sq) + c);
    f32x4 w = stream_load(reinterpret_cast<const f32x4 *>(master) + c);
    const f32x4 as_read = g;
    if (CLIP) {
#pragma unroll
        for (int i = 0; i < 4; i++) g[i] = g[i] * coef;
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        float ma = m[i], va = v[i], wa = w[i];
        adam_update(g[i], ma, va, wa, s);
        m[i] = ma; v[i] = va; w[i] = wa;
    }
    stream_store<PAST>(exp_avg, m);
    stream_store<PAST>(exp_avg_sq, v);
    stream_store<PAST>(master, w);
    if (CLIP == 2 && changed(__builtin_bit_cast(u32x4, g), __builtin_bit_cast(u32x4, as_read))) stream_store<PAST>(grad_rw, g);
}

}  // namespace

// clip: 0 = gradient used as is, 1 = scaled by *grad_scale, 2 = scaled and stored back;
// ADAMW_PROBE = the bf16 kernel's loads and stores without the arithmetic.
constexpr int ADAMW_PROBE = 3;
static int adamw_launch(void *param, void *grad, float *master, float *exp_avg, float *exp_avg_sq,
                        int64_t n, double lr, double beta1, double beta2, double eps,
                        double weight_decay, int64_t step, int param_dtype, const float *grad_scale,
                        int clip, void *stream) {
    if (param_dtype != OM_BF16 && param_dtype != OM_F32) return OM_ERR_DTYPE;
    if (n < 0 || step < 1) return OM_ERR_SHAPE;
    if (n == 0) return OM_OK;
    if (!grad || !master || !exp_avg || !exp_avg_sq) return OM_ERR_NULL;
    if (param_dtype == OM_BF16 && !param) return OM_ERR_NULL;
    if ((clip == 1 || clip == 2) && !grad_scale) return OM_ERR_NULL;
    if (!om_aligned16(grad) || !om_aligned16(master) || !om_aligned16(exp_avg) ||
        !om_aligned16(exp_avg_sq) || (param_dtype == OM_BF16 && !om_aligned16(param)))
        return OM_ERR_ALIGN;
    // One launch gives every lane one 4-element vector and the runtime takes fewer than 2^32 threads
    // per launch, so buffers beyond 2^33 elements are updated in consecutive launches over
    // sub-ranges (the update is element-wise: the same bits as one pass).
    constexpr int64_t MAX_PER_LAUNCH = 1LL << 33;
    if (n > MAX_PER_LAUNCH) {
        const int64_t esz = param_dtype == OM_BF16 ? 2 : 4;
        for (int64_t lo = 0; lo < n; lo += MAX_PER_LAUNCH) {
            const int64_t len = n - lo < MAX_PER_LAUNCH ? n - lo : MAX_PER_LAUNCH;
            const int rc = adamw_launch(param ? static_cast<char *>(param) + lo * esz : nullptr,
                                        static_cast<char *>(grad) + lo * esz, master + lo, exp_avg + lo,
                                        exp_avg_sq + lo, len, lr, beta1, beta2, eps, weight_decay, step,
                                        param_dtype, grad_scale, clip, stream);
            if (rc != OM_OK) return rc;
        }
        return OM_OK;
    }

    // Scalars exactly as the reference forms them: Python doubles, narrowed to fp32 where they
    // meet an fp32 tensor (optimizers.py:193-202).
    AdamScalars s;
    s.b1 = static_cast<float>(beta1);
    s.b2 = static_cast<float>(beta2);
    s.omb1 = static_cast<float>(1.0 - beta1);
    s.omb2 = static_cast<float>(1.0 - beta2);
    s.bc1 = static_cast<float>(1.0 - pow(beta1, static_cast<double>(step)));
    s.bc2 = static_cast<float>(1.0 - pow(beta2, static_cast<double>(step)));
    s.eps = static_cast<float>(eps);
    s.neg_lr = static_cast<float>(-lr);
    s.neg_lr_wd = static_cast<float>(-lr * weight_decay);
    s.use_wd = weight_decay > 0.0 ? 1 : 0;

    hipStream_t st = om_stream(stream);
    const int64_t n_vec = n / 4;
    // A launch that fits the chip at full occupancy (32 wavefronts on each of 256 CUs) is over in one wave of
    // blocks and bound by latency, not by the queues that the residency bound keeps short, and takes its tail
    // along: 1.3e6 float32 elements 9.5 + 3 us as two bounded launches, 7 as one.  A larger one leaves the
    // tail to a second launch over the last few elements.
    constexpr int64_t SMALL_BLOCKS = 256 * 32;
    const int64_t tail = n - n_vec * 4;
    const bool small = (n_vec + ADAMW_THREADS) / ADAMW_THREADS <= SMALL_BLOCKS;
    const bool with_tail = small && tail > 0;
    const int64_t lanes = n_vec + (with_tail ? 1 : 0), blocks = (lanes + ADAMW_THREADS - 1) / ADAMW_THREADS;
    if (blocks * ADAMW_THREADS >= (1LL << 32)) return OM_ERR_SHAPE;   // (not reached: see MAX_PER_LAUNCH)
    const size_t lds = small ? 0 : ADAMW_OCCUPANCY_LDS;
    const dim3 block(ADAMW_THREADS);
    // `lo`: first element, `vecs` full vectors and (TAIL) the elements up to `count`
    auto go = [&](auto tail_tag, auto past_tag, unsigned grid, int64_t lo, int64_t vecs, int64_t count) {
        constexpr bool TAIL = decltype(tail_tag)::value, PAST = decltype(past_tag)::value;
        float *w = master + lo, *m = exp_avg + lo, *v = exp_avg_sq + lo;
        if (param_dtype == OM_BF16) {
            uint16_t *p = static_cast<uint16_t *>(param) + lo, *g = static_cast<uint16_t *>(grad) + lo;
            if (clip == ADAMW_PROBE) adamw_bf16_kernel<0, false, false, PAST><<<grid, block, lds, st>>>(p, g, nullptr, nullptr, w, m, v, vecs, count, s);
            else if (clip == 0) adamw_bf16_kernel<0, true, TAIL, PAST><<<grid, block, lds, st>>>(p, g, nullptr, nullptr, w, m, v, vecs, count, s);
            else if (clip == 1) adamw_bf16_kernel<1, true, TAIL, PAST><<<grid, block, lds, st>>>(p, g, nullptr, grad_scale, w, m, v, vecs, count, s);
            else adamw_bf16_kernel<2, true, TAIL, PAST><<<grid, block, lds, st>>>(p, nullptr, g, grad_scale, w, m, v, vecs, count, s);
        } else {
            float *g = static_cast<float *>(grad) + lo;
            if (clip == 0) adamw_f32_kernel<0, TAIL, PAST><<<grid, block, lds, st>>>(w, g, nullptr, nullptr, m, v, vecs, count, s);
            else if (clip == 1) adamw_f32_kernel<1, TAIL, PAST><<<grid, block, lds, st>>>(w, g, nullptr, grad_scale, m, v, vecs, count, s);
            else adamw_f32_kernel<2, TAIL, PAST><<<grid, block, lds, st>>>(w, nullptr, g, grad_scale, m, v, vecs, count, s);
        }
    };
    if (param_dtype == OM_F32 && clip == ADAMW_PROBE) return OM_ERR_DTYPE;
    if (with_tail) {
        go(std::true_type(), std::false_type(), static_cast<unsigned>(blocks), 0, n_vec, n);
    } else {
        if (n_vec > 0 && n > PAST_CACHES) go(std::false_type(), std::true_type(), static_cast<unsigned>(blocks), 0, n_vec, n);
        else if (n_vec > 0) go(std::false_type(), std::false_type(), static_cast<unsigned>(blocks), 0, n_vec, n);
        if (tail > 0 && clip != ADAMW_PROBE) go(std::true_type(), std::false_type(), 1u, n_vec * 4, 0, tail);
    }
    return om_launch_status();
}

extern "C" int om_adamw_step(void *param, const void *grad, float *master, float *exp_avg,
                             float *exp_avg_sq, int64_t n, double lr, double beta1, double beta2,
                             double eps, double weight_decay, int64_t step, int param_dtype,
                             void *stream) {
    return adamw_launch(param, const_cast<void *>(grad), master, exp_avg, exp_avg_sq, n, lr, beta1,
                        beta2, eps, weight_decay, step, param_dtype, nullptr, 0, stream);
}

extern "C" int om_adamw_step_clipped(void *param, void *grad, float *master, float *exp_avg,
                                     float *exp_avg_sq, int64_t n, double lr, double beta1,
                                     double beta2, double eps, double weight_decay, int64_t step,
                                     int param_dtype, const float *grad_scale, int store_scaled_grad,
                                     void *stream) {
    if (!grad_scale) return OM_ERR_NULL;
    return adamw_launch(param, grad, master, exp_avg, exp_avg_sq, n, lr, beta1, beta2, eps,
                        weight_decay, step, param_dtype, grad_scale, store_scaled_grad ? 2 : 1,
                        stream);
}

extern "C" int om_adamw_traffic_probe(void *param, const void *grad, float *master, float *exp_avg,
                                      float *exp_avg_sq, int64_t n, void *stream) {
    return adamw_launch(param, const_cast<void *>(grad), master, exp_avg, exp_avg_sq, n, 0.0, 0.0, 0.0,
                        0.0, 0.0, 1, OM_BF16, nullptr, ADAMW_PROBE, stream);
}

// The router's gate projection for float32 modules (the reference's small CPU-runnable
// configuration keeps the whole block in float32): logits = x W^T of the gate nn.Linear
// (optimus/models/common/moe.py:456, optimus/models/olmoe/modeling_olmoe.py:284) and the two
// products of its backward, in plain float32 arithmetic with sums in a fixed order.  This is the
// parity path at fp32 accuracy (the bf16 gate runs on MFMA, gate_fwd.hip and gate_bwd.hip).
#include "common.h"

namespace {

// logits[t,n] = sum_h x[t,h] W[n,h]: one wavefront per token, lanes over h, the 64 partial sums
// added by a butterfly.
__global__ __launch_bounds__(256) void gate_logits_f32_kernel(const float *__restrict__ x,
                                                              const float *__restrict__ w, int64_t T,
                                                              int H, int N, float *__restrict__ logits) {
    const int lane = threadIdx.x & 63;
    const int64_t t = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (t >= T) return;
    const float *xr = x + t * H;
    for (int n = 0; n < N; n++) {
        const float *wr = w + static_cast<int64_t>(n) * H;
        float s = 0.0f;
        for (int h = lane; h < H; h += 64) s += xr[h] * wr[h];
        s = wave_sum(s);
        if (lane == 0) logits[t * N + n] = s;
    }
}

// dx[t,h] = (base[t,h] +) sum_n dlogits[t,n] W[n,h]: one thread per element, n ascending.
__global__ __launch_bounds__(256) void gate_dgrad_f32_kernel(const float *__restrict__ dlogits,
                                                             const float *__restrict__ w,
                                                             const float *__restrict__ base, int64_t T,
                                                             int H, int N, float *__restrict__ dx) {
    const int h = blockIdx.x * 256 + threadIdx.x;
    const int64_t t = blockIdx.y;
    if (h >= H) return;
    float s = 0.0f;
    for (int n = 0; n < N; n++) s += dlogits[t * N + n] * w[static_cast<int64_t>(n) * H + h];
    dx[t * H + h] = base ? s + base[t * H + h] : s;
}

// dW[n,h] = sum_t dlogits[t,n] x[t,h], the sum kept in double (thousands of terms) and rounded once.  A
// block owns 16 columns of h and 4 experts and spreads the tokens over 64 groups of 16 lanes, whose sums
// are added in a fixed order.  Latency-bound: with one thread per element walking all tokens (8 blocks for
// 2048 x 256 x 8) this took 500 us, more than the rest of the layer's step; 64 groups take 7 us.
constexpr int GW_H = 16, GW_N = 4, GW_WAVES = 16;
__global__ __launch_bounds__(GW_WAVES * 64) void gate_wgrad_f32_kernel(const float *__restrict__ x,
                                                                       const float *__restrict__ dlogits,
                                                                       int64_t T, int H, int N,
                                                                       float *__restrict__ dw) {
    __shared__ double part[GW_WAVES][GW_N][GW_H];
    const int hl = threadIdx.x & (GW_H - 1), group = threadIdx.x / GW_H;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int h = blockIdx.x * GW_H + hl, n0 = blockIdx.y * GW_N;
    double acc[GW_N] = {0.0, 0.0, 0.0, 0.0};
    if (h < H) {
#pragma unroll 4
        for (int64_t t = group; t < T; t += GW_WAVES * 64 / GW_H) {
            const double xv = static_cast<double>(x[t * H + h]);
#pragma unroll
            for (int j = 0; j < GW_N; j++) acc[j] += static_cast<double>(dlogits[t * N + min(n0 + j, N - 1)]) * xv;
        }
    }
#pragma unroll
    for (int j = 0; j < GW_N; j++) {
        // the wavefront's four token groups
        acc[j] += __shfl_xor(acc[j], 16, 64);
        acc[j] += __shfl_xor(acc[j], 32, 64);
        if (lane < GW_H) part[wave][j][hl] = acc[j];
    }
    __syncthreads();
    if (threadIdx.x < GW_N * GW_H) {
        const int j = threadIdx.x / GW_H;
        double s = 0.0;
        for (int w = 0; w < GW_WAVES; w++) s += part[w][j][hl];
        if (h < H && n0 + j < N) dw[static_cast<int64_t>(n0 + j) * H + h] = static_cast<float>(s);
    }
}

inline bool gate_f32_shape_ok(int64_t T, int H, int N) {
    return T >= 0 && T <= 0x7fffffffLL && H >= 1 && N >= 1 && N <= 65535;
}

}  // namespace

extern "C" int om_router_gate_logits_f32(const float *x, const float *gate_weight, int64_t T, int H, int N,
                                         float *logits_out, void *stream) {
    if (!gate_f32_shape_ok(T, H, N)) return OM_ERR_SHAPE;
    if (T == 0) return OM_OK;
    if (!x || !gate_weight || !logits_out) return OM_ERR_NULL;
    gate_logits_f32_kernel<<<static_cast<unsigned>((T + 3) / 4), 256, 0, om_stream(stream)>>>(
        x, gate_weight, T, H, N, logits_out);
    return om_launch_status();
}

extern "C" int om_router_gate_dgrad_f32_add(const float *dlogits, const float *gate_weight, const float *base, int64_t T,
                                            int H, int N, float *dx, void *stream) {
    if (!gate_f32_shape_ok(T, H, N) || T > 65535LL * 32768) return OM_ERR_SHAPE;
    if (T == 0) return OM_OK;
    if (!dlogits || !gate_weight || !dx) return OM_ERR_NULL;
    hipStream_t st = om_stream(stream);
    // the grid's y extent is limited to 65535: tokens go in slabs
    for (int64_t t0 = 0; t0 < T; t0 += 65535) {
        const int64_t nt = T - t0 < 65535 ? T - t0 : 65535;
        gate_dgrad_f32_kernel<<<dim3((H + 255) / 256, static_cast<unsigned>(nt)), 256, 0, st>>>(
            dlogits + t0 * N, gate_weight, base ? base + t0 * H : nullptr, nt, H, N, dx + t0 * H);
    }
    return om_launch_status();
}

extern "C" int om_router_gate_dgrad_f32(const float *dlogits, const float *gate_weight, int64_t T, int H,
                                        int N, float *dx, void *stream) {
    return om_router_gate_dgrad_f32_add(dlogits, gate_weight, nullptr, T, H, N, dx, stream);
}

extern "C" int om_router_gate_wgrad_f32(const float *x, const float *dlogits, int64_t T, int H, int N,
                                        float *dweight, void *stream) {
    if (!gate_f32_shape_ok(T, H, N)) return OM_ERR_SHAPE;
    if (!dweight) return OM_ERR_NULL;
    if (T > 0 && (!x || !dlogits)) return OM_ERR_NULL;
    gate_wgrad_f32_kernel<<<dim3((H + GW_H - 1) / GW_H, (N + GW_N - 1) / GW_N), GW_WAVES * 64, 0, om_stream(stream)>>>(
        x, dlogits, T, H, N, dweight);
    return om_launch_status();
}

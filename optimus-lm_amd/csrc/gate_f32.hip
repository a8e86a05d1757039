// The router's gate projection for float32 modules (the reference's small CPU-runnable
// configuration keeps the whole block in float32): the two products of the backward of
// logits = x W^T of the gate nn.Linear (optimus/models/common/moe.py:456,
// optimus/models/olmoe/modeling_olmoe.py:284; the projection is in route.hip, where the routing follows in the same
// launch), in plain float32 arithmetic with sums in a fixed order.  This is the
// parity path at fp32 accuracy (the bf16 gate runs on MFMA, gate_fwd.hip and gate_bwd.hip).
#include "common.h"

namespace {

// dx[t,h] = (base[t,h] +) sum_n dlogits[t,n] W[n,h]: one thread per element, n ascending.
__device__ __forceinline__ void gate_dgrad_f32_element(const float *__restrict__ dlogits, const float *__restrict__ w,
                                                       const float *__restrict__ base, int64_t t, int H, int N, int h,
                                                       float *__restrict__ dx) {
    float s = 0.0f;
    for (int n = 0; n < N; n++) s += dlogits[t * N + n] * w[static_cast<int64_t>(n) * H + h];
    dx[t * H + h] = base ? s + base[t * H + h] : s;
}
__global__ __launch_bounds__(256) void gate_dgrad_f32_kernel(const float *__restrict__ dlogits,
                                                             const float *__restrict__ w,
                                                             const float *__restrict__ base, int64_t T,
                                                             int H, int N, float *__restrict__ dx) {
    const int h = blockIdx.x * 256 + threadIdx.x;
    if (h < H) gate_dgrad_f32_element(dlogits, w, base, blockIdx.y, H, N, h, dx);
}

// dW[n,h] = sum_t dlogits[t,n] x[t,h], the sum kept in double (thousands of terms) and rounded once.  A
// block owns 16 columns of h and 4 experts and spreads the tokens over 64 groups of 16 lanes, whose sums
// are added in a fixed order.  Latency-bound: with one thread per element walking all tokens (8 blocks for
// 2048 x 256 x 8) this took 500 us, more than the rest of the layer's step; with 64 groups what counts is how many of a
// thread's tokens are under way at once: four 13.3 us, eight, with the input gradient in the same launch (5.4 alone), 10.5, sixteen 11.3.
constexpr int GW_H = 16, GW_N = 4, GW_WAVES = 16, GW_AHEAD = 8;
typedef double GwPart[GW_WAVES][GW_N][GW_H];
__device__ __forceinline__ void gate_wgrad_f32_block(const float *__restrict__ x, const float *__restrict__ dlogits, int64_t T, int H, int N,
                                                     int slice, int experts, float *__restrict__ dw, GwPart &part) {
    constexpr int GROUPS = GW_WAVES * 64 / GW_H;
    const int hl = threadIdx.x & (GW_H - 1), group = threadIdx.x / GW_H;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int h = slice * GW_H + hl, n0 = experts * GW_N, hc = min(h, H - 1);
    double acc[GW_N] = {0.0, 0.0, 0.0, 0.0};
    for (int64_t t0 = group; t0 < T; t0 += GW_AHEAD * GROUPS) {
        float xv[GW_AHEAD], d[GW_AHEAD][GW_N];
#pragma unroll
        for (int u = 0; u < GW_AHEAD; u++) {             // past the last token: it again, not added
            const int64_t t = min(t0 + u * GROUPS, T - 1);
            xv[u] = x[t * H + hc];
#pragma unroll
            for (int j = 0; j < GW_N; j++) d[u][j] = dlogits[t * N + min(n0 + j, N - 1)];
        }
#pragma unroll
        for (int u = 0; u < GW_AHEAD; u++)
            if (t0 + u * GROUPS < T)
#pragma unroll
                for (int j = 0; j < GW_N; j++) acc[j] += static_cast<double>(d[u][j]) * static_cast<double>(xv[u]);
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
__global__ __launch_bounds__(GW_WAVES * 64) void gate_wgrad_f32_kernel(const float *__restrict__ x, const float *__restrict__ dlogits, int64_t T,
                                                                       int H, int N, float *__restrict__ dw) {
    __shared__ GwPart part;
    gate_wgrad_f32_block(x, dlogits, T, H, N, blockIdx.x, blockIdx.y, dw, part);
}
// Both, independent of each other: the first `wgrad_blocks` blocks are those of the weight gradient, the others have 1024 elements of a
// 256-column slice of dx each.
__global__ __launch_bounds__(GW_WAVES * 64) void gate_bwd_f32_kernel(const float *__restrict__ x, const float *__restrict__ dlogits,
                                                                     const float *__restrict__ w, const float *__restrict__ base, int64_t T,
                                                                     int H, int N, float *__restrict__ dx, float *__restrict__ dw,
                                                                     int wgrad_blocks) {
    __shared__ GwPart part;
    const int slices = (H + GW_H - 1) / GW_H, wide = (H + 255) / 256, id = static_cast<int>(blockIdx.x) - wgrad_blocks;
    if (id < 0) {
        gate_wgrad_f32_block(x, dlogits, T, H, N, blockIdx.x % slices, blockIdx.x / slices, dw, part);
        return;
    }
    const int h = id % wide * 256 + (threadIdx.x & 255);
    const int64_t t = static_cast<int64_t>(id / wide) * 4 + (threadIdx.x >> 8);
    if (h < H && t < T) gate_dgrad_f32_element(dlogits, w, base, t, H, N, h, dx);
}

inline bool gate_f32_shape_ok(int64_t T, int H, int N) {
    return T >= 0 && T <= 0x7fffffffLL && H >= 1 && N >= 1 && N <= 65535;
}

}  // namespace

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

extern "C" int om_router_gate_bwd_f32(const float *x, const float *dlogits, const float *gate_weight, const float *base, int64_t T, int H,
                                      int N, float *dx, float *dweight, void *stream) {
    if (!gate_f32_shape_ok(T, H, N) || T < 1) return OM_ERR_SHAPE;
    if (!x || !dlogits || !gate_weight || !dx || !dweight) return OM_ERR_NULL;
    const int64_t wgrad_blocks = static_cast<int64_t>((H + GW_H - 1) / GW_H) * ((N + GW_N - 1) / GW_N);
    const int64_t blocks = wgrad_blocks + (H + 255) / 256 * ((T + 3) / 4);
    if (blocks * (GW_WAVES * 64) > 0xffffffffLL) {   // (a launch of more threads runs a part of them, without an error)
        const int code = om_router_gate_wgrad_f32(x, dlogits, T, H, N, dweight, stream);
        return code == OM_OK ? om_router_gate_dgrad_f32_add(dlogits, gate_weight, base, T, H, N, dx, stream) : code;
    }
    gate_bwd_f32_kernel<<<static_cast<unsigned>(blocks), GW_WAVES * 64, 0, om_stream(stream)>>>(x, dlogits, gate_weight, base, T, H, N, dx,
                                                                                              dweight, static_cast<int>(wgrad_blocks));
    return om_launch_status();
}

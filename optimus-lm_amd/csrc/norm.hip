// RMSNorm of the decoder layer, optionally fused with the residual add that precedes it
// (reference optimus/models/olmoe/modeling_olmoe.py:93-104 and the layer body :402-409;
// optimus/models/deepseek_v3/modeling_deepseek_v3.py:29-41 is the same expression):
//     h  = x (+ residual)                      rounded to the model dtype, as the tensor add is
//     v  = mean(float(h)^2);  r = rsqrt(v + eps)
//     y  = weight * cast(float(h) * r)         two roundings in bf16: the normalised value, then
//                                              the product with the bf16 weight
// One wavefront per row, 16-byte accesses, HBM-bound.  Backward: per row
//     dxn = dy * weight;  dx = r * (dxn - xn * mean(dxn * xn)),  xn = float(h) * r
// in fp32 (one wavefront per row), and the weight gradient sum_rows dy * cast(xn) column-wise in
// chunks of rows whose partial sums a last kernel adds in a fixed order (deterministic).
// Rows of up to 64 * 16 * ROW_VECS bytes stay in registers: each operand is read once, forward and backward
// (rmsnorm_fwd_row_kernel, rmsnorm_bwd_rows_kernel); longer ones are read again from the caches.
#include "common.h"
#include <algorithm>
#include <type_traits>

namespace {

#pragma clang fp contract(off)

constexpr int DW_ROWS = 128;     // rows of a chunk of the weight gradient, at most
constexpr int NORM_ROWS = 4;     // rows (wavefronts) per block
constexpr int ROW_VECS = 4;      // 16-byte vectors a lane keeps per pass: 4 KB of a row per pass

template <typename T> __device__ __forceinline__ float round_like(float x);
template <> __device__ __forceinline__ float round_like<float>(float x) { return x; }
template <> __device__ __forceinline__ float round_like<uint16_t>(float x) {
    return bf16_bits_to_f32(f32_to_bf16_bits(x));
}

// This many elements and more are loaded past the caches: 16 MB and more of each operand, most of which is used here for the last time for a
// while, do not push out of the caches what other kernels wrote, which would have to be written back first.  16384 rows of
// 2048 bf16 with a residual, us, ordinary loads -> past the caches: caches full of written data (a pass) 76 -> 52, operands in the caches
// 42 -> 44; 4096 rows 24 -> 18 and 13.1 -> 14.6; 512 rows 8.3 -> 8.0 and 4.9 -> 5.3.
constexpr int64_t NORM_PAST_CACHES = 8 << 20;
template <bool PAST> __device__ __forceinline__ u32x4 norm_load(const u32x4 *p) { return PAST ? __builtin_nontemporal_load(p) : *p; }

// Rows that a wavefront holds, VECS 16-byte vectors a lane; one wavefront per block.  All loads, the weight's too, are on their way
// before the first is used (lanes past the end re-read the last vector).
template <typename T, int VECS, bool PAST>
__global__ __launch_bounds__(64) void rmsnorm_fwd_row_kernel(const T *__restrict__ x, const T *__restrict__ residual,
                                                             const T *__restrict__ weight, float eps, T *__restrict__ out,
                                                             T *__restrict__ h_out, float *__restrict__ rstd_out, int64_t E) {
    constexpr int V = Elem<T>::VEC;
    const int lane = threadIdx.x, nv = static_cast<int>(E / V);
    const int64_t at = static_cast<int64_t>(blockIdx.x) * E;
    u32x4 q[VECS], w[VECS];
#pragma unroll
    for (int u = 0; u < VECS; u++) q[u] = norm_load<PAST>(reinterpret_cast<const u32x4 *>(x + at) + min(u * 64 + lane, nv - 1));
    if (residual) {
        u32x4 b[VECS];
#pragma unroll
        for (int u = 0; u < VECS; u++) b[u] = norm_load<PAST>(reinterpret_cast<const u32x4 *>(residual + at) + min(u * 64 + lane, nv - 1));
#pragma unroll
        for (int u = 0; u < VECS; u++) w[u] = reinterpret_cast<const u32x4 *>(weight)[min(u * 64 + lane, nv - 1)];
#pragma unroll
        for (int u = 0; u < VECS; u++) {
            float s[V], t[V];
            Elem<T>::unpack(q[u], s);
            Elem<T>::unpack(b[u], t);
#pragma unroll
            for (int j = 0; j < V; j++) s[j] = s[j] + t[j];
            q[u] = Elem<T>::pack(s);        // the sum as the model dtype holds it
        }
    } else {
#pragma unroll
        for (int u = 0; u < VECS; u++) w[u] = reinterpret_cast<const u32x4 *>(weight)[min(u * 64 + lane, nv - 1)];
    }
    float ss = 0.0f;
#pragma unroll
    for (int u = 0; u < VECS; u++) {
        const int c = u * 64 + lane;
        if (c < nv) {
            if (h_out) reinterpret_cast<u32x4 *>(h_out + at)[c] = q[u];
            float f[V];
            Elem<T>::unpack(q[u], f);
#pragma unroll
            for (int j = 0; j < V; j++) ss += f[j] * f[j];
        }
    }
    ss = wave_sum(ss);
    const float r = 1.0f / sqrtf(ss / static_cast<float>(E) + eps);
    if (lane == 0 && rstd_out) rstd_out[blockIdx.x] = r;
#pragma unroll
    for (int u = 0; u < VECS; u++) {
        const int c = u * 64 + lane;
        float f[V], wf[V], y[V];
        Elem<T>::unpack(q[u], f);
        Elem<T>::unpack(w[u], wf);
#pragma unroll
        for (int j = 0; j < V; j++) y[j] = wf[j] * round_like<T>(f[j] * r);
        if (c < nv) reinterpret_cast<u32x4 *>(out + at)[c] = Elem<T>::pack(y);
    }
}

// o = o as the dtype holds it + the 16 bytes of b: what the add of the two tensors gives
template <typename T> __device__ __forceinline__ void add_rounded(const u32x4 &b, float (&o)[Elem<T>::VEC]) {
    float t[Elem<T>::VEC];
    Elem<T>::unpack(b, t);
#pragma unroll
    for (int j = 0; j < Elem<T>::VEC; j++) o[j] = round_like<T>(o[j]) + t[j];
}

// Longer rows.  PAST: with h_out, which the second pass reads.
template <typename T, bool PAST>
__global__ __launch_bounds__(256) void rmsnorm_fwd_kernel(const T *__restrict__ x,
                                                          const T *__restrict__ residual,
                                                          const T *__restrict__ weight, float eps,
                                                          T *__restrict__ out, T *__restrict__ h_out,
                                                          float *__restrict__ rstd_out, int64_t rows,
                                                          int64_t E) {
    constexpr int V = Elem<T>::VEC;
    const int lane = threadIdx.x & 63;
    const int64_t row = static_cast<int64_t>(blockIdx.x) * NORM_ROWS + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int64_t nv = E / V;
    const u32x4 *xr = reinterpret_cast<const u32x4 *>(x + row * E);
    const u32x4 *rr = residual ? reinterpret_cast<const u32x4 *>(residual + row * E) : nullptr;
    u32x4 *hr = h_out ? reinterpret_cast<u32x4 *>(h_out + row * E) : nullptr;
    // pass 1: h = x + residual, sum of squares
    float ss = 0.0f;
    for (int64_t c0 = 0; c0 < nv; c0 += 64 * ROW_VECS) {
        // both operands of the whole pass first (lanes past the end re-read the last vector): a load
        // behind a condition is waited for before the next one starts
        u32x4 q[ROW_VECS], b[ROW_VECS];
#pragma unroll
        for (int u = 0; u < ROW_VECS; u++) q[u] = norm_load<PAST>(xr + min(c0 + u * 64 + lane, nv - 1));
        if (rr) {
#pragma unroll
            for (int u = 0; u < ROW_VECS; u++) b[u] = norm_load<PAST>(rr + min(c0 + u * 64 + lane, nv - 1));
#pragma unroll
            for (int u = 0; u < ROW_VECS; u++) {
                float s[V], t[V];
                Elem<T>::unpack(q[u], s);
                Elem<T>::unpack(b[u], t);
#pragma unroll
                for (int j = 0; j < V; j++) s[j] = s[j] + t[j];
                q[u] = Elem<T>::pack(s);        // the sum as the model dtype holds it
            }
        }
#pragma unroll
        for (int u = 0; u < ROW_VECS; u++) {
            const int64_t c = c0 + u * 64 + lane;
            if (c < nv) {
                if (hr) hr[c] = q[u];
                float f[V];
                Elem<T>::unpack(q[u], f);
#pragma unroll
                for (int j = 0; j < V; j++) ss += f[j] * f[j];
            }
        }
    }
    ss = wave_sum(ss);
    const float r = 1.0f / sqrtf(ss / static_cast<float>(E) + eps);
    if (lane == 0 && rstd_out) rstd_out[row] = r;
    // pass 2: y = weight * cast(h * r)
    const u32x4 *wr = reinterpret_cast<const u32x4 *>(weight);
    u32x4 *orow = reinterpret_cast<u32x4 *>(out + row * E);
    for (int64_t c0 = 0; c0 < nv; c0 += 64 * ROW_VECS) {
#pragma unroll
        for (int u = 0; u < ROW_VECS; u++) {
            const int64_t c = c0 + u * 64 + lane;
            if (c < nv) {
                u32x4 q;
                if (hr) q = hr[c];
                else {
                    q = xr[c];
                    if (rr) {
                        float a[V], b[V];
                        Elem<T>::unpack(q, a);
                        Elem<T>::unpack(rr[c], b);
#pragma unroll
                        for (int j = 0; j < V; j++) a[j] = a[j] + b[j];
                        q = Elem<T>::pack(a);
                    }
                }
                float f[V], w[V], y[V];
                Elem<T>::unpack(q, f);
                Elem<T>::unpack(wr[c], w);
#pragma unroll
                for (int j = 0; j < V; j++) y[j] = w[j] * round_like<T>(f[j] * r);
                orow[c] = Elem<T>::pack(y);
            }
        }
    }
}

// dx and the partial weight gradient of `chunk` rows, of rows that a wavefront holds: wavefront w of the block's four takes rows
// w, w + 4, ... and keeps the columns' sums in registers, so both operands are read once (by a kernel for each they were read
// twice).  The next row is on its way under this one.  chunk: as many as make 512 blocks, two on a CU, and no more than DW_ROWS.
// Whole backward, us, a kernel for dx, one for dw and a reduction of one wavefront a column -> this and one of four, caches full of written
// data / operands in the caches: 16384 rows of 2048 bf16 90 -> 63 / 59 -> 46, 4096 40 -> 27 / 32 -> 21, 512 29 -> 11.6 / 18.7 -> 8; 16384 of
// 512 40 -> 22 / 33 -> 17; 2048 of 256 26 -> 11 / 17 -> 8; 4096 of 1024 float32 35 -> 24 / 26 -> 15.  (128-row chunks: 512 rows 68.)
template <typename T, int VECS, bool PAST>
__global__ __launch_bounds__(256) void rmsnorm_bwd_rows_kernel(const T *__restrict__ dy, const T *__restrict__ h,
                                                               const T *__restrict__ weight, const float *__restrict__ rstd,
                                                               const T *__restrict__ h_grad, T *__restrict__ dx,
                                                               float *__restrict__ dw_part, int64_t rows, int64_t E, int chunk) {
    constexpr int V = Elem<T>::VEC;
    __shared__ __attribute__((aligned(16))) float lds_dw[4][64 * VECS * V];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nv = static_cast<int>(E / V);
    const int64_t begin = static_cast<int64_t>(blockIdx.x) * chunk, end = min(begin + chunk, rows);
    const u32x4 *dyv = reinterpret_cast<const u32x4 *>(dy), *hv = reinterpret_cast<const u32x4 *>(h);
    u32x4 w[VECS], g_next[VECS], h_next[VECS];
    float r_next = 0.0f, dw[VECS][V];
    auto fetch = [&](int64_t row) {
        const int64_t at = min(row, rows - 1) * nv;
        r_next = rstd[min(row, rows - 1)];
#pragma unroll
        for (int u = 0; u < VECS; u++) {
            g_next[u] = dyv[at + min(u * 64 + lane, nv - 1)];
            h_next[u] = norm_load<PAST>(hv + at + min(u * 64 + lane, nv - 1));
        }
    };
    fetch(begin + wave);
#pragma unroll
    for (int u = 0; u < VECS; u++) {
        w[u] = reinterpret_cast<const u32x4 *>(weight)[min(u * 64 + lane, nv - 1)];
#pragma unroll
        for (int j = 0; j < V; j++) dw[u][j] = 0.0f;
    }
    for (int64_t row = begin + wave; row < end; row += 4) {
        float dxn[VECS][V], xn[VECS][V], dot = 0.0f;
        const float r = r_next;
#pragma unroll
        for (int u = 0; u < VECS; u++) {
            float g[V], f[V], wf[V];
            Elem<T>::unpack(g_next[u], g);
            Elem<T>::unpack(h_next[u], f);
            Elem<T>::unpack(w[u], wf);
#pragma unroll
            for (int j = 0; j < V; j++) {
                xn[u][j] = f[j] * r;
                dxn[u][j] = g[j] * wf[j];
                dw[u][j] += g[j] * round_like<T>(xn[u][j]);
            }
            if (u * 64 + lane < nv)
#pragma unroll
                for (int j = 0; j < V; j++) dot += dxn[u][j] * xn[u][j];
        }
        u32x4 add[VECS];
        if (h_grad) {
#pragma unroll
            for (int u = 0; u < VECS; u++) add[u] = norm_load<PAST>(reinterpret_cast<const u32x4 *>(h_grad) + row * nv + min(u * 64 + lane, nv - 1));
        }
        if (row + 4 < end) fetch(row + 4);
        dot = wave_sum(dot) / static_cast<float>(E);
#pragma unroll
        for (int u = 0; u < VECS; u++) {
            const int c = u * 64 + lane;
            float o[V];
#pragma unroll
            for (int j = 0; j < V; j++) o[j] = r * (dxn[u][j] - xn[u][j] * dot);
            if (h_grad) add_rounded<T>(add[u], o);
            if (c < nv) reinterpret_cast<u32x4 *>(dx + row * E)[c] = Elem<T>::pack(o);
        }
    }
#pragma unroll
    for (int u = 0; u < VECS; u++)
#pragma unroll
        for (int j = 0; j < V; j += 4)
            *reinterpret_cast<f32x4 *>(&lds_dw[wave][(u * 64 + lane) * V + j]) = f32x4{dw[u][j], dw[u][j + 1], dw[u][j + 2], dw[u][j + 3]};
    __syncthreads();
    for (int e = threadIdx.x; e < E; e += 256)
        dw_part[blockIdx.x * E + e] = (lds_dw[0][e] + lds_dw[1][e]) + (lds_dw[2][e] + lds_dw[3][e]);
}
inline int64_t bwd_chunk(int64_t rows) { return (rows + 2047) / 2048 * 4; }

// dx of longer rows, and with little workspace, one wavefront per row.  Rows that fit the registers are read once, VECS vectors a lane: the whole
// backward with little workspace, operands in the caches, us, read twice -> so: 16384 rows of 2048 bf16 71 -> 55, 4096 33.0 -> 30.4, 16384 of 512
// 30.4 -> 29.1 (32.6 with registers for the longest row), 4096 of 1024 float32 29.0 -> 25.5.  Longer rows twice (VECS = 0).
template <typename T, int VECS, bool ADD>
__global__ __launch_bounds__(256) void rmsnorm_dx_kernel(const T *__restrict__ dy,
                                                         const T *__restrict__ h,
                                                         const T *__restrict__ weight,
                                                         const float *__restrict__ rstd, const T *__restrict__ h_grad,
                                                         T *__restrict__ dx, int64_t rows, int64_t E) {
    constexpr int V = Elem<T>::VEC, U = VECS ? VECS : ROW_VECS;
    const int lane = threadIdx.x & 63;
    const int64_t row = static_cast<int64_t>(blockIdx.x) * NORM_ROWS + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int64_t nv = E / V;
    const float r = rstd[row];
    const u32x4 *wr = reinterpret_cast<const u32x4 *>(weight);
    const u32x4 *dyr = reinterpret_cast<const u32x4 *>(dy + row * E);
    const u32x4 *hr = reinterpret_cast<const u32x4 *>(h + row * E);
    u32x4 *dxr = reinterpret_cast<u32x4 *>(dx + row * E);
    float dxn[U][V], xn[U][V];   // VECS: of the whole row
    float dot = 0.0f;
    for (int64_t c0 = 0; c0 < nv; c0 += 64 * U) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int64_t c = c0 + u * 64 + lane;
            if (c < nv) {
                float g[V], f[V], w[V];
                Elem<T>::unpack(dyr[c], g);
                Elem<T>::unpack(hr[c], f);
                Elem<T>::unpack(wr[c], w);
#pragma unroll
                for (int j = 0; j < V; j++) {
                    xn[u][j] = f[j] * r;
                    dxn[u][j] = g[j] * w[j];
                    dot += dxn[u][j] * xn[u][j];
                }
            }
        }
    }
    dot = wave_sum(dot) / static_cast<float>(E);
    for (int64_t c0 = 0; c0 < nv; c0 += 64 * U) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int64_t c = c0 + u * 64 + lane;
            if (c < nv) {
                if (!VECS) {
                    float g[V], f[V], w[V];
                    Elem<T>::unpack(dyr[c], g);
                    Elem<T>::unpack(hr[c], f);
                    Elem<T>::unpack(wr[c], w);
#pragma unroll
                    for (int j = 0; j < V; j++) { xn[u][j] = f[j] * r; dxn[u][j] = g[j] * w[j]; }
                }
                float o[V];
#pragma unroll
                for (int j = 0; j < V; j++) o[j] = r * (dxn[u][j] - xn[u][j] * dot);
                if (ADD) add_rounded<T>(reinterpret_cast<const u32x4 *>(h_grad + row * E)[c], o);
                dxr[c] = Elem<T>::pack(o);
            }
        }
    }
}

// Partial weight gradient of a chunk of DW_ROWS rows for 64 * V columns: a lane owns V columns,
// the four wavefronts of the block take the rows in turn and are added through LDS.
template <typename T>
__global__ __launch_bounds__(256) void rmsnorm_dw_kernel(const T *__restrict__ dy,
                                                         const T *__restrict__ h,
                                                         const float *__restrict__ rstd,
                                                         float *__restrict__ dw_part, int64_t rows,
                                                         int64_t E) {
    constexpr int V = Elem<T>::VEC;
    __shared__ float lds_dw[4][64 * V];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t c = static_cast<int64_t>(blockIdx.x) * 64 + lane;      // 16-byte column
    const int64_t r0 = static_cast<int64_t>(blockIdx.y) * DW_ROWS;
    float dw[V];
#pragma unroll
    for (int j = 0; j < V; j++) dw[j] = 0.0f;
    if (c * V < E) {
        for (int i = wave; i < DW_ROWS; i += 4) {
            const int64_t row = r0 + i;
            if (row >= rows) break;
            const float r = rstd[row];
            float g[V], f[V];
            Elem<T>::unpack(reinterpret_cast<const u32x4 *>(dy + row * E)[c], g);
            Elem<T>::unpack(reinterpret_cast<const u32x4 *>(h + row * E)[c], f);
#pragma unroll
            for (int j = 0; j < V; j++) dw[j] += g[j] * round_like<T>(f[j] * r);
        }
    }
#pragma unroll
    for (int j = 0; j < V; j++) lds_dw[wave][lane * V + j] = dw[j];
    __syncthreads();
    for (int t = threadIdx.x; t < 64 * V; t += 256) {
        const int64_t e = static_cast<int64_t>(blockIdx.x) * 64 * V + t;
        if (e < E)
            dw_part[static_cast<int64_t>(blockIdx.y) * E + e] =
                (lds_dw[0][t] + lds_dw[1][t]) + (lds_dw[2][t] + lds_dw[3][t]);
    }
}

// The chunks' partial sums: a quarter of the chunks, in their order, to each of four wavefronts, 16 loads in flight (one load at a time in
// eight blocks took 32 us at 16384 rows of 2048, 128 chunks).
constexpr int DW_REDUCE = 64;   // columns per block
template <typename T>
__global__ __launch_bounds__(4 * DW_REDUCE) void rmsnorm_dw_reduce_kernel(const float *__restrict__ dw_part, int n_blocks, int64_t E,
                                                                          T *__restrict__ dweight) {
    __shared__ float quarter[4][DW_REDUCE];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t e = static_cast<int64_t>(blockIdx.x) * DW_REDUCE + lane;
    const int end = n_blocks * (wave + 1) / 4;
    int b = n_blocks * wave / 4;
    float s = 0.0f;
    if (e < E) {
        for (; b + 16 <= end; b += 16) {
            float v[16];
#pragma unroll
            for (int u = 0; u < 16; u++) v[u] = dw_part[static_cast<int64_t>(b + u) * E + e];
#pragma unroll
            for (int u = 0; u < 16; u++) s += v[u];
        }
        // the rest together too (past the last of them: it again, not added): 3001 rows of 1000 bf16, whole backward, 13.6 -> 10.7 us; in every
        // round it cost 16384 rows of 2048 1.6 us
        if (b < end) {
            float v[16];
#pragma unroll
            for (int u = 0; u < 16; u++) v[u] = dw_part[static_cast<int64_t>(min(b + u, end - 1)) * E + e];
#pragma unroll
            for (int u = 0; u < 16; u++) s += b + u < end ? v[u] : 0.0f;
        }
    }
    quarter[wave][lane] = s;
    __syncthreads();
    if (wave == 0 && e < E) Elem<T>::store(dweight + e, (quarter[0][lane] + quarter[1][lane]) + (quarter[2][lane] + quarter[3][lane]));
}

// f(vectors a lane of one wavefront holds of a row of nv) where that is at most ROW_VECS
template <typename F> bool with_vecs(int64_t nv, F f) {
    if (nv <= 64) f(std::integral_constant<int, 1>());
    else if (nv <= 128) f(std::integral_constant<int, 2>());
    else if (nv <= 192) f(std::integral_constant<int, 3>());
    else if (nv <= 256) f(std::integral_constant<int, 4>());
    else return false;
    static_assert(ROW_VECS == 4, "the cases above");
    return true;
}

}  // namespace

extern "C" int om_rmsnorm_fwd(const void *x, const void *residual, const void *weight, double eps,
                              void *out, void *h_out, float *rstd_out, int64_t rows, int64_t E,
                              int dtype, void *stream) {
    if (dtype != OM_F32 && dtype != OM_BF16) return OM_ERR_DTYPE;
    const int V = dtype == OM_F32 ? 4 : 8;
    if (rows < 0 || E < 1 || E % V != 0 || rows > 0x7fffffffLL) return OM_ERR_SHAPE;
    if (rows == 0) return OM_OK;
    if (!x || !weight || !out) return OM_ERR_NULL;
    if (!om_aligned16(x) || !om_aligned16(weight) || !om_aligned16(out) ||
        (residual && !om_aligned16(residual)) || (h_out && !om_aligned16(h_out)))
        return OM_ERR_ALIGN;
    hipStream_t st = om_stream(stream);
    auto run = [&](auto type) {
        using T = decltype(type);
        const T *xt = static_cast<const T *>(x), *rt = static_cast<const T *>(residual), *wt = static_cast<const T *>(weight);
        T *ot = static_cast<T *>(out), *ht = static_cast<T *>(h_out);
        const float e = static_cast<float>(eps);
        const bool past = rows * E >= NORM_PAST_CACHES;
        const bool fits = with_vecs(E / V, [&](auto vecs) {
            constexpr int N = decltype(vecs)::value;
            const unsigned nb = static_cast<unsigned>(rows);
            if (past) rmsnorm_fwd_row_kernel<T, N, true><<<nb, 64, 0, st>>>(xt, rt, wt, e, ot, ht, rstd_out, E);
            else rmsnorm_fwd_row_kernel<T, N, false><<<nb, 64, 0, st>>>(xt, rt, wt, e, ot, ht, rstd_out, E);
        });
        const unsigned nb = static_cast<unsigned>((rows + NORM_ROWS - 1) / NORM_ROWS);
        if (fits) return;
        if (past && h_out) rmsnorm_fwd_kernel<T, true><<<nb, 256, 0, st>>>(xt, rt, wt, e, ot, ht, rstd_out, rows, E);
        else rmsnorm_fwd_kernel<T, false><<<nb, 256, 0, st>>>(xt, rt, wt, e, ot, ht, rstd_out, rows, E);
    };
    if (dtype == OM_BF16) run(uint16_t());
    else run(float());
    return om_launch_status();
}

extern "C" int64_t om_rmsnorm_bwd_workspace_bytes(int64_t rows, int64_t E) {
    if (rows < 0 || E < 1) return 0;
    return ((rows + DW_ROWS - 1) / DW_ROWS) * E * 4;
}

extern "C" int64_t om_rmsnorm_bwd_workspace_spread_bytes(int64_t rows, int64_t E) {
    if (rows < 0 || E < 1) return 0;
    const int64_t chunk = std::min<int64_t>(bwd_chunk(rows), DW_ROWS);
    return chunk ? ((rows + chunk - 1) / chunk) * E * 4 : 0;
}

extern "C" int om_rmsnorm_bwd(const void *dy, const void *h, const void *weight, const float *rstd,
                              void *dx, void *dweight, void *workspace, int64_t workspace_bytes,
                              int64_t rows, int64_t E, int dtype, void *stream) {
    return om_rmsnorm_bwd_residual(dy, h, weight, rstd, nullptr, dx, dweight, workspace, workspace_bytes, rows, E, dtype, stream);
}

extern "C" int om_rmsnorm_bwd_residual(const void *dy, const void *h, const void *weight, const float *rstd, const void *h_grad,
                                       void *dx, void *dweight, void *workspace, int64_t workspace_bytes,
                                       int64_t rows, int64_t E, int dtype, void *stream) {
    if (dtype != OM_F32 && dtype != OM_BF16) return OM_ERR_DTYPE;
    const int V = dtype == OM_F32 ? 4 : 8;
    if (rows < 1 || E < 1 || E % V != 0 || rows > 0x7fffffffLL) return OM_ERR_SHAPE;
    if (!dy || !h || !weight || !rstd || !dx || !dweight || !workspace) return OM_ERR_NULL;
    if (!om_aligned16(dy) || !om_aligned16(h) || !om_aligned16(weight) || !om_aligned16(dx) || !om_aligned16(h_grad))
        return OM_ERR_ALIGN;
    if (workspace_bytes < om_rmsnorm_bwd_workspace_bytes(rows, E)) return OM_ERR_WORKSPACE;
    hipStream_t st = om_stream(stream);
    float *part = static_cast<float *>(workspace);
    auto run = [&](auto type) {
        using T = decltype(type);
        const T *g = static_cast<const T *>(dy), *hh = static_cast<const T *>(h), *wt = static_cast<const T *>(weight);
        T *to = static_cast<T *>(dx);
        const T *hg = static_cast<const T *>(h_grad);
        // (a smaller workspace: the kernels of longer rows, whose chunks' sums it holds; 128-row chunks of this one would be a few blocks)
        const int chunk = static_cast<int>(std::min<int64_t>(bwd_chunk(rows), DW_ROWS));
        int chunks = static_cast<int>((rows + chunk - 1) / chunk);
        const bool fits = workspace_bytes >= om_rmsnorm_bwd_workspace_spread_bytes(rows, E) && with_vecs(E / V, [&](auto vecs) {
            constexpr int N = decltype(vecs)::value;
            if (rows * E >= NORM_PAST_CACHES) rmsnorm_bwd_rows_kernel<T, N, true><<<chunks, 256, 0, st>>>(g, hh, wt, rstd, hg, to, part, rows, E, chunk);
            else rmsnorm_bwd_rows_kernel<T, N, false><<<chunks, 256, 0, st>>>(g, hh, wt, rstd, hg, to, part, rows, E, chunk);
        });
        if (!fits) {
            chunks = static_cast<int>((rows + DW_ROWS - 1) / DW_ROWS);
            const dim3 grid(static_cast<unsigned>((rows + NORM_ROWS - 1) / NORM_ROWS));
            auto rows_dx = [&](auto vecs) {
                constexpr int N = decltype(vecs)::value;
                if (hg) rmsnorm_dx_kernel<T, N, true><<<grid, 256, 0, st>>>(g, hh, wt, rstd, hg, to, rows, E);
                else rmsnorm_dx_kernel<T, N, false><<<grid, 256, 0, st>>>(g, hh, wt, rstd, hg, to, rows, E);
            };
            if (!with_vecs(E / V, rows_dx)) rows_dx(std::integral_constant<int, 0>());
            rmsnorm_dw_kernel<T><<<dim3(static_cast<unsigned>((E / V + 63) / 64), static_cast<unsigned>(chunks)), 256, 0, st>>>(g, hh, rstd, part, rows, E);
        }
        rmsnorm_dw_reduce_kernel<T><<<static_cast<unsigned>((E + DW_REDUCE - 1) / DW_REDUCE), 4 * DW_REDUCE, 0, st>>>(part, chunks, E, static_cast<T *>(dweight));
    };
    if (dtype == OM_BF16) run(uint16_t());
    else run(float());
    return om_launch_status();
}

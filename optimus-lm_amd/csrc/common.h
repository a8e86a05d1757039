// Shared device/host helpers for the gfx950 kernels of liboptimus_mi355x.so.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "../../include/optimus_mi355x.h"

#define OM_WAVE 64

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;
typedef __attribute__((ext_vector_type(4))) short s16x4;

static inline hipStream_t om_stream(void *s) { return reinterpret_cast<hipStream_t>(s); }

static inline int om_launch_status() {
    return hipGetLastError() == hipSuccess ? OM_OK : OM_ERR_LAUNCH;
}

static inline bool om_aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// bf16 <-> fp32 on raw bits; round-to-nearest-even, NaN kept quiet (what at::BFloat16 does).
__device__ __forceinline__ float bf16_bits_to_f32(uint16_t h) {
    return __uint_as_float(static_cast<uint32_t>(h) << 16);
}
__device__ __forceinline__ uint16_t f32_to_bf16_bits(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0;
    u += 0x7fffu + ((u >> 16) & 1u);
    return static_cast<uint16_t>(u >> 16);
}

// Element traits for the row movers: a 16-byte vector of T and fp32 views of it.
template <typename T> struct Elem;
template <> struct Elem<float> {
    static constexpr int VEC = 4;
    __device__ static __forceinline__ void unpack(const u32x4 &v, float *f) {
        for (int i = 0; i < 4; i++) f[i] = __uint_as_float(v[i]);
    }
    __device__ static __forceinline__ u32x4 pack(const float *f) {
        u32x4 v;
        for (int i = 0; i < 4; i++) v[i] = __float_as_uint(f[i]);
        return v;
    }
    __device__ static __forceinline__ float load(const float *p) { return *p; }
    __device__ static __forceinline__ void store(float *p, float f) { *p = f; }
};
template <> struct Elem<uint16_t> {  // bf16 as raw bits
    static constexpr int VEC = 8;
    __device__ static __forceinline__ void unpack(const u32x4 &v, float *f) {
        for (int i = 0; i < 4; i++) {
            f[2 * i] = __uint_as_float(v[i] << 16);
            f[2 * i + 1] = __uint_as_float(v[i] & 0xffff0000u);
        }
    }
    __device__ static __forceinline__ u32x4 pack(const float *f) {
        u32x4 v;
        for (int i = 0; i < 4; i++)
            v[i] = static_cast<uint32_t>(f32_to_bf16_bits(f[2 * i])) |
                   (static_cast<uint32_t>(f32_to_bf16_bits(f[2 * i + 1])) << 16);
        return v;
    }
    __device__ static __forceinline__ float load(const uint16_t *p) { return bf16_bits_to_f32(*p); }
    __device__ static __forceinline__ void store(uint16_t *p, float f) { *p = f32_to_bf16_bits(f); }
};

// Wave-wide reductions over 64 lanes (xor butterfly: every lane ends with the result).
__device__ __forceinline__ float wave_sum(float v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ int wave_sum_i(int v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Stores a vector (8 or 16 bytes a lane) past the caches, `bytes` behind a block-uniform address; bytes < 2^31.  Of the cache
// policies of a store nt alone leaves the lines in the L2s, which write them back in their own order, when the kernel ends or under the
// next one; with sc1 as well they go on to memory at once.  Weight gradients of 64 experts of 2048/1024, 512 tokens with popularity as
// rank^-1.2, whole training steps, us: through the caches 656, nt 618, sc1 656, sc0 sc1 658, sc1 nt 593, sc0 sc1 nt 596 (two
// boxes, one side of each 604 to 606).  No gain for gradients that were just read to be added to.
template <typename T> __device__ __forceinline__ void store_past_caches(void *base, uint32_t bytes, T v) {
    constexpr int SC1_NT = 16 | 2;
    auto rsrc = __builtin_amdgcn_make_buffer_rsrc(base, 0, 0x7fffffff, 0x00020000);
    static_assert(sizeof(T) == 16 || sizeof(T) == 8, "one vector a lane");
    if constexpr (sizeof(T) == 16) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), rsrc, bytes, 0, SC1_NT);
    else __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), rsrc, bytes, 0, SC1_NT);
}

// Direct load of 16 bytes from each lane's address to LDS at lds + 16 * lane.  Outside the compiler's view: the code waits
// for it itself (vmcnt counts it).
__device__ __forceinline__ void dma16_lane(const char *lane_address, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(lane_address) : "memory");
}
__device__ __forceinline__ uint32_t lds_address(char *shared) {
    typedef __attribute__((address_space(3))) char *lds_bytes;
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_bytes)shared));
}

// Whether two arrays of n blocks (`bytes` each, `pitch` bytes apart, positive) have a byte in common: block by block, since
// the gradients of per-expert modules in a flat buffer lie between one another.
inline bool om_blocks_overlap(const void *a, int64_t a_pitch, int64_t a_bytes, const void *b, int64_t b_pitch, int64_t b_bytes, int n) {
    const int64_t d = static_cast<int64_t>(reinterpret_cast<uintptr_t>(b)) - static_cast<int64_t>(reinterpret_cast<uintptr_t>(a));
    if (d >= (n - 1) * a_pitch + a_bytes || d + (n - 1) * b_pitch + b_bytes <= 0) return false;
    // is there a block j in [lo, hi] of b with -b_bytes < d + j * b_pitch - at < a_bytes, `at` the offset of a block of a?
    auto floor_div = [](int64_t x, int64_t y) { return x >= 0 ? x / y : -((-x + y - 1) / y); };
    auto hit = [&](int64_t at, int64_t lo, int64_t hi) {
        const int64_t first = floor_div(at - d - b_bytes, b_pitch) + 1, last = floor_div(at - d + a_bytes - 1, b_pitch);
        return (first > lo ? first : lo) <= (last < hi ? last : hi);
    };
    if (a_pitch == b_pitch) return hit(0, 1 - n, n - 1);   // (only the difference of the block numbers matters)
    for (int i = 0; i < n; i++)
        if (hit(i * a_pitch, 0, n - 1)) return true;
    return false;
}

// 1 / (1 + e^-x) with the hardware exponential and reciprocal (about 1 ulp each, far inside one
// bf16 rounding of the results it feeds).  An IEEE division here costs ten instructions per
// element, and the SwiGLU epilogues are bound by vector-ALU issue.
__device__ __forceinline__ float fast_sigmoid(float x) {
    return __builtin_amdgcn_rcpf(1.0f + __expf(-x));
}

// The grouped products of few rows per expert (ggemm_stream.hip): the rule, and the launches that the entry
// points of ggemm.hip make under it.  Arguments are checked by the caller.  `expected`: the rows to choose by,
// `rows` where they are known and fewer where `rows` is a bound.
bool om_ggemm_streams(int64_t rows, int n_experts, int cols, bool past_caches);   // cols: weight rows per expert (gate and up: both)
// Elements of weights, or of their gradients, that the caches cannot hold from one use to the next (see ggemm.hip).
constexpr int64_t CACHED_WEIGHTS = 128 << 20;
// Whether the tiled kernels load a launch's weights (`elements` in all, rows `pitch` apart) past the caches, or store its weight
// gradients so: only where the 128-byte pieces that they load or store are whole lines.  A line of two pieces would be fetched twice, which the caches otherwise
// spare: forward of 64 experts, ffn 1024, us, through the caches -> past them: hidden 2600, 37 tokens 225 -> 243, 512 tokens 283 -> 326, hidden
// 2624 207 -> 181, 249 -> 241; 16 experts of 7000/2040, 2 tokens 280 -> 328, of 7168/2048 231 -> 208.  Written gradients
// 16 bytes off a line: 32 experts of 2048/7168, 128 rows 597 -> 1552, on a line 576 -> 524.
inline bool om_weights_pass_caches(const void *w, int64_t elements, int64_t pitch, int64_t expert_pitch) {
    return elements >= CACHED_WEIGHTS && pitch % 64 == 0 && expert_pitch % 64 == 0 && reinterpret_cast<uintptr_t>(w) % 128 == 0;
}
int om_ggemm_stream_gate_up(const void *x, const int32_t *x_rows, const void *w_gate, const void *w_up,
                            const float *row_weights, void *g, void *u, void *h, const int32_t *cum, int64_t rows, int64_t expected,
                            int G, int I, int H, int64_t w_stride, hipStream_t st);
int om_ggemm_stream_fwd(const void *x, const void *w, void *out, const int32_t *cum, int64_t rows, int64_t expected, int G,
                        int N, int K, int64_t w_stride, hipStream_t st);

// The split gate projection (gate_fwd.hip) as the routing kernels' producer (route.hip): slices of H, and
// the launch that leaves partial[splits][T][N].  Arguments are checked by the caller.
int om_gate_route_splits(int64_t T, int H, int N);
void om_launch_gate_partials(const void *x, const void *gate_weight, int64_t T, int H, int N, int splits, float *partial,
                             hipStream_t stream);
// The softmax router's backward (route.hip) as the gate's gradients' producer: dlogits in float32 (rounded to the logits' type on the
// way, as the separate entry point stores them; `more`: another gradient of the logits, in their type, is added with that type's rounding), and `n_zero` words zeroed.
void om_launch_softmax_bwd(const void *logits, int logits_dtype, const int64_t *experts, const void *dweights, int dweights_dtype,
                           const void *more, int64_t T, int N, int K, int renorm, float *dlogits, unsigned *zero, int n_zero,
                           hipStream_t stream);

// Grouped expert GEMMs in float32 (v_mfma_f32_32x32x2_f32, fp32 operands and accumulation), for
// modules kept in float32 like the reference's small CPU-runnable configuration
// (GroupedGemmFunction, optimus/models/common/moe.py:163-215, runs torch.matmul per expert in
// whatever dtype the module has).  Same products and the same variable-rows-per-expert contract as
// the bf16 kernels: forward, input gradient, weight gradient, and the merged MLP's forms of them (gate
// and up in one launch with the SwiGLU or its backward in the epilogue, the token gather in the loads; in the backward
// the input gradient and all three weight gradients).
//
// What bounds these launches is that they are small (the tiny layer, 2048 tokens, hidden 256, ffn 512, 8 experts, top-2:
// 1.07 GFLOP a product, 7 us at the matrix rate): whole tiles per CU, and a tile's own chain of latencies.  Tiles are 64
// columns wide and 32 or 64 rows high; each 32x32 block of the output is worked by two wavefronts, one for each half of a
// step's indices, in two sums that take turns.  A step is 32 indices, 8 MFMAs a wavefront; the loads run four steps ahead
// and the fragments one, so that nothing but the MFMAs is waited for inside a step.  In the backward the input gradient
// and the weight gradients, independent of each other, are one launch, whose tiles fill the CUs that each alone leaves
// idle.  The matrix cores do not reach their sustained rate in these bursts: MFMAs alone, on every SIMD for 60 us, take
// 31 ns each where they take 27 for 2 ms.
// Tiny layer with 520 rows an expert, us a launch in a replayed graph, with 64x64 tiles staged through registers two
// 64-deep steps ahead -> now: gate+up 39 -> 33, down 24 -> 20, down input gradient 28 -> 23, the rest of the backward
// 88 (44 + 28 + 16) -> 73; with 64 rows an expert 10.5 -> 7.4, 13 -> 9.3, 10.7 -> 7.8, 35 -> 20.
//
// A tile's operands come in steps of 32 contraction indices c through a ring of LDS slots, by direct global->LDS loads
// (as in ggemm.hip: written as assembly, with waits and barriers of their own).  CONTIG operands ([row][c] in memory)
// lie as 128-byte rows, STRIDED ones ([c][row] in memory: the weight in dgrad, both operands in wgrad) as 256-byte
// c-rows (B) or 128-byte ones (wgrad's A), their 16-byte chunks XOR-permuted so that fragment reads meet no bank
// conflict; a direct load writes LDS at (wave-uniform base + lane*16), so each lane fetches the chunk that belongs there.
#include "common.h"
#include <algorithm>
#include <type_traits>

namespace {

constexpr int TN = 64;            // tile columns
constexpr int KS = 32;            // contraction step: 16 indices for each of the two halves of the wavefronts
constexpr int SLOTS = 4;
constexpr int PITCH = TN + 4;     // floats between the rows of a finished tile in LDS
// A tile of 32 * MW rows: MW x 2 wavefronts of 32x32 for each half of a step's indices.
template <int MW> struct Tile {
    static constexpr int ROWS = 32 * MW, THREADS = 256 * MW;
    static constexpr int A_BYTES = ROWS * KS * 4, SLOT = A_BYTES + TN * KS * 4;
    static constexpr int B_LOADS = 2 / MW;              // direct loads per wavefront and step; one of A
    static_assert(SLOTS * SLOT >= 2 * ROWS * PITCH * 4, "the finished tile lies where the ring was");
};
constexpr int IDX_CACHE = 1024;   // weight gradient: row indices of a segment kept in LDS
typedef __attribute__((ext_vector_type(4))) float f4;

enum { F_CONTIG = 0, F_STRIDED = 1 };
enum { E_STORE = 0, E_SWIGLU = 1, E_SWIGLU_BWD = 2 };

struct F32Params {
    const float *A[2], *B[2];   // second pair: up matrix (E_SWIGLU) or second phase
    float *C[3];                // output; E_SWIGLU: g, u, h; E_SWIGLU_BWD: dg, du
    const float *G, *U;         // E_SWIGLU_BWD: saved g, u
    const int32_t *cum;
    const int32_t *row_index;   // row r of A is row row_index[r]
    int64_t lda, ldb, ldc, strideB[2];
    int n_experts, n_cols, kc, phases;
};
// Weight gradients over the same rows: dW[s][g][n][k] (+)= sum_r A[s][r][n] * B[s][r][k]
struct F32Wgrad {
    const float *A[3], *B[3];
    float *C[3];
    const int32_t *b_rows[3];   // not null: row r of B[s] is row b_rows[s][r]
    int64_t strideC[3];
    int n[3], k[3];
    const int32_t *cum;
    int n_experts, sets, accumulate;   // accumulate, bit s: C[s] += product
};

template <int V> using IntC = std::integral_constant<int, V>;

// 16 bytes per lane global -> LDS at lds_base + lane * 16; nothing with fewer than NEED steps `left`
template <int NEED> __device__ __forceinline__ void dma16_if(int left, const char *lane_address, uint32_t lds_base) {
    asm volatile("s_cmp_lt_i32 %2, %3\n\ts_cbranch_scc1 .Lom_skip%=\n\ts_mov_b32 m0, %0\n\ts_nop 0\n\t"
                 "global_load_lds_dwordx4 %1, off\n.Lom_skip%=:"
                 :: "s"(lds_base), "v"(lane_address), "s"(left), "n"(NEED) : "scc");
}
// All loads but those of the two (one, no) youngest steps have landed, by the steps that follow; LDS reads are back.
template <int PER_STEP> __device__ __forceinline__ void wait_step(int left, uint32_t lds) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_cmp_ge_i32 %2, 4\n\ts_cbranch_scc1 .Lom_wait%=\n\ts_waitcnt vmcnt(%1)\n\t"
                 "s_cmp_ge_i32 %2, 3\n\ts_cbranch_scc1 .Lom_wait%=\n\ts_waitcnt vmcnt(0)\n.Lom_wait%=:"
                 :: "n"(2 * PER_STEP), "n"(PER_STEP), "s"(left), "s"(lds) : "memory", "scc");
}
__device__ __forceinline__ void block_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

__device__ __forceinline__ int swz(int row) { return (row >> 1) & 7; }   // CONTIG: 128-byte rows
// STRIDED B (256-byte c-rows): the c-rows that the two halves of a wavefront read lie in different halves of the banks.
// The halves of a wavefront take c and c + 4 beside a CONTIG A, whose lanes read four neighbouring indices, c and c + 1
// beside a STRIDED one.
template <int AKIND> __device__ __forceinline__ int half_bit(int c) { return AKIND == F_CONTIG ? (c >> 2) & 1 : c & 1; }

// Where this lane's slot of direct load `load` lies in a tile of COLS rows (CONTIG) or columns (STRIDED): the
// row or contraction row, and the chunk of 4 floats.
template <int COLS, int AKIND, int KIND> __device__ __forceinline__ void dma_slot(int load, int lane, int &row, int &chunk) {
    if (KIND == F_CONTIG || COLS == 32) {
        row = load * 8 + (lane >> 3);
        chunk = KIND == F_CONTIG ? (lane & 7) ^ swz(row) : lane & 7;
    } else {
        row = load * 4 + (lane >> 4);
        chunk = (lane & 15) ^ (half_bit<AKIND>(row) << 3);
    }
}

// This lane's source of one operand, stepped through the contraction.  Steps 0 .. steps - 1 are `stride` bytes apart; with
// a second phase the next `steps` follow at `second` bytes from the first ones.  A phase's last step may hold fewer than KS
// indices: `back` bytes less there re-read valid data (zeroed in LDS).
struct Source {
    const char *at;
    int64_t stride, jump;       // jump: from a phase's last step to the next one's first
    uint32_t back;
    __device__ __forceinline__ void next(bool wraps) { at += wraps ? jump : stride; }
    __device__ __forceinline__ const char *address(uint32_t tail_mask) const { return at - (back & tail_mask); }
};

// The main loop.  load_a() / load_b(i): this lane's addresses of the step that is loaded next; advance(): to the one after
// it; tail_of(t): does step t hold fewer than KS indices; a_past, b_past: do the lane's slots then lie past them.  Those hold
// other data and are zeroed, of both operands: zeros of one alone would turn an infinity of the other into a NaN.
// acc: this wavefront's 32x32 block (columns 32 * (wave & 1), rows 32 * the next bit with MW 2) over its half of every step.
template <int MW, int AKIND, int BKIND, typename FA, typename FB, typename FN, typename FT>
__device__ __forceinline__ void multiply(char *lds, int n_steps, FA &&load_a, FB &&load_b, FN &&advance, FT &&tail_of, bool a_past,
                                         const bool (&b_past)[Tile<MW>::B_LOADS], f32x16 &acc) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int SLOT = Tile<MW>::SLOT, A_BYTES = Tile<MW>::A_BYTES, B_LOADS = Tile<MW>::B_LOADS, LOADS = 1 + B_LOADS;
    constexpr int S = KS / 16;                           // fragments of 8 indices per wavefront and step
    const int kh = wave / (2 * MW), half = lane >> 5, l32 = lane & 31, m32 = MW == 1 ? l32 : ((wave >> 1) & 1) * 32 + l32;
    const uint32_t lds_addr = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char *)lds));
    const uint32_t a_dst = __builtin_amdgcn_readfirstlane(lds_addr + wave * 1024);
    const uint32_t b_dst = __builtin_amdgcn_readfirstlane(lds_addr + A_BYTES + wave * (B_LOADS * 1024));
    f32x16 sum[2];                                       // of the first and the second half of a wavefront's fragments
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = sum[0][r] = sum[1][r] = 0.0f;
    if (n_steps <= 0) return;
    auto issue = [&](int left, auto slot) {              // (`left` - 4 steps follow the one to load)
        constexpr int O = decltype(slot)::value * SLOT;
        dma16_if<4>(left, load_a(), a_dst + O);
        dma16_if<4>(left, load_b(0), b_dst + O);
        if (B_LOADS == 2) dma16_if<4>(left, load_b(1), b_dst + O + 1024);
        advance();
    };
    auto zero = [&](int t, auto slot) {
        if (!tail_of(t)) return;
        char *own = lds + decltype(slot)::value * SLOT + lane * 16;
        const f4 zeros = {0.0f, 0.0f, 0.0f, 0.0f};
        if (a_past) *reinterpret_cast<f4 *>(own + wave * 1024) = zeros;
#pragma unroll
        for (int i = 0; i < B_LOADS; i++)
            if (b_past[i]) *reinterpret_cast<f4 *>(own + A_BYTES + (wave * B_LOADS + i) * 1024) = zeros;
    };
    // fragment addresses; element j of fragment s goes to MFMA 4 * s + j
    int a_frag[S], b_frag[S];
    const int c0 = kh * 16 + (AKIND == F_CONTIG ? 4 * half : half);
    const int col = (wave & 1) * 32 + l32;
#pragma unroll
    for (int s = 0; s < S; s++) {
        a_frag[s] = AKIND == F_CONTIG ? m32 * 128 + (((kh * 4 + 2 * s + half) ^ swz(m32)) << 4)
                    : MW == 1 ? (c0 + 8 * s) * 128 + m32 * 4
                              : (c0 + 8 * s) * 256 + (((m32 >> 2) ^ (half << 3)) << 4) + (m32 & 3) * 4;
        b_frag[s] = A_BYTES + (BKIND == F_CONTIG ? col * 128 + (((kh * 4 + 2 * s + half) ^ swz(col)) << 4)
                                                 : (c0 + 8 * s) * 256 + (((col >> 2) ^ (half << 3)) << 4) + (col & 3) * 4);
    }
    float fa[2][S][4], fb[2][S][4];
    auto read = [&](auto slot, auto buf) {
        constexpr int O = decltype(slot)::value * SLOT, P = decltype(buf)::value;
        constexpr int J = AKIND == F_CONTIG ? 1 : 2;      // c-rows from element to element (STRIDED)
#pragma unroll
        for (int s = 0; s < S; s++) {
            if (AKIND == F_CONTIG) {
                const f4 v = *reinterpret_cast<const f4 *>(lds + a_frag[s] + O);
#pragma unroll
                for (int j = 0; j < 4; j++) fa[P][s][j] = v[j];
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++) fa[P][s][j] = *reinterpret_cast<const float *>(lds + a_frag[0] + O + s * 8 * (128 * MW) + j * J * (128 * MW));
            }
            if (BKIND == F_CONTIG) {
                const f4 v = *reinterpret_cast<const f4 *>(lds + b_frag[s] + O);
#pragma unroll
                for (int j = 0; j < 4; j++) fb[P][s][j] = v[j];
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++) fb[P][s][j] = *reinterpret_cast<const float *>(lds + b_frag[0] + O + s * 8 * 256 + j * J * 256);
            }
        }
    };
    // step t, whose fragments are in registers: loads of step t + 4 into its slot, fragments of step t + 1
    auto step = [&](auto slot, int t) {
        constexpr int Q = decltype(slot)::value;
        const int left = __builtin_amdgcn_readfirstlane(n_steps - 1 - t);
        read(IntC<(Q + 1) & 3>{}, IntC<(Q + 1) & 1>{});
        issue(left, slot);
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int s = 0; s < S; s++) {
                // (the two sums in turn: no MFMA waits for the one before it)
                const int x = (s & 1) * (S / 2) + s / 2;
                // operands swapped: lane l then holds output row l%32 and columns 8*(r/4) + 4*(l/32) + r%4
                sum[s & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[Q & 1][x][j], fa[Q & 1][x][j], sum[s & 1], 0, 0, 0);
            }
        // one MFMA, the LDS reads behind it, the other MFMAs (with the loads and their addresses between them), the wait
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, S * ((AKIND == F_CONTIG ? 1 : 2) + (BKIND == F_CONTIG ? 1 : 2)), 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 4 * S - 1, 0);
        __builtin_amdgcn_sched_barrier(0);
        wait_step<LOADS>(left, lds_addr);
        zero(t + 2, IntC<(Q + 2) & 3>{});
        block_barrier();
    };
    issue(4, IntC<0>{});
    issue(n_steps + 2, IntC<1>{});
    issue(n_steps + 1, IntC<2>{});
    issue(n_steps, IntC<3>{});
    wait_step<LOADS>(n_steps, lds_addr);     // steps 0 and 1
    zero(0, IntC<0>{});
    zero(1, IntC<1>{});
    block_barrier();
    read(IntC<0>{}, IntC<0>{});
    block_barrier();                         // (step 0 loads into what was read here)
    for (int t = 0;; t += 4) {
        step(IntC<0>{}, t);
        if (t + 1 >= n_steps) break;
        step(IntC<1>{}, t + 1);
        if (t + 2 >= n_steps) break;
        step(IntC<2>{}, t + 2);
        if (t + 3 >= n_steps) break;
        step(IntC<3>{}, t + 3);
        if (t + 4 >= n_steps) break;
    }
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = sum[0][r] + sum[1][r];
}

// The wavefronts' blocks into LDS ([half][row][PITCH]); after it any thread finds the tile there.
template <int MW> __device__ __forceinline__ void finish(char *lds, const f32x16 &acc) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();
    float *plane = reinterpret_cast<float *>(lds) + ((wave >> 1) * 32 + (lane & 31)) * PITCH + (wave & 1) * 32 + (lane >> 5) * 4;
#pragma unroll
    for (int q = 0; q < 4; q++) *reinterpret_cast<f4 *>(plane + q * 8) = f4{acc[q * 4], acc[q * 4 + 1], acc[q * 4 + 2], acc[q * 4 + 3]};
    __syncthreads();
}
template <int MW> __device__ __forceinline__ f4 finished(const char *lds, int row, int col) {
    const float *q = reinterpret_cast<const float *>(lds) + row * PITCH + col;
    const f4 v = *reinterpret_cast<const f4 *>(q);
    return v + *reinterpret_cast<const f4 *>(q + Tile<MW>::ROWS * PITCH);
}

// Which expert owns row tile `tile`: every wavefront scans the counts 64 experts at a time.
template <int TM>
__device__ __forceinline__ bool find_row_tile(const int32_t *cum, int n_experts, int tile, int &expert, int &begin, int &end) {
    const int lane = threadIdx.x & 63;
    int base = 0;
    for (int e0 = 0; e0 < n_experts; e0 += 64) {
        const int e = e0 + lane;
        int s = 0, cnt = 0;
        if (e < n_experts) { s = cum[e]; cnt = cum[e + 1] - s; }
        const int tiles = (cnt + TM - 1) / TM;
        int incl = tiles;
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(incl, o, 64);
            if (lane >= o) incl += v;
        }
        const unsigned long long mine = __ballot(tile >= base + incl - tiles && tile < base + incl);
        if (mine) {
            const int src = __ffsll(static_cast<long long>(mine)) - 1;
            expert = e0 + src;
            begin = __shfl(s + (tile - base - (incl - tiles)) * TM, src, 64);
            end = __shfl(s + cnt, src, 64);
            return true;
        }
        base += __shfl(incl, 63, 64);
    }
    return false;
}

#pragma clang fp contract(off)

// One tile of a forward / input-gradient product: row tile (cut per expert) and column tile (E_SWIGLU: 32 columns of gate
// and the same 32 of up, side by side in the tile)
template <int MW, int BKIND, int EPI, bool GATHER>
__device__ __forceinline__ void rows_tile(const F32Params &p, char *lds, int row_tile, int col_tile) {
    int expert, m0, m_end;
    if (!find_row_tile<Tile<MW>::ROWS>(p.cum, p.n_experts, row_tile, expert, m0, m_end)) return;   // (the whole block)
    expert = __builtin_amdgcn_readfirstlane(expert);
    constexpr int COLS = EPI == E_SWIGLU ? TN / 2 : TN;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = col_tile * COLS;
    const int steps = (p.kc + KS - 1) / KS, tail = p.kc % KS ? steps - 1 : -1;
    const int left_in_tail = p.kc - (steps - 1) * KS;    // indices in a phase's last step
    constexpr int B_LOADS = Tile<MW>::B_LOADS;
    Source a, b[B_LOADS];
    bool b_past[B_LOADS];
    const float *B0 = p.B[0] + expert * p.strideB[0], *B1 = p.phases > 1 || EPI == E_SWIGLU ? p.B[1] + expert * p.strideB[1] : B0;
    int a_row, a_chunk;
    dma_slot<Tile<MW>::ROWS, F_CONTIG, F_CONTIG>(wave, lane, a_row, a_chunk);
    int64_t m = min(m0 + a_row, m_end - 1);              // rows past the segment: valid memory, result unused
    if (GATHER) m = p.row_index[m];
    a.at = reinterpret_cast<const char *>(p.A[0] + m * p.lda) + a_chunk * 16;
    a.stride = KS * 4;
    a.jump = reinterpret_cast<const char *>(p.A[1]) - reinterpret_cast<const char *>(p.A[0]) - (steps - 1) * (KS * 4);
    a.back = max(a_chunk * 4 + 4 - left_in_tail, 0) * 4;
    const int64_t b_stride = BKIND == F_CONTIG ? KS * 4 : KS * 4 * p.ldb;
#pragma unroll
    for (int i = 0; i < B_LOADS; i++) {
        int r, ch;
        dma_slot<TN, F_CONTIG, BKIND>(wave * B_LOADS + i, lane, r, ch);
        b[i].stride = b_stride;
        b[i].jump = reinterpret_cast<const char *>(B1) - reinterpret_cast<const char *>(B0) - (steps - 1) * b_stride;
        if (BKIND == F_CONTIG) {
            const int n = min(n0 + (EPI == E_SWIGLU ? r & 31 : r), p.n_cols - 1);
            b[i].at = reinterpret_cast<const char *>((EPI == E_SWIGLU && r >= 32 ? B1 : B0) + static_cast<int64_t>(n) * p.ldb) + ch * 16;
            b[i].back = max(ch * 4 + 4 - left_in_tail, 0) * 4;
            b_past[i] = ch * 4 >= left_in_tail;
        } else {
            b[i].at = reinterpret_cast<const char *>(B0 + static_cast<int64_t>(r) * p.ldb + min(n0 + ch * 4, p.n_cols - 4));
            b[i].back = static_cast<uint32_t>(max(r - (left_in_tail - 1), 0)) * static_cast<uint32_t>(p.ldb) * 4u;
            b_past[i] = r >= left_in_tail;
        }
    }
    int at = 0;                                          // the step of the phase that is loaded next
    auto mask = [&]() -> uint32_t { return at == tail ? ~0u : 0u; };
    auto load_a = [&]() { return a.address(mask()); };
    auto load_b = [&](int i) { return b[i].address(mask()); };
    auto advance = [&]() {
        const bool wraps = at + 1 == steps;
        a.next(wraps);
#pragma unroll
        for (int i = 0; i < B_LOADS; i++) b[i].next(wraps);
        at = wraps ? 0 : at + 1;
    };
    auto tail_of = [&](int t) { return tail >= 0 && (t == tail || t - steps == tail); };
    f32x16 acc;
    multiply<MW, F_CONTIG, BKIND>(lds, steps * p.phases, load_a, load_b, advance, tail_of, a_chunk * 4 >= left_in_tail, b_past, acc);
    finish<MW>(lds, acc);
    // 8 threads to a row: 8 neighbouring columns each (E_SWIGLU: 4 of gate and the same 4 of up)
    const int part = threadIdx.x & 7, row = threadIdx.x >> 3, n = n0 + part * (EPI == E_SWIGLU ? 4 : 8);
    if (m0 + row < m_end && n < p.n_cols) {
        const int64_t o = static_cast<int64_t>(m0 + row) * p.ldc + n;
        if (EPI == E_SWIGLU) {
            const f4 g = finished<MW>(lds, row, part * 4), u = finished<MW>(lds, row, 32 + part * 4);
            f4 h;
#pragma unroll
            for (int j = 0; j < 4; j++) h[j] = (g[j] / (1.0f + expf(-g[j]))) * u[j];
            *reinterpret_cast<f4 *>(p.C[0] + o) = g;
            *reinterpret_cast<f4 *>(p.C[1] + o) = u;
            *reinterpret_cast<f4 *>(p.C[2] + o) = h;
            return;
        }
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const f4 v = finished<MW>(lds, row, part * 8 + q * 4);
            if (EPI == E_SWIGLU_BWD) {
                const f4 a = *reinterpret_cast<const f4 *>(p.G + o + q * 4), b = *reinterpret_cast<const f4 *>(p.U + o + q * 4);
                f4 og, ou;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float sg = 1.0f / (1.0f + expf(-a[j]));
                    ou[j] = v[j] * (a[j] / (1.0f + expf(-a[j])));
                    og[j] = (v[j] * b[j]) * (sg * (1.0f + a[j] * (1.0f - sg)));
                }
                *reinterpret_cast<f4 *>(p.C[0] + o + q * 4) = og;
                *reinterpret_cast<f4 *>(p.C[1] + o + q * 4) = ou;
            } else {
                *reinterpret_cast<f4 *>(p.C[0] + o + q * 4) = v;
            }
        }
    }
}

// One tile of a weight gradient: 32 * MW rows and 64 columns of dW[set][expert]
template <int MW>
__device__ __forceinline__ void wgrad_tile(const F32Wgrad &p, char *lds, int *idx_cache, int set_id, int expert, int row_tile, int col_tile) {
    const int r0 = p.cum[expert], len = p.cum[expert + 1] - r0;
    const int n_rows = p.n[set_id], n_cols = p.k[set_id];
    const int n0 = row_tile * Tile<MW>::ROWS, k0 = col_tile * TN;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int32_t *b_rows = p.b_rows[set_id];
    if (b_rows) {
        for (int i = threadIdx.x; i < min(len, IDX_CACHE); i += Tile<MW>::THREADS) idx_cache[i] = b_rows[r0 + i];
        __syncthreads();
    }
    // columns past the extent re-read its last 4; rows past the segment its last row (zeroed in LDS)
    constexpr int B_LOADS = Tile<MW>::B_LOADS;
    const int steps = (len + KS - 1) / KS, tail = len % KS ? steps - 1 : -1;
    const int left_in_tail = len - (steps - 1) * KS;     // rows in the last step
    Source a, b[B_LOADS];
    int a_c, b_c[B_LOADS];
    bool b_past[B_LOADS];
    auto set = [&](Source &s, const float *base, int ld, int c, int col) {
        s.at = reinterpret_cast<const char *>(base + static_cast<int64_t>(c) * ld + min(col, ld - 4));
        s.stride = s.jump = static_cast<int64_t>(KS) * ld * 4;
        s.back = static_cast<uint32_t>(max(c - (left_in_tail - 1), 0)) * static_cast<uint32_t>(ld) * 4u;
    };
    int chunk;
    dma_slot<Tile<MW>::ROWS, F_STRIDED, F_STRIDED>(wave, lane, a_c, chunk);
    set(a, p.A[set_id] + static_cast<int64_t>(r0) * n_rows, n_rows, a_c, n0 + chunk * 4);
#pragma unroll
    for (int i = 0; i < B_LOADS; i++) {
        dma_slot<TN, F_STRIDED, F_STRIDED>(wave * B_LOADS + i, lane, b_c[i], chunk);
        b_past[i] = b_c[i] >= left_in_tail;
        set(b[i], p.B[set_id] + (b_rows ? 0 : static_cast<int64_t>(r0) * n_cols), n_cols, b_rows ? 0 : b_c[i], k0 + chunk * 4);
    }
    int at = 0;
    auto mask = [&]() -> uint32_t { return at == tail ? ~0u : 0u; };
    auto load_a = [&]() { return a.address(mask()); };
    auto load_b = [&](int i) -> const char * {
        if (!b_rows) return b[i].address(mask());
        int r = min(at * KS + b_c[i], len - 1);
        if (at * KS + KS <= IDX_CACHE) {
            r = idx_cache[r];
        } else {   // (waited for here: at the join the compiler would wait for the direct loads too, on either path)
            r = b_rows[r0 + r];
            asm volatile("" : "+v"(r));
        }
        return b[i].at + static_cast<int64_t>(r) * n_cols * 4;
    };
    auto advance = [&]() {
        a.next(false);
#pragma unroll
        for (int i = 0; i < B_LOADS; i++)
            if (!b_rows) b[i].next(false);
        at++;
    };
    auto tail_of = [&](int t) { return t == tail; };
    f32x16 acc;
    multiply<MW, F_STRIDED, F_STRIDED>(lds, steps, load_a, load_b, advance, tail_of, a_c >= left_in_tail, b_past, acc);
    finish<MW>(lds, acc);
    const bool add = (p.accumulate >> set_id) & 1;
    const int row = threadIdx.x >> 3, k = k0 + (threadIdx.x & 7) * 8;
    if (n0 + row < n_rows && k < n_cols) {
        f4 *dst = reinterpret_cast<f4 *>(p.C[set_id] + expert * p.strideC[set_id] + static_cast<int64_t>(n0 + row) * n_cols + k);
#pragma unroll
        for (int q = 0; q < 2; q++) {
            f4 v = finished<MW>(lds, row, (threadIdx.x & 7) * 8 + q * 4);
            if (add) v += dst[q];
            dst[q] = v;
        }
    }
}

// Tiles in the order of the block ids, the column tiles of a row tile side by side; the ids past the last row tile, of
// which there are as many as the bound on the row tiles is too high, come last and find nothing.
// (second launch bound: the wavefronts per SIMD of the blocks that fit a CU's LDS, three of MW 1 or two of MW 2)
template <int MW, int BKIND, int EPI, bool GATHER>
__global__ __launch_bounds__(Tile<MW>::THREADS, MW == 1 ? 3 : 4) void ggemm_f32_rows_kernel(const F32Params p, int n_tiles) {
    __shared__ __attribute__((aligned(1024))) char lds[SLOTS * Tile<MW>::SLOT];
    rows_tile<MW, BKIND, EPI, GATHER>(p, lds, blockIdx.x / n_tiles, blockIdx.x % n_tiles);
}

template <int MW> __device__ __forceinline__ void wgrad_block(const F32Wgrad &w, char *lds, int *idx_cache, int id) {
    auto tiles_up = [](int v, int tile) { return (v + tile - 1) / tile; };
    int tk = tiles_up(w.k[0], TN), tn = tiles_up(w.n[0], Tile<MW>::ROWS), set = 0;
    const int first = tk * tn * w.n_experts;
    if (w.sets > 1 && id >= first) {   // (set 0 may be the down projection, whose extents are the other two's swapped)
        tk = tiles_up(w.k[1], TN); tn = tiles_up(w.n[1], Tile<MW>::ROWS);
        id -= first;
        set = 1 + id / (tk * tn * w.n_experts);
        id %= tk * tn * w.n_experts;
    }
    const int expert = id / (tk * tn), tile = id - expert * (tk * tn);
    wgrad_tile<MW>(w, lds, idx_cache, set, expert, tile / tk, tile % tk);
}
template <int MW> __global__ __launch_bounds__(Tile<MW>::THREADS, MW == 1 ? 3 : 4) void ggemm_f32_wgrad_kernel(const F32Wgrad w) {
    __shared__ __attribute__((aligned(1024))) char lds[SLOTS * Tile<MW>::SLOT];
    __shared__ int idx_cache[IDX_CACHE];
    wgrad_block<MW>(w, lds, idx_cache, blockIdx.x);
}
// dx = dg W_gate + du W_up and the three weight gradients: independent of each other, so that their tiles fill the chip
// together.  The input gradient's tiles, whose contraction is the longest, come first.
template <int MW>
__global__ __launch_bounds__(Tile<MW>::THREADS, MW == 1 ? 3 : 4) void ggemm_f32_backward_kernel(const F32Params p, const F32Wgrad w,
                                                                                                int row_blocks, int n_tiles) {
    __shared__ __attribute__((aligned(1024))) char lds[SLOTS * Tile<MW>::SLOT];
    __shared__ int idx_cache[IDX_CACHE];
    const int id = blockIdx.x;
    if (id < row_blocks) rows_tile<MW, F_STRIDED, E_STORE, false>(p, lds, id / n_tiles, id % n_tiles);
    else wgrad_block<MW>(w, lds, idx_cache, id - row_blocks);
}

inline bool mult8(int64_t v) { return v > 0 && v % 8 == 0; }
inline int64_t tiles_of(int64_t v, int tile) { return (v + tile - 1) / tile; }
inline bool fits31(int64_t v) { return v >= 0 && v < (1LL << 31); }

// blocks of a forward / input-gradient launch of tiles of `tile_rows` rows
int64_t rows_blocks(const F32Params &p, int64_t rows, int cols, int tile_rows) {
    return (tiles_of(rows, tile_rows) + p.n_experts) * tiles_of(p.n_cols, cols);
}
// 64-row tiles or 32-row ones, by the rounds that the busiest CU has (an expert's last tile is partly empty): half tiles cost
// a little more than half.  dx of the tiny layer with 520 rows an expert, about 276 tiles or 536 half ones on 256 CUs,
// 41 and 34 us; with 1024 rows 43 and 47; with 64, one round either way, 22 and 16.
bool two_high(int64_t tiles, int64_t half_tiles) {
    return 100 * ((tiles + 255) / 256) <= 56 * ((half_tiles + 255) / 256);
}
template <int MW, int BKIND, int EPI> int rows_launch(const F32Params &p, int64_t blocks, int n_tiles, void *stream) {
    if (blocks > 0x7fffffffLL) return OM_ERR_SHAPE;
    const dim3 grid(static_cast<unsigned>(blocks)), block(Tile<MW>::THREADS);
    if (p.row_index) ggemm_f32_rows_kernel<MW, BKIND, EPI, true><<<grid, block, 0, om_stream(stream)>>>(p, n_tiles);
    else ggemm_f32_rows_kernel<MW, BKIND, EPI, false><<<grid, block, 0, om_stream(stream)>>>(p, n_tiles);
    return om_launch_status();
}
template <int BKIND, int EPI> int rows_launch(const F32Params &p, int64_t rows, void *stream) {
    constexpr int COLS = EPI == E_SWIGLU ? TN / 2 : TN;
    const int n_tiles = static_cast<int>(tiles_of(p.n_cols, COLS));
    const int64_t partial = std::min<int64_t>(rows, p.n_experts) / 2;
    return two_high((tiles_of(rows, 64) + partial) * n_tiles, (tiles_of(rows, 32) + partial) * n_tiles)
               ? rows_launch<2, BKIND, EPI>(p, rows_blocks(p, rows, COLS, 64), n_tiles, stream)
               : rows_launch<1, BKIND, EPI>(p, rows_blocks(p, rows, COLS, 32), n_tiles, stream);
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

namespace {
// dx = dg W_gate + du W_up, one accumulation over both
int gate_up_dgrad_params(F32Params &p, const float *dg, const float *du, const float *w_gate, const float *w_up, float *dx,
                         const int32_t *cum_token_counts, int64_t rows, int G, int I, int H, int64_t gate_stride,
                         int64_t up_stride) {
    if (!dg || !du || !w_gate || !w_up || !dx || !cum_token_counts) return OM_ERR_NULL;
    if (!om_aligned16(dg) || !om_aligned16(du) || !om_aligned16(w_gate) || !om_aligned16(w_up) || !om_aligned16(dx))
        return OM_ERR_ALIGN;
    p.A[0] = dg; p.A[1] = du; p.B[0] = w_gate; p.B[1] = w_up; p.C[0] = dx; p.cum = cum_token_counts;
    p.lda = I; p.ldb = H; p.ldc = H;
    p.strideB[0] = gate_stride ? gate_stride : static_cast<int64_t>(I) * H;
    p.strideB[1] = up_stride ? up_stride : static_cast<int64_t>(I) * H;
    if (p.strideB[0] % 4 != 0 || p.strideB[1] % 4 != 0) return OM_ERR_ALIGN;
    if (!fits31(rows * H) || !fits31(rows * I) || !fits31(p.strideB[0] * G) || !fits31(p.strideB[1] * G)) return OM_ERR_SHAPE;
    p.n_experts = G; p.n_cols = H; p.kc = I; p.phases = 2;
    return OM_OK;
}
}  // namespace

extern "C" int om_merged_mlp_gate_up_dgrad_f32(const float *dg, const float *du, const float *w_gate, const float *w_up,
                                               float *dx, const int32_t *cum_token_counts, int64_t rows, int G, int I,
                                               int H, int64_t gate_stride, int64_t up_stride, void *stream) {
    if (rows < 0 || G < 1 || !mult8(I) || !mult8(H)) return OM_ERR_SHAPE;
    if (rows == 0) return OM_OK;
    F32Params p = {};
    const int code = gate_up_dgrad_params(p, dg, du, w_gate, w_up, dx, cum_token_counts, rows, G, I, H, gate_stride, up_stride);
    return code == OM_OK ? rows_launch<F_STRIDED, E_STORE>(p, rows, stream) : code;
}

namespace {
// Checks one weight gradient and enters it as set s.
int wgrad_set(F32Wgrad &w, int s, const float *dout, const float *in, const int32_t *in_rows, int64_t src_rows, float *dw,
              int64_t stride, int64_t rows, int G, int N, int K) {
    if (!dw || (rows > 0 && (!dout || !in))) return OM_ERR_NULL;
    if (!om_aligned16(dout) || !om_aligned16(in) || !om_aligned16(dw)) return OM_ERR_ALIGN;
    w.A[s] = dout; w.B[s] = in; w.C[s] = dw; w.b_rows[s] = in_rows;
    w.n[s] = N; w.k[s] = K;
    w.strideC[s] = stride ? stride : static_cast<int64_t>(N) * K;
    if (w.strideC[s] % 4 != 0) return OM_ERR_ALIGN;
    if (!fits31(w.strideC[s] * G) || !fits31((in_rows ? src_rows : rows) * K) || !fits31(rows * N)) return OM_ERR_SHAPE;
    return OM_OK;
}
// Whether the gradients of two sets have memory in common (their weights are one parameter): they are then written, or added
// to, in launches one after another.
bool wgrad_sets_overlap(const F32Wgrad &w) {
    for (int a = 0; a < w.sets; a++)
        for (int b = a + 1; b < w.sets; b++)
            if (om_blocks_overlap(w.C[a], w.strideC[a] * 4, 4 * static_cast<int64_t>(w.n[a]) * w.k[a], w.C[b], w.strideC[b] * 4,
                                  4 * static_cast<int64_t>(w.n[b]) * w.k[b], w.n_experts))
                return true;
    return false;
}
int64_t wgrad_blocks(const F32Wgrad &w, int tile_rows) {
    int64_t blocks = 0;
    for (int s = 0; s < w.sets; s++) blocks += tiles_of(w.n[s], tile_rows) * tiles_of(w.k[s], TN) * w.n_experts;
    return blocks;
}

// Weight gradients over the same rows times experts that are accepted: what these entry points refuse, not a bound of the
// launch (`blocks` is that).  The whole backward takes the experts that its gate and up gradients take.
constexpr int64_t MAX_GRADIENTS = 65535;

// n_sets 1 or 2: dW[s] (+)= dout[s]^T in, over the same rows of `input` (through input_rows when given)
int wgrad_f32_launch(int n_sets, const float *const *output_grad, const float *input, const int32_t *input_rows,
                     int64_t src_rows, float *const *weight_grad, const int32_t *cum_token_counts, int64_t rows, int G,
                     int N, int K, const int64_t *w_stride, void *stream, int accumulate) {
    if (rows < 0 || G < 1 || n_sets * static_cast<int64_t>(G) > MAX_GRADIENTS || !mult8(N) || !mult8(K)) return OM_ERR_SHAPE;
    if (!cum_token_counts) return OM_ERR_NULL;
    F32Wgrad w = {};
    for (int s = 0; s < n_sets; s++) {
        const int code = wgrad_set(w, s, output_grad[s], input, input_rows, src_rows, weight_grad[s], w_stride[s], rows, G, N, K);
        if (code != OM_OK) return code;
    }
    w.cum = cum_token_counts; w.n_experts = G; w.sets = n_sets; w.accumulate = accumulate;
    if (wgrad_sets_overlap(w)) {
        for (int s = 0; s < n_sets; s++) {
            const int code = wgrad_f32_launch(1, output_grad + s, input, input_rows, src_rows, weight_grad + s, cum_token_counts, rows, G,
                                              N, K, w_stride + s, stream, (accumulate >> s) & 1);
            if (code != OM_OK) return code;
        }
        return OM_OK;
    }
    const bool high = two_high(wgrad_blocks(w, 64), wgrad_blocks(w, 32));
    const int64_t blocks = wgrad_blocks(w, high ? 64 : 32);
    if (blocks > 0x7fffffffLL) return OM_ERR_SHAPE;
    const dim3 grid(static_cast<unsigned>(blocks));
    if (high) ggemm_f32_wgrad_kernel<2><<<grid, dim3(Tile<2>::THREADS), 0, om_stream(stream)>>>(w);
    else ggemm_f32_wgrad_kernel<1><<<grid, dim3(Tile<1>::THREADS), 0, om_stream(stream)>>>(w);
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

namespace {
int backward_f32_launch(const float *dy, const float *h, const float *dg, const float *du, const float *x, const int32_t *x_rows,
                        int64_t src_rows, const float *w_gate, const float *w_up, float *dx, float *dw_down, float *dw_gate,
                        float *dw_up, const int32_t *cum_token_counts, int64_t rows, int G, int I, int H, int64_t gate_stride,
                        int64_t up_stride, int64_t dw_down_stride, int64_t dw_gate_stride, int64_t dw_up_stride, bool accumulate,
                        void *stream) {
    if (rows < 0 || G < 1 || 2 * static_cast<int64_t>(G) > MAX_GRADIENTS || !mult8(I) || !mult8(H)) return OM_ERR_SHAPE;
    if (x_rows && rows > 0 && src_rows < 1) return OM_ERR_SHAPE;
    if (!cum_token_counts) return OM_ERR_NULL;
    F32Params p = {};
    F32Wgrad w = {};
    int code = rows == 0 ? OM_OK : gate_up_dgrad_params(p, dg, du, w_gate, w_up, dx, cum_token_counts, rows, G, I, H, gate_stride, up_stride);
    if (code == OM_OK) code = wgrad_set(w, 0, dy, h, nullptr, 0, dw_down, dw_down_stride, rows, G, H, I);
    if (code == OM_OK) code = wgrad_set(w, 1, dg, x, x_rows, src_rows, dw_gate, dw_gate_stride, rows, G, I, H);
    if (code == OM_OK) code = wgrad_set(w, 2, du, x, x_rows, src_rows, dw_up, dw_up_stride, rows, G, I, H);
    if (code != OM_OK) return code;
    w.cum = cum_token_counts; w.n_experts = G; w.sets = 3; w.accumulate = accumulate ? 7 : 0;
    if (wgrad_sets_overlap(w)) {
        const float *dout[2] = {dg, du};
        float *dw[2] = {dw_gate, dw_up};
        const int64_t strides[2] = {dw_gate_stride, dw_up_stride};
        if (rows > 0) code = rows_launch<F_STRIDED, E_STORE>(p, rows, stream);
        if (code == OM_OK) code = wgrad_f32_launch(1, &dy, h, nullptr, 0, &dw_down, cum_token_counts, rows, G, H, I, &dw_down_stride, stream, accumulate);
        if (code == OM_OK) code = wgrad_f32_launch(2, dout, x, x_rows, src_rows, dw, cum_token_counts, rows, G, I, H, strides, stream, accumulate ? 3 : 0);
        return code;
    }
    const int n_tiles = rows > 0 ? static_cast<int>(tiles_of(p.n_cols, TN)) : 1;
    auto row_blocks = [&](int tile_rows) { return rows > 0 ? rows_blocks(p, rows, TN, tile_rows) : 0; };
    // 64-row tiles unless the input gradient's few long ones would be the last to end: the tiny layer with 64 rows an expert
    // (32 such tiles) 25 us and 20 with half tiles, 128 rows 27 and 24, 256 rows 37 and 38, 1024 rows 110 and 124
    const bool high = tiles_of(rows, 64) * n_tiles > 64;
    const int64_t first = row_blocks(high ? 64 : 32), blocks = first + wgrad_blocks(w, high ? 64 : 32);
    if (blocks > 0x7fffffffLL) return OM_ERR_SHAPE;
    const dim3 grid(static_cast<unsigned>(blocks));
    if (high) ggemm_f32_backward_kernel<2><<<grid, dim3(Tile<2>::THREADS), 0, om_stream(stream)>>>(p, w, static_cast<int>(first), n_tiles);
    else ggemm_f32_backward_kernel<1><<<grid, dim3(Tile<1>::THREADS), 0, om_stream(stream)>>>(p, w, static_cast<int>(first), n_tiles);
    return om_launch_status();
}
}  // namespace

extern "C" int om_grouped_gemm_wgrad_merged_dgrad_f32(const float *dy, const float *h, const float *dg,
                                                      const float *du, const float *x, const int32_t *x_rows,
                                                      int64_t src_rows, const float *w_gate, const float *w_up,
                                                      float *dx, float *dw_down, float *dw_gate, float *dw_up,
                                                      const int32_t *cum_token_counts, int64_t rows, int G, int I,
                                                      int H, int64_t gate_stride, int64_t up_stride,
                                                      int64_t dw_down_stride, int64_t dw_gate_stride,
                                                      int64_t dw_up_stride, void *stream) {
    return backward_f32_launch(dy, h, dg, du, x, x_rows, src_rows, w_gate, w_up, dx, dw_down, dw_gate, dw_up,
                               cum_token_counts, rows, G, I, H, gate_stride, up_stride, dw_down_stride, dw_gate_stride,
                               dw_up_stride, false, stream);
}

extern "C" int om_grouped_gemm_wgrad_merged_dgrad_f32_accumulate(const float *dy, const float *h, const float *dg,
                                                                 const float *du, const float *x,
                                                                 const int32_t *x_rows, int64_t src_rows,
                                                                 const float *w_gate, const float *w_up, float *dx,
                                                                 float *dw_down, float *dw_gate, float *dw_up,
                                                                 const int32_t *cum_token_counts, int64_t rows, int G,
                                                                 int I, int H, int64_t gate_stride, int64_t up_stride,
                                                                 int64_t dw_down_stride, int64_t dw_gate_stride,
                                                                 int64_t dw_up_stride, void *stream) {
    return backward_f32_launch(dy, h, dg, du, x, x_rows, src_rows, w_gate, w_up, dx, dw_down, dw_gate, dw_up,
                               cum_token_counts, rows, G, I, H, gate_stride, up_stride, dw_down_stride, dw_gate_stride,
                               dw_up_stride, true, stream);
}

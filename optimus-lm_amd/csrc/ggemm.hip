// Grouped expert GEMMs on bf16 MFMA (v_mfma_f32_16x16x32_bf16), fp32 accumulation.
//
// One kernel template covers every product of the merged MLP.  An output tile of 256x256 (8 wavefronts) or 128x128
// (4) is worked by a grid of wavefronts two high; each has 32 rows of a row unit and 64 columns, as 2 x 4 accumulators of
// 16x16.  Operands are
// staged through LDS in steps of 64 along the contraction index c with direct global->LDS loads
// (global_load_lds_dwordx4: no register staging, no ds_write), two stages.
//
// An operand is either
//   CONTIG  — stored [row][c] with c contiguous (activations in fwd/dgrad, weights in fwd):
//             fragments are one ds_read_b128 per lane;
//   STRIDED — stored [c][row] with row contiguous (weights in dgrad, both operands in wgrad):
//             fragments come from the gfx950 transposing LDS read (ds_read_b64_tr_b16), two per lane.
// A stage is made of units of 8 KB: 64 rows x 64 c with 128-byte rows (CONTIG), or 64 c x 64 rows with 128-byte c-rows
// (STRIDED), their 16-byte chunks XOR-permuted so that fragment reads meet no bank conflict.  A direct load writes LDS
// at (wave-uniform base + lane*16), so the permutation is applied by choosing which global chunk each lane fetches.
// The per-lane order of the 8 contraction indices is the same for both kinds, so they can be mixed in one MFMA.
//
// Main loop.  What bounds a step is how long its loads have to arrive.  With one barrier a step, that waits for all of
// them, they have 0.6 to 0.9 of a step, and a step of the 256x256 tile took 1.5 us at full clock where its MFMAs take
// 0.85; the 128x128 kernels, two blocks per CU, spent three quarters of their time waiting.  So a step's buffers are
// given back piecemeal.  A wavefront keeps all of its B fragments of a step in registers (64 c x 64 columns) and works
// through the row units of A one after the other (a phase: 16 MFMAs); it reads the fragments of the next phase, and in
// the later phases B of the next step, under the MFMAs of this one.  Two barriers a step, P in the middle and Q at its
// end, give the buffers back:
//   after Q(t-1)  B of step t was read during step t-1, as was A's first unit: both are free for step t+2, and
//                 (256x256) A's last unit for step t+1;
//   after P(t)    A's remaining units of step t are free for step t+2.
// 256x256: the loads go out evenly, one for every eight MFMAs: eight wavefronts that issue three each at once wait for one
// another's addresses, and the matrix cores for them.  (128x128: as soon as a buffer is free; few rows wait for weights, and
// evenly a decode batch of 37 took 155 us instead of 150.)  A wavefront passes P (Q) once all but its 6 (8; 128x128 8) youngest
// loads have landed, so every load has 1 to 1.5 steps.  The waits are written as assembly, and so are the loads: with the
// builtin the compiler waits for every load in flight before a barrier, since it cannot tell which LDS bytes they will write.
// Loads at a phase's start, six of a step's eight after Q -> evenly, us: 64 experts of 2048/1024 with 2048 rows, gate+up 950 ->
// 916, down 493 -> 477, gate/up input gradient 907 -> 883, weight gradients 1465 -> 1446 (added 1583 -> 1545); with 512 rows
// gate/up input gradient 250 -> 239; 32 experts of 7168/2048, 400 uneven rows, gate+up 847 -> 829, gate/up input gradient 829 ->
// 805.  (At full clock, on operands of zeros, one product of 8192^3 is slower: 700 -> 757.)
// Measured on one box against the single-barrier loop, us: 3001 tokens, hidden 1000, ffn 712, 12 experts, top-3
// (128x128): down 32.6 -> 28.6, gate/up input gradient 55.7 -> 46.8, weight gradients 34 -> 31; decode of 37 tokens,
// 64 experts of 2048/1024, 112.7 -> 104.4 and 57.0 -> 50.8 (that loop with its operands staged through registers two
// steps ahead); 32 experts of 7168/2048 with 0 to 2849 rows (256x256): gate+up 967 -> 859, gate/up input gradient 959
// -> 886; 64 experts of 2048/1024 with 2048 rows, where the power limit sets the rate, 1020 -> 1004 and 521 -> 518.
//
// The 16x16x32 instruction takes less energy per operation than 32x32x16 (alone, random operands, under the power limit
// 2.00 against 1.77 PFLOP/s), which is what the large launches are bound by; fragments and accumulators take as many
// registers, and the sums are the same bits.  Whole passes, us, 32x32x16 -> 16x16x32: 64 experts of 2048/1024, forward of
// 4096 tokens 522 -> 509, training step of 16384 5344 -> 5287; 32 experts of 7168/2048 and a shared one, 8192 tokens
// 6169 -> 6005.
//
// A tile's rows are worked in units of 64 (32 per wavefront row), and units past the expert's last row cost no MFMA.
//
// Variable rows per expert: the M extent of fwd/dgrad is cut into tiles per expert.  Each block
// scans the device-resident cum_token_counts once into an LDS table (row tiles up to and including
// each expert) and looks its (expert, row block) up there per tile, so no host copy of the counts
// and no max-rows-per-expert is needed, and the blocks share out the tiles that really exist.  In wgrad the rows are the
// contraction range of expert g; rows past its end are zero-filled in LDS.
//
// Block order: consecutive block ids go to different XCDs (8 per chip, each with its own L2), so
// block ids are remapped to give every XCD a contiguous run of tiles, which share operand tiles, or, with large experts,
// a part of each expert (GemmParams::share).
//
// Two things that surround the expert GEMMs in the layer are folded into them (template parameters
// GATHER and ROWW): the token gather (an operand's rows are fetched through an index: the A rows of
// fwd/dgrad, or the contraction rows of either operand in wgrad), and the routing weight of the
// combine (the SwiGLU epilogue scales h by the weight of its row; the SwiGLU-backward epilogue
// scales dh by it and produces the per-row sums that make up the weight's gradient).
#include "common.h"
#include <type_traits>

namespace {

enum { CONTIG = 0, STRIDED = 1 };
// An operand's rows can be taken through an index instead of in order: the token gather that
// precedes the expert GEMMs (ggemm_input = hidden_states[input_indices]) folded into the loads.
enum {
    GATHER_NONE = 0,
    GATHER_A = 1,    // fwd/dgrad: A rows
    GATHER_B = 2,    // wgrad: contraction rows of B
    GATHER_WA = 3,   // wgrad: contraction rows of A
    MERGED = 4       // the three weight gradients of a merged MLP in one launch (see WgradSet)
};
enum {
    EPI_STORE = 0,        // C = acc
    EPI_SWIGLU = 1,       // even 32-col accumulators = gate, odd = up: store g, u, h
    EPI_SWIGLU_BWD = 2,   // acc = dh: read g,u, store dg, du
    EPI_WGRAD = 3         // C[g] = acc, no row masking
};

constexpr int BK = 64;  // contraction step, elements
constexpr int NUM_XCD = 8;

// MERGED: one weight gradient C[e] (+)= A^T B over expert e's rows; A [rows, m], B [rows, n], C [m, n] per expert.
struct WgradSet {
    const uint16_t *A, *B;
    uint16_t *C;
    const int32_t *a_rows, *b_rows;   // at most one not null: rows taken through an index
    int64_t strideC;
    int m, n;
};

// DENSE: one more expert behind the others, with operands and outputs of its own and all of its rows known to the host (the
// shared expert beside a window of routed ones).  Its rows are not taken through an index and have the weight 1.
struct DenseExpert {
    const uint16_t *A[2], *B[2];
    uint16_t *C, *C1, *C2;
    const uint16_t *G, *U;
    int rows;
};

template <int BM> constexpr int WAVES_N = BM / 64;        // 256x256: 2 x 4 wavefronts, 128x128: 2 x 2
template <int BM> constexpr int THREADS = 2 * WAVES_N<BM> * 64;

struct GemmParams {
    // operands; for the two-phase products (gate+up) index 1 is the second pair
    const uint16_t *A[2];
    const uint16_t *B[2];
    uint16_t *C;         // EPI_STORE / EPI_WGRAD output;  EPI_SWIGLU: g ; EPI_SWIGLU_BWD: dg
    uint16_t *C1;        // EPI_SWIGLU: u ; EPI_SWIGLU_BWD: du
    uint16_t *C2;        // EPI_SWIGLU: h
    const uint16_t *G;   // EPI_SWIGLU_BWD: saved g
    const uint16_t *U;   // EPI_SWIGLU_BWD: saved u
    const int32_t *cum;  // [G+1] device
    const int32_t *row_index;   // GATHER_A: A row of sorted row r; GATHER_B / GATHER_WA: B / A row of contraction row c
    // ROWW kernels (the routing weight folded into the expert MLP):
    const float *row_scale;     // [rows] weight of each sorted row
    float *row_dot;             // EPI_SWIGLU_BWD: [n_cols / COLS][rows] partial sums of dh * silu(g) * u
    int64_t lda, ldb, ldc;      // leading dimensions, elements
    int64_t strideB, strideC;   // per-expert strides, elements
    int64_t rows;               // allocated activation rows (upper bound of cum[G])
    int n_experts;
    int n_cols;                 // output columns (fwd/dgrad) — tiles along N = n_cols / BN_OUT
    int kc;                     // contraction length per phase (fwd/dgrad), multiple of 8
    int phases;                 // 1 or 2
    int total_tiles;            // wgrad: tiles of the launch (the blocks loop over them)
    int tiles_e;                // wgrad: tiles per expert (MERGED: of all three)
    bool stream;                // wgrad: the gradients are stored past the caches (see CACHED_WEIGHTS)
    int share;                  // XCDs that share an expert's tiles; 0: contiguous runs of tiles per XCD
    WgradSet set[3];            // MERGED
    DenseExpert dense;          // DENSE
};

typedef __attribute__((address_space(3))) s16x4 *lds_s16x4_ptr;
typedef __attribute__((address_space(3))) void *lds_void_ptr;

// A block-uniform 64-bit value, pinned to scalar registers (the compiler cannot always prove that
// per-tile state carried around the tile loop is uniform).
__device__ __forceinline__ int64_t uniform64(int64_t v) {
    const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(static_cast<uint64_t>(v) >> 32));
    return static_cast<int64_t>((static_cast<uint64_t>(hi) << 32) | lo);
}

// One of two fields of the kernel's arguments.  Both are read: of a read on either side of a branch the compiler makes one through an
// address that it chooses, and then reads every argument where it is used instead of all of them, a few at a time, when the kernel starts.
// 128x128 tiles, us, so -> read together: 8 experts of 256/512, 4096 rows, gate+up 15.0 -> 14.5, down 13.2 -> 12.7, gate/up input gradient
// 19.0 -> 18.5; 12 of 1000/712, 9003 rows, down 34.0 -> 33.1, SwiGLU backward 38.0 -> 37.4, gate/up input gradient 54.9 -> 53.4; 64 of 2048/1024, 296
// rows, gate+up 88.9 -> 87.9, down 48.1 -> 47.0.
template <typename T> __device__ __forceinline__ T pick(bool first, T a, T b) { return first ? a : b; }

// CONTIG unit (64 rows x 64 c, 128-byte rows): chunk position = chunk ^ swz(row), conflict-free for ds_read_b128, whose
// lanes are served sixteen at a time, with 16 consecutive rows; period 16, so rows 16 apart share it.
__device__ __forceinline__ int swz(int row) { return (row >> 1) & 7; }
// STRIDED unit (64 c-rows x 64 columns, 128-byte c-rows): a transposing read takes 32 bytes of four c-rows for every 16
// lanes, of c-rows 8 apart for the next 16; the eight pieces land in eight different 32-byte windows of the banks
__device__ __forceinline__ int unit_swz(int crow) { return (((crow >> 1) & 1) << 2) | (((crow >> 3) & 1) << 1); }

__device__ __forceinline__ uint32_t pack2_bf16(float a, float b) {
    typedef __attribute__((ext_vector_type(2))) float f32x2;
    f32x2 f = {a, b};
    bf16x2 h = __builtin_convertvector(f, bf16x2);
    return __builtin_bit_cast(uint32_t, h);
}

// Sum over aligned groups of eight neighbouring lanes; every lane of the group gets it.  DPP: swap within pairs, swap
// pairs within quads, mirror within 8.
template <int CTRL> __device__ __forceinline__ float dpp_move(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float eight_lanes_sum(float v) {
    v += dpp_move<0xB1>(v);
    v += dpp_move<0x4E>(v);
    return v + dpp_move<0x141>(v);
}

// Row tiles of fwd/dgrad are cut per expert (BM rows each, the last one of an expert partial).
// One wavefront builds, once per block, a table in LDS from the device-resident cum_token_counts:
// tile_end[e] = number of row tiles of experts 0..e, seg[e] = cum_token_counts[e].
constexpr int MAX_EXPERTS = 1024;
template <int BM>
__device__ __forceinline__ void build_tile_table(const int32_t *cum, int n_experts, int lane,
                                                 int *tile_end, int *seg) {
    int base_tiles = 0;
    for (int e0 = 0; e0 < n_experts; e0 += 64) {
        const int e = e0 + lane;
        int s = 0, cnt = 0;
        if (e < n_experts) { s = cum[e]; cnt = cum[e + 1] - s; }
        int incl = (cnt + BM - 1) / BM;  // inclusive scan over the wavefront
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(incl, o, 64);
            if (lane >= o) incl += v;
        }
        if (e < n_experts) {
            tile_end[e] = base_tiles + incl;
            seg[e] = s;
            if (e == n_experts - 1) seg[n_experts] = s + cnt;
        }
        base_tiles += __shfl(incl, 63, 64);
    }
}

// Which expert owns row tile `tile`, and which rows are the tile's?  False past the last tile.
template <int BM>
__device__ __forceinline__ bool find_tile(const int *tile_end, const int *seg, int n_experts, int tile,
                                          int lane, int &expert, int &row_begin, int &row_end) {
    for (int e0 = 0; e0 < n_experts; e0 += 64) {
        const int e = e0 + lane;
        const bool mine = e < n_experts && tile < tile_end[e];   // tile_end is non-decreasing
        const unsigned long long vote = __ballot(mine);
        if (vote) {
            expert = e0 + __ffsll(static_cast<long long>(vote)) - 1;
            const int first = expert > 0 ? tile_end[expert - 1] : 0;
            row_begin = seg[expert] + (tile - first) * BM;
            row_end = seg[expert + 1];
            return true;
        }
    }
    return false;
}

// Launches with large experts (p.share != 0) share each expert among several XCDs.  An expert of many tiles, XCD by XCD, would
// keep one XCD busy for several rounds of its blocks, all of them multiplying (many rows) or all of them moving the
// weights (few), and those with the few-row experts are then bound by what one XCD can load or store.
// So the experts are taken in the order of their rows; `share` XCDs have each a part of every expert of a group; with
// two or more groups (share < 8) the experts go to them to and fro; and a part is neighbouring columns of tiles along the longer
// extent (row products: the columns of the weight matrix, which its part of the weights then crosses once).
// The rounds run over the XCD's blocks to and fro as well, so that the sums of a block's tiles differ little.
// us, contiguous runs of equal work per XCD -> shared, 32 experts of 2048/7168.  12510 rows, between 0 and 2663 an expert (in a
// training pass): gate+up 865 -> 792, down 431 -> 415, SwiGLU backward 541 -> 437, gate/up input gradient 908 -> 789,
// accumulating weight gradients 715 -> 590.  Alone, rows as 1 / rank with mean 64 / 512 / 2048, even rows with mean 512 / 2048:
// gate+up 490 -> 422, 1001 -> 1027, 3619 -> 3565, 796 -> 835, 3312 -> 2992; gate/up input gradient 548 -> 432, 1071 -> 1020,
// 3771 -> 3588, 916 -> 821, 3674 -> 3100; SwiGLU backward 287 -> 277, 566 -> 562, 1817 -> 1943, 427 -> 438, 1630 -> 1647; weight
// gradients, writing 224 -> 245, 688 -> 570, 1936 -> 1736, 529 -> 544, 1770 -> 1668, accumulating 444 -> 399, 757 -> 689, 2069 -> 1821,
// 676 -> 664, 1920 -> 1787.  Smaller experts lose what they share in the caches: 64 of 1024/2048, even, 512 rows,
// four XCDs, gate+up 257 -> 269, all eight 307; the weight gradients, one round of an XCD each, 170 -> 179 and 205.  Nor is
// it better to mix experts of many and of few rows in time: alternating them, weight gradients 590 -> 670.
constexpr int SHARE_MAX_EXPERTS = 256;
// order[i]: the expert with the i-th most rows.  The whole block, with a barrier at the end.
__device__ __forceinline__ void expert_order(const int32_t *cum, int n_experts, int tid, int lane, int *order) {
    static_assert(SHARE_MAX_EXPERTS <= THREADS<128>, "a thread per expert");
    if (tid - lane < n_experts) {
        const int e = min(tid, n_experts - 1), mine = cum[e + 1] - cum[e];
        int rank = 0;
        for (int j0 = 0; j0 < n_experts; j0 += 64) {
            const int j = min(j0 + lane, n_experts - 1), rows = j0 + lane < n_experts ? cum[j + 1] - cum[j] : -1;
#pragma unroll 16
            for (int l = 0; l < 64; l++) {
                const int other = __builtin_amdgcn_readlane(rows, l);
                rank += other > mine || (other == mine && j0 + l < e) ? 1 : 0;
            }
        }
        if (tid < n_experts) order[rank] = e;
    }
    __syncthreads();
}
// First tile of the part of an XCD in the i-th expert of `order`; where `share` does not divide them the XCDs take turns
// with the odd ones.
__device__ __forceinline__ int part_begin(int tiles, int i, int member, int share) {
    return (member * tiles + (i * 5 & (share - 1))) / share;
}
// An expert of `order` as an XCD sees it: its rows, and what turns the XCD's tile number into the expert's.
struct Part { int expert, row_begin, row_end, shift; };
// part[i], and tile_end[i] = number of tiles, of the first i + 1 experts in `order`, that are this XCD's.  tiles_of(rows): of an expert.  One wavefront.
template <typename TILES>
__device__ __forceinline__ void build_part_table(const int32_t *cum, const int *order, int n_experts, int share, int xcd, int lane,
                                                 TILES tiles_of, int *tile_end, Part *part) {
    const int groups = NUM_XCD / share, member = xcd % share;
    int base_tiles = 0;
    for (int i0 = 0; i0 < n_experts; i0 += 64) {
        const int i = i0 + lane, there = i % groups, group = (i / groups) & 1 ? groups - 1 - there : there;
        const int e = order[min(i, n_experts - 1)];
        int begin = cum[e], end = cum[e + 1];
        asm volatile("" : "+v"(begin), "+v"(end));   // waited for here: around their use the compiler would wait for them, and all else, in every tile
        const int tiles = tiles_of(end - begin);
        const int first = part_begin(tiles, i, member, share);
        const int mine = i < n_experts && group == xcd / share ? part_begin(tiles, i, member + 1, share) - first : 0;
        int incl = mine;
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(incl, o, 64);
            if (lane >= o) incl += v;
        }
        if (i < n_experts) {
            tile_end[i] = base_tiles + incl;
            part[i] = {e, begin, end, first - (base_tiles + incl - mine)};
        }
        base_tiles += __shfl(incl, 63, 64);
    }
}
// first[e]: row tiles of the experts before e.  One wavefront.
template <int BM> __device__ __forceinline__ void build_first_tiles(const int32_t *cum, int n_experts, int lane, int *first) {
    int base_tiles = 0;
    for (int e0 = 0; e0 < n_experts; e0 += 64) {
        const int e = min(e0 + lane, n_experts - 1), tiles = e0 + lane < n_experts ? (cum[e + 1] - cum[e] + BM - 1) / BM : 0;
        int incl = tiles;
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(incl, o, 64);
            if (lane >= o) incl += v;
        }
        if (e0 + lane < n_experts) first[e] = base_tiles + incl - tiles;
        base_tiles += __shfl(incl, 63, 64);
    }
}
// The part that tile `at` of the XCD (less than the last tile_end) belongs to.
__device__ __forceinline__ Part find_part(const int *tile_end, const Part *part, int n_experts, int lane, int at) {
    int i = 0;
    asm volatile("" : "+v"(lane));   // addresses recomputed per tile, not kept across the main loop
    for (int i0 = 0; i0 < n_experts; i0 += 64) {
        const unsigned long long vote = __ballot(i0 + lane < n_experts && at < tile_end[min(i0 + lane, n_experts - 1)]);
        if (vote) { i = i0 + __ffsll(static_cast<long long>(vote)) - 1; break; }
    }
    const Part p = part[__builtin_amdgcn_readfirstlane(i)];
    return {__builtin_amdgcn_readfirstlane(p.expert), __builtin_amdgcn_readfirstlane(p.row_begin),
            __builtin_amdgcn_readfirstlane(p.row_end), __builtin_amdgcn_readfirstlane(p.shift)};
}

// Weight gradient: the tiles of expert e cost about (contraction steps of e + a few steps' worth of
// epilogue) each, so with skewed routing equal tile counts per XCD are far from equal work.  The
// tiles are numbered expert-major; boundary j of 0..8 is the tile at which j/8 of the launch's work
// lies behind, and XCD x takes the run [boundary x, boundary x+1).  A boundary that falls within an
// eighth of an XCD's share of an expert's first or last tile moves there: all tiles of dW[g] share
// the expert's rows of both operands, and with near-uniform routing whole experts per XCD (what
// equal tile counts give) is the better cut.  Every wavefront computes the two boundaries it needs
// by itself from cum_token_counts (two strided passes, no LDS, no barrier).
constexpr int WGRAD_EPILOGUE_STEPS = 3;   // a tile's stores take about as long as 3 steps
constexpr int WGRAD_BALANCE_MAX_EXPERTS = 4096;
__device__ __forceinline__ int wgrad_tile_units(int rows, int bk) {
    const int steps = (rows + bk - 1) / bk;
    return steps + WGRAD_EPILOGUE_STEPS;
}
__device__ __forceinline__ void wgrad_xcd_run(const int32_t *cum, int n_experts, int tiles_e, int bk, int xcd,
                                              int n_xcd, int lane, int &lo, int &hi) {
    int mine = 0;
    for (int e = lane; e < n_experts; e += 64) mine += wgrad_tile_units(cum[e + 1] - cum[e], bk);
    const long long work = static_cast<long long>(wave_sum_i(mine)) * tiles_e;
    const long long t_lo = work * xcd / n_xcd, t_hi = work * (xcd + 1) / n_xcd;
    lo = 0;
    hi = n_experts * tiles_e;
    int base = 0;   // units of the experts before this chunk
    for (int e0 = 0; e0 < n_experts; e0 += 64) {
        const int e = e0 + lane;
        const int u = e < n_experts ? wgrad_tile_units(cum[e + 1] - cum[e], bk) : 0;
        int incl = u;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(incl, o, 64);
            if (lane >= o) incl += v;
        }
        const long long before = static_cast<long long>(base + incl - u) * tiles_e;
        const long long after = before + static_cast<long long>(u) * tiles_e;
        // exactly one expert of the launch holds a target below the total; the total itself
        // (boundary n_xcd) keeps the initial value of hi
        const bool has_lo = u > 0 && t_lo >= before && t_lo < after;
        const bool has_hi = u > 0 && t_hi >= before && t_hi < after;
        const long long snap = work / (n_xcd * 8);
        auto cut = [&](long long t) -> int {   // tile of this expert at which work t lies behind
            if (t - before <= after - t) {
                if (t - before <= snap) return e * tiles_e;
            } else if (after - t <= snap) {
                return (e + 1) * tiles_e;
            }
            return e * tiles_e + static_cast<int>((t - before) / (u > 0 ? u : 1));
        };
        const int tile_lo = cut(t_lo), tile_hi = cut(t_hi);
        const unsigned long long m_lo = __ballot(has_lo), m_hi = __ballot(has_hi);
        if (m_lo) lo = __shfl(tile_lo, __ffsll(static_cast<long long>(m_lo)) - 1, 64);
        if (m_hi) hi = __shfl(tile_hi, __ffsll(static_cast<long long>(m_hi)) - 1, 64);
        base += __shfl(incl, 63, 64);
    }
    if (xcd == 0) lo = 0;
}

// 16 bytes per lane global -> LDS at lds_base + OFS + lane * 16, nothing with fewer than two steps `left` (block-uniform).
// Written as assembly so that the compiler neither waits for such a load nor takes it for an LDS access: the main loop's own
// waits and barriers order them.  The branch lies inside, so that a step stays one block for the compiler's scheduler.
template <int OFS>
__device__ __forceinline__ void dma16_if(int left, const void *base, uint32_t lane_bytes, uint32_t lds_base) {
    asm volatile("s_cmp_lt_i32 %4, 2\n\ts_cbranch_scc1 .Lom_skip%=\n\ts_add_u32 m0, %0, %3\n\ts_nop 0\n\t"
                 "global_load_lds_dwordx4 %1, %2\n.Lom_skip%=:"
                 :: "s"(lds_base), "v"(lane_bytes), "s"(base), "n"(OFS), "s"(left) : "scc");
}
// dma16_if of data that is read once: kept out of the caches where `once` is set
template <int OFS>
__device__ __forceinline__ void dma16_if_once(int left, int once, const void *base, uint32_t lane_bytes, uint32_t lds_base) {
    asm volatile("s_cmp_lt_i32 %4, 2\n\ts_cbranch_scc1 .Lom_skip%=\n\ts_add_u32 m0, %0, %3\n\ts_cmp_eq_u32 %5, 0\n\t"
                 "s_cbranch_scc1 .Lom_keep%=\n\tglobal_load_lds_dwordx4 %1, %2 nt\n\ts_branch .Lom_skip%=\n.Lom_keep%=:\n\t"
                 "global_load_lds_dwordx4 %1, %2\n.Lom_skip%=:"
                 :: "s"(lds_base), "v"(lane_bytes), "s"(base), "n"(OFS), "s"(left), "s"(once) : "scc");
}
// This wavefront's direct loads but the N youngest have landed, and its LDS reads are back.
template <int N> __device__ __forceinline__ void wait_loads(uint32_t lds) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(N), "s"(lds) : "memory");
}
// The same inside a tile's main loop, by the number of steps that follow: N2 with two or more, N1 with one, 0 with none;
// no load is waited for with a negative number.
template <int N2, int N1> __device__ __forceinline__ void wait_step_loads(int left, uint32_t lds) {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_cmp_lt_i32 %2, 0\n\ts_cbranch_scc1 .Lom_wait%=\n\ts_waitcnt vmcnt(%0)\n\t"
                 "s_cmp_ge_i32 %2, 2\n\ts_cbranch_scc1 .Lom_wait%=\n\ts_waitcnt vmcnt(%1)\n\t"
                 "s_cmp_ge_i32 %2, 1\n\ts_cbranch_scc1 .Lom_wait%=\n\ts_waitcnt vmcnt(0)\n.Lom_wait%=:"
                 :: "n"(N2), "n"(N1), "s"(left), "s"(lds) : "memory", "scc");
}
__device__ __forceinline__ void block_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <int V> using IntC = std::integral_constant<int, V>;

// EDGE: output extents and contraction lengths that are any multiple of 8: the last tile along an extent and the last
// step of a phase may be partial (loads past them are clamped, A is zeroed, stores are masked).  The 256x256 kernels are
// launched on whole tiles and steps only and carry none of that.
// (second launch bound: two wavefronts per SIMD, i.e. at most 256 registers, for the 128x128 tile, whose two blocks per
// CU depend on it; the 256x256 tile's 8 wavefronts imply it already)
// What a block of a kernel keeps in LDS beside its two stages: how many of each.
template <int BM, int EPI, int GATHER, bool EDGE> struct Tables {
    static constexpr bool WGRAD = EPI == EPI_WGRAD, GATHER_W = WGRAD && GATHER != GATHER_NONE;
    static constexpr bool SHARES = !WGRAD || !EDGE;                                  // whether the launch may be one with p.share != 0
    static constexpr int LDS = 4 * (BM / 64) * 8192;                                 // A of even and odd steps, then B
    static constexpr int IDX_CACHE = GATHER_W ? (BM == 256 ? 4096 : 2048) : 1;
    static constexpr int PARTS = SHARES ? SHARE_MAX_EXPERTS : 1;
    static constexpr int ENDS = !WGRAD ? MAX_EXPERTS : PARTS;                        // see build_tile_table, build_part_table
    static constexpr int SEGS = WGRAD ? 1 : MAX_EXPERTS + 1;                         // see build_tile_table; p.share: build_first_tiles
};

// A block's tiles, counted from the other end of its XCD's blocks with FROM_END.  (The tables one by one: as members of one object the compiler keeps their accesses in order
// with those of the stages, which in the weight gradients cost registers.)
template <int BM, int AKIND, int BKIND, int EPI, int GATHER, bool ROWW, bool ACCUM, bool EDGE, bool ONCE, bool DENSE, bool FROM_END = false,
          typename D = Tables<BM, EPI, GATHER, EDGE>>
__device__ __forceinline__ void ggemm_tiles(const GemmParams p, char (&lds)[D::LDS], int (&idx_cache)[D::IDX_CACHE], int (&order)[D::PARTS],
                                            Part (&part)[D::PARTS], int (&tile_end)[D::ENDS], int (&seg)[D::SEGS]) {
    constexpr int BN = BM, WAVES_N = BN / 64, NW = 2 * WAVES_N;
    constexpr int TM = BM / 64, TN = 2;     // row units of a tile, accumulators of a wavefront in each
    static_assert(GATHER == GATHER_NONE || (GATHER == GATHER_A && AKIND == CONTIG && EPI != EPI_WGRAD) ||
                      (GATHER == GATHER_B && BKIND == STRIDED && EPI == EPI_WGRAD) ||
                      ((GATHER == GATHER_WA || GATHER == MERGED) && AKIND == STRIDED && EPI == EPI_WGRAD), "gather variants");
    static_assert(!DENSE || (BM == 128 && EPI != EPI_WGRAD), "few rows per expert");
    static_assert(!ACCUM || EPI == EPI_WGRAD, "only the weight gradient adds into its output");
    static_assert(!ROWW || EPI == EPI_SWIGLU || EPI == EPI_SWIGLU_BWD, "row weights belong to the SwiGLU epilogues");
    constexpr bool WGRAD = EPI == EPI_WGRAD;
    constexpr bool GATHER_W = GATHER == GATHER_B || GATHER == GATHER_WA || GATHER == MERGED;
    constexpr int UNIT = 8192;             // bytes of an operand unit: 64 rows (CONTIG) or 64 columns (STRIDED) x 64 c
    constexpr int UA = TM, UB = BN / 64;   // units of a step
    constexpr int L = 8 / NW;              // direct loads per wavefront per unit
    constexpr int A_STAGE = UA * UNIT, B_STAGE = UB * UNIT;
    constexpr int B0 = 2 * A_STAGE;        // A of even and odd steps, then B of even and odd steps
    static_assert(D::LDS == 2 * A_STAGE + 2 * B_STAGE, "two stages");
    constexpr int IDX_CACHE = D::IDX_CACHE;
    int cached_expert = -1;            // (MERGED: and product)
    constexpr bool SHARES = D::SHARES;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;

    const int xcd = blockIdx.x % NUM_XCD;
    // ---- per-tile state (set by setup_tile) ---------------------------------------------------
    int expert = 0, row_begin = 0, row_end = 0, n0 = 0, c_begin = 0, c_len = 0;
    int steps_per_phase = 0, c_wrap = 0, n_steps = 0, rot = 0;
    int active = TM;      // row units that hold rows of the expert
    bool dense = false;   // DENSE: whether the tile is the dense expert's
    auto own = [&](auto of_dense, auto of_routed) { return DENSE ? pick(dense, of_dense, of_routed) : of_routed; };
    int once = 0;         // ONCE: whether no other row tile reads the expert's weights
    // the slot of this wavefront's direct load l of a unit: row (CONTIG) or contraction row (STRIDED) and chunk
    auto slot = [&](int l) { return (wave * L + l) * 8 + (lane >> 3); };
    uint32_t a_off[AKIND == CONTIG ? UA : 1][L];   // bytes from the step's base: CONTIG, the row of each unit
    uint32_t b_off[EDGE ? UB : 1][L];         // CONTIG as above; STRIDED, the column
    const char *a_tile[2] = {}, *b_tile[2] = {};   // base addresses of the tile's operands (two phases), block-uniform
    int tail_c0 = -1;     // first contraction index of the partial step, if the tile has one
    int src[GATHER_W ? 3 : 1][L];             // GATHER_W: source rows of this lane's slots, steps t, t + 1, t + 2
    // of the current product (MERGED: set by setup_tile, otherwise the launch's)
    int lda32 = static_cast<int>(p.lda), ldb32 = static_cast<int>(p.ldb), n_cols = p.n_cols, m_rows = p.kc, product = 0;
    const int32_t *row_index = p.row_index;
    bool a_indexed = GATHER == GATHER_WA, b_indexed = GATHER == GATHER_B;
    constexpr bool TWO_PHASE = EPI == EPI_STORE && BKIND == STRIDED;   // the merged MLP's dx = dg Wg + du Wu
    const int64_t b_unit = static_cast<int64_t>(EPI == EPI_SWIGLU ? 32 : 64) * p.ldb * 2;   // CONTIG: bytes between units
    const uint32_t lds_addr = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void_ptr)lds));
    const uint32_t wave_lds = __builtin_amdgcn_readfirstlane(lds_addr + wave * (L * 1024));

    // Contraction steps run from `rot` to the end of the range and on from its start (both phases alike).
    auto next_c0 = [&](int c0) { return c0 + BK >= c_wrap ? 0 : c0 + BK; };
    // GATHER_W: the source rows of the step at c0; the first IDX_CACHE of an expert's rows come from LDS
    auto look_up = [&](int c0, int (&out)[L]) {
        if (!GATHER_W || (GATHER == MERGED && !row_index)) return;
#pragma unroll
        for (int l = 0; l < L; l++) {
            const int c = min(c0 + slot(l), c_len - 1);
            if (c0 + BK <= IDX_CACHE) {
                out[l] = idx_cache[c];
            } else {   // (waited for here: at the join the compiler would wait for the direct loads too, on either path)
                int v = row_index[c_begin + c];
                asm volatile("" : "+v"(v));
                out[l] = v;
            }
        }
    };

    auto tiles_of = [&](int rows) {
        constexpr int BN_OUT = (EPI == EPI_SWIGLU) ? BN / 2 : BN;
        return WGRAD ? p.tiles_e : (rows + BM - 1) / BM * ((p.n_cols + BN_OUT - 1) / BN_OUT);
    };
    // p.share: `logical` counts this XCD's tiles, otherwise the launch's
    auto setup_tile = [&](int logical) -> bool {
        int rot_a, rot_b;
        if (WGRAD) {
            int tile;
            if (SHARES && p.share) {
                const Part q = find_part(tile_end, part, p.n_experts, lane, logical);
                expert = q.expert;
                tile = logical + q.shift;
                c_begin = q.row_begin;
                c_len = q.row_end - q.row_begin;
            } else {
                expert = logical / p.tiles_e;
                tile = logical - expert * p.tiles_e;
                c_begin = p.cum[expert];
                c_len = p.cum[expert + 1] - c_begin;
            }
            if (GATHER == MERGED) {
                const int each = p.tiles_e / 3;     // (the three have the same extents, one of them transposed)
                product = __builtin_amdgcn_readfirstlane(tile / each);
                tile -= product * each;
                const WgradSet &w = p.set[product];
                m_rows = w.m; n_cols = w.n;
                lda32 = m_rows; ldb32 = n_cols;
                a_indexed = w.a_rows != nullptr; b_indexed = w.b_rows != nullptr;
                row_index = a_indexed ? w.a_rows : w.b_rows;
            }
            const int tiles_n = (n_cols + BN - 1) / BN;
            int tm = tile / tiles_n, tn = tile % tiles_n;
            if (SHARES && p.share && n_cols > m_rows) {   // columns of tiles instead of rows
                const int tiles_m = m_rows / BM;
                tn = tile / tiles_m;
                tm = tile % tiles_m;
            }
            rot_a = tn; rot_b = tm;
            row_begin = tm * BM;
            row_end = m_rows;
            n0 = tn * BN;
        } else {
            constexpr int BN_OUT = (EPI == EPI_SWIGLU) ? BN / 2 : BN;
            const int tiles_n = (p.n_cols + BN_OUT - 1) / BN_OUT;
            int tile_m = logical / tiles_n, tile_n = logical % tiles_n, row_tile = tile_m;
            if (p.share) {
                const Part q = find_part(tile_end, part, p.n_experts, lane, logical);
                const int tile = logical + q.shift, tiles_m = (q.row_end - q.row_begin + BM - 1) / BM;
                tile_n = tile / tiles_m;
                tile_m = tile - tile_n * tiles_m;
                expert = q.expert;
                row_begin = q.row_begin + tile_m * BM;
                row_end = q.row_end;
                row_tile = __builtin_amdgcn_readfirstlane(seg[expert]) + tile_m;
            } else if (!find_tile<BM>(tile_end, seg, p.n_experts + DENSE, tile_m, lane, expert, row_begin, row_end)) return false;
            int first_row = p.share ? 0 : seg[expert];   // (p.share: not used)
            if (DENSE) {
                dense = __builtin_amdgcn_readfirstlane(expert) == p.n_experts;
                if (dense) {
                    row_tile -= tile_end[p.n_experts - 1];
                    row_begin = row_tile * BM;
                    row_end = p.dense.rows;
                    first_row = 0;
                }
            }
            if (ONCE) once = __builtin_amdgcn_readfirstlane(row_end - row_begin <= BM && (p.share ? tile_m == 0 : row_begin == first_row) ? 1 : 0);
            // (`row_tile` among all experts' with and without p.share: the sums begin at the same step, the same bits)
            rot_a = tile_n; rot_b = row_tile & 7;
            n0 = tile_n * BN_OUT;
            c_begin = 0;
            c_len = p.kc;
        }
        expert = __builtin_amdgcn_readfirstlane(expert);
        row_begin = __builtin_amdgcn_readfirstlane(row_begin);
        row_end = __builtin_amdgcn_readfirstlane(row_end);
        n0 = __builtin_amdgcn_readfirstlane(n0);
        c_begin = __builtin_amdgcn_readfirstlane(c_begin);
        c_len = __builtin_amdgcn_readfirstlane(c_len);
        steps_per_phase = (c_len + BK - 1) / BK;
        n_steps = steps_per_phase * p.phases;
        rot = (rot_a + rot_b) % (steps_per_phase > 0 ? steps_per_phase : 1);
        c_wrap = steps_per_phase * BK;
        tail_c0 = (WGRAD || EDGE) && c_wrap != c_len ? c_wrap - BK : -1;
        active = WGRAD && !EDGE ? TM : min((row_end - row_begin + 63) >> 6, TM);
        int lane_s = lane;
        asm volatile("" : "+v"(lane_s));   // recomputed per tile, not kept across the main loop
        const int ch8 = lane_s & 7;
#pragma unroll
        for (int l = 0; l < L; l++) {
            const int r = (wave * L + l) * 8 + (lane_s >> 3);
            if (AKIND == CONTIG) {
                const int ch = ch8 ^ swz(r);
#pragma unroll
                for (int u = 0; u < UA; u++) {
                    int m = min(row_begin + u * 64 + r, row_end - 1);   // rows past the segment: valid memory, result unused
                    if (GATHER == GATHER_A && !dense) m = p.row_index[m];
                    else if (GATHER != GATHER_A) m -= row_begin;
                    a_off[u][l] = (static_cast<uint32_t>(m) * lda32 + ch * 8) * 2u;
                }
            } else {
                a_off[0][l] = (ch8 ^ unit_swz(r)) * 16;    // bytes of the column within the unit
            }
            if (BKIND == CONTIG) {
                const int ch = ch8 ^ swz(r);
                // EPI_SWIGLU: a unit holds 32 gate rows and the same 32 up rows (see B_first)
                constexpr int PER_UNIT = EPI == EPI_SWIGLU ? 32 : 64;
                const int n = EPI == EPI_SWIGLU ? (r & 31) : r;
#pragma unroll
                for (int u = 0; u < (EDGE ? UB : 1); u++)
                    b_off[u][l] = (static_cast<uint32_t>(EDGE ? min(u * PER_UNIT + n, p.n_cols - 1 - n0) : n) * ldb32 + ch * 8) * 2u;
            } else {
                const int col = (ch8 ^ unit_swz(r)) * 8;
#pragma unroll
                for (int u = 0; u < (EDGE ? UB : 1); u++)
                    b_off[u][l] = (EDGE ? min(u * 64 + col, n_cols - 8 - n0) : col) * 2;
            }
        }
        const int64_t a_base = AKIND == CONTIG ? (GATHER == GATHER_A ? 0 : static_cast<int64_t>(row_begin) * p.lda)
                                               : row_begin + (a_indexed ? 0 : static_cast<int64_t>(c_begin) * lda32);
        const int64_t matrix = dense ? 0 : expert * p.strideB;
        const int64_t b_base = BKIND == CONTIG ? matrix + static_cast<int64_t>(n0) * p.ldb
                               : WGRAD ? n0 + (b_indexed ? 0 : static_cast<int64_t>(c_begin) * ldb32)
                                       : matrix + n0;
        // EPI_SWIGLU: LDS rows 0..31 of a unit are gate rows, 32..63 up rows; a wavefront's loads lie in one of the two
        const bool second = EPI == EPI_SWIGLU && wave * L * 8 >= 32;
        const uint16_t *A_first = GATHER == MERGED ? p.set[product].A : own(p.dense.A[0], p.A[0]);
        const uint16_t *B_first = GATHER == MERGED ? p.set[product].B
                                : EPI == EPI_SWIGLU ? pick(second, own(p.dense.B[1], p.B[1]), own(p.dense.B[0], p.B[0])) : own(p.dense.B[0], p.B[0]);
        a_tile[0] = reinterpret_cast<const char *>(uniform64(reinterpret_cast<int64_t>(A_first + a_base)));
        b_tile[0] = reinterpret_cast<const char *>(uniform64(reinterpret_cast<int64_t>(B_first + b_base)));
        if (TWO_PHASE) {
            const bool two = p.phases > 1;
            const uint16_t *A_second = pick(two, own(p.dense.A[1], p.A[1]), own(p.dense.A[0], p.A[0]));
            const uint16_t *B_second = pick(two, own(p.dense.B[1], p.B[1]), own(p.dense.B[0], p.B[0]));
            a_tile[1] = reinterpret_cast<const char *>(uniform64(reinterpret_cast<int64_t>(A_second + a_base)));
            b_tile[1] = reinterpret_cast<const char *>(uniform64(reinterpret_cast<int64_t>(B_second + b_base)));
        }
        const int cache_key = GATHER == MERGED ? expert * 2 + (row_index != p.set[1].b_rows ? 1 : 0) : expert;
        if (GATHER_W && (GATHER != MERGED || row_index) && cache_key != cached_expert) {
            // every wavefront is past the barrier that ends the previous tile's main loop, so no one still reads
            // the cache; `expert` is block-uniform, so all take this branch together
            const int n_cached = min(c_len, IDX_CACHE);
            for (int i = tid; i < n_cached; i += NW * 64) idx_cache[GATHER_W ? i : 0] = row_index[c_begin + i];
            cached_expert = cache_key;
            __syncthreads();
        }
        if (GATHER_W && n_steps > 0) {
            const int c0 = rot * BK, c1 = next_c0(c0);
            look_up(c0, src[0]);
            look_up(c1, src[GATHER_W ? 1 : 0]);
            look_up(next_c0(c1), src[GATHER_W ? 2 : 0]);
        }
        return true;
    };

    // ---- direct loads of one unit into the buffers of parity P; base: a_step / b_step of the unit's step -------
    auto a_step = [&](int c0, int t) -> const char * {
        const char *q = TWO_PHASE && t >= steps_per_phase ? a_tile[1] : a_tile[0];
        if (WGRAD && a_indexed) return q;
        return q + (AKIND == CONTIG ? static_cast<uint64_t>(static_cast<uint32_t>(c0)) * 2 : static_cast<uint64_t>(static_cast<uint32_t>(c0)) * static_cast<uint32_t>(lda32 * 2));
    };
    auto b_step = [&](int c0, int t) -> const char * {
        const char *q = TWO_PHASE && t >= steps_per_phase ? b_tile[1] : b_tile[0];
        if (WGRAD && b_indexed) return q;
        return q + (BKIND == CONTIG ? static_cast<uint64_t>(static_cast<uint32_t>(c0)) * 2 : static_cast<uint64_t>(static_cast<uint32_t>(c0)) * static_cast<uint32_t>(ldb32 * 2));
    };
    // bytes of the contraction row (STRIDED): rows past the range re-read its last row (A is zeroed there)
    auto crow_bytes = [&](int c0, int l, int ld32, const int (&rows)[L], bool indexed) -> uint32_t {
        if (indexed) return static_cast<uint32_t>(rows[l]) * (ld32 * 2u);
        const uint32_t r = static_cast<uint32_t>(slot(l)) * (ld32 * 2u);
        return WGRAD || EDGE ? min(r, static_cast<uint32_t>(min(c_len - 1 - c0, BK)) * (ld32 * 2u)) : r;
    };
    // CONTIG, a partial last step: its chunks past the end re-read the last one (A's are zeroed)
    auto tail_bytes = [&](int c0, int l) -> uint32_t {
        return EDGE ? max(((lane & 7) ^ swz(slot(l))) - (((c_len - c0) >> 3) - 1), 0) * 16 : 0;
    };
    auto issue_a = [&](int left, const char *base, int c0, auto par, auto unit, const int (&rows)[L]) {
        constexpr int P = decltype(par)::value, U = decltype(unit)::value;
#pragma unroll
        for (int l = 0; l < L; l++) {
            uint32_t off;
            if (AKIND == CONTIG) off = a_off[AKIND == CONTIG ? U : 0][l] - tail_bytes(c0, l);
            else off = crow_bytes(c0, l, lda32, rows, a_indexed) +
                       (EDGE ? min(a_off[0][l] + U * 128, static_cast<uint32_t>(m_rows - 8 - row_begin) * 2) : a_off[0][l]);
            const char *q = AKIND == CONTIG || EDGE ? base : base + U * 128;
            if (l == 0) dma16_if<P * A_STAGE + U * UNIT>(left, q, off, wave_lds);
            else dma16_if<P * A_STAGE + U * UNIT + 1024>(left, q, off, wave_lds);
        }
    };
    auto issue_b = [&](int left, const char *base, int c0, auto par, auto unit, const int (&rows)[L]) {
        constexpr int P = decltype(par)::value, U = decltype(unit)::value;
        const int past = ONCE ? __builtin_amdgcn_readfirstlane(once) : 0;
#pragma unroll
        for (int l = 0; l < L; l++) {
            uint32_t off = b_off[EDGE ? U : 0][l];
            if (BKIND == CONTIG) off -= tail_bytes(c0, l);
            else off += crow_bytes(c0, l, ldb32, rows, b_indexed);
            const char *q = EDGE ? base : BKIND == CONTIG ? base + U * b_unit : base + U * 128;
            if (ONCE && l == 0) dma16_if_once<B0 + P * B_STAGE + U * UNIT>(left, past, q, off, wave_lds);
            else if (ONCE) dma16_if_once<B0 + P * B_STAGE + U * UNIT + 1024>(left, past, q, off, wave_lds);
            else if (l == 0) dma16_if<B0 + P * B_STAGE + U * UNIT>(left, q, off, wave_lds);
            else dma16_if<B0 + P * B_STAGE + U * UNIT + 1024>(left, q, off, wave_lds);
        }
    };
    auto issue_b_all = [&](const char *base, int c0, auto par, const int (&rows)[L]) {
        issue_b(2, base, c0, par, IntC<0>{}, rows);
        issue_b(2, base, c0, par, IntC<1>{}, rows);
        if constexpr (UB == 4) { issue_b(2, base, c0, par, IntC<2>{}, rows); issue_b(2, base, c0, par, IntC<3>{}, rows); }
    };
    // zero what lies past the contraction range in A (B holds finite data there, so the products vanish):
    // this wavefront's own slots of a unit, after its loads have landed and before the barrier
    auto zero_tail = [&](int c0, auto par, auto unit) {
        if ((!WGRAD && !EDGE) || c0 != tail_c0) return;
        char *q = lds + decltype(par)::value * A_STAGE + decltype(unit)::value * UNIT + wave * (L * 1024) + lane * 16;
#pragma unroll
        for (int l = 0; l < L; l++) {
            const int c = AKIND == CONTIG ? ((lane & 7) ^ swz(slot(l))) * 8 : slot(l);
            if (c0 + c >= c_len) {
                // made here: four registers of zeros kept for the whole loop were spilled in the accumulating 256x256 weight gradients, and
                // registers were short in the others.  us, kept -> made: 64 experts of 2048/1024, 32768 rows, uneven, 1049 -> 1029 (added 1050 ->
                // 1046), 131072 rows 1401 -> 1379 (1506 -> 1487); 32 of 7168/2048, 12510 rows, uneven, 1277 -> 1259 (1681 -> 1669)
                uint32_t zero = 0;
                asm volatile("" : "+v"(zero));
                *reinterpret_cast<u32x4 *>(q + l * 1024) = u32x4{zero, zero, zero, zero};
            }
        }
    };

    // ---- fragments --------------------------------------------------------------------------------
    int a_frag[2], b_frag[BKIND == CONTIG ? 2 : 4];   // byte addresses within a unit region: CONTIG by kk, STRIDED by block
    auto set_fragments = [&]() {
        int lane_f = lane;
        asm volatile("" : "+v"(lane_f));   // recomputed per tile, not kept across the epilogue
        const int l16 = lane_f & 15, g4 = lane_f >> 4;
        const int q16 = lane_f & 3, cr = 8 * g4 + (l16 >> 2);
#pragma unroll
        for (int x = 0; x < 2; x++) {
            if (AKIND == CONTIG) {
                a_frag[x] = (wm * 32 + l16) * 128 + (((x * 4 + g4) ^ swz(l16)) << 4);
            } else {
                const int m = wm * 32 + x * 16 + 4 * q16;
                a_frag[x] = cr * 128 + (((m >> 3) ^ unit_swz(cr)) << 4) + (m & 7) * 2;
            }
        }
#pragma unroll
        for (int x = 0; x < (BKIND == CONTIG ? 2 : 4); x++) {
            if (BKIND == CONTIG) {
                b_frag[x] = B0 + wn * UNIT + l16 * 128 + (((x * 4 + g4) ^ swz(l16)) << 4);
            } else {
                const int m = x * 16 + 4 * q16;
                b_frag[x] = B0 + wn * UNIT + cr * 128 + (((m >> 3) ^ unit_swz(cr)) << 4) + (m & 7) * 2;
            }
        }
    };
    auto read_tr = [&](const char *q) -> bf16x8 {
        typedef __attribute__((ext_vector_type(8))) short s16x8;
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(q));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(q + 4 * 128));
        return __builtin_bit_cast(bf16x8, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    bf16x8 fa[2][2][2], fb[2][4][2];   // [..][16-row block][32 indices]
    f32x4 acc[TM][2][4];
    auto read_a = [&](auto par, auto unit, auto k_lo, auto k_hi) {
        constexpr int O = decltype(par)::value * A_STAGE + decltype(unit)::value * UNIT, buf = decltype(unit)::value & 1;
#pragma unroll
        for (int kk = decltype(k_lo)::value; kk < decltype(k_hi)::value; kk++)
#pragma unroll
            for (int i = 0; i < 2; i++) {
                if (AKIND == CONTIG) fa[buf][i][kk] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(lds + a_frag[kk] + O + i * 2048));
                else fa[buf][i][kk] = read_tr(lds + a_frag[i] + O + kk * 4096);
            }
    };
    // fragments f_lo .. f_hi of the eight (four of every 32 indices)
    auto read_b = [&](auto par, auto f_lo, auto f_hi) {
        constexpr int P = decltype(par)::value, O = P * B_STAGE;
#pragma unroll
        for (int f = decltype(f_lo)::value; f < decltype(f_hi)::value; f++) {
            const int kk = f >> 2, j = f & 3;
            if (BKIND == CONTIG) fb[P][j][kk] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(lds + b_frag[BKIND == CONTIG ? kk : 0] + O + j * 2048));
            else fb[P][j][kk] = read_tr(lds + b_frag[BKIND == CONTIG ? 0 : j] + O + kk * 4096);
        }
    };
    auto multiply = [&](auto par, auto unit, auto k) {
        constexpr int P = decltype(par)::value, I = decltype(unit)::value, kk = decltype(k)::value;
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                // operands swapped: the lane then holds 4 consecutive output columns per row
                acc[I][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[P][j][kk], fa[I & 1][i][kk], acc[I][i][j], 0, 0, 0);
    };
    // one MFMA, then the LDS reads of the next phase behind the leading MFMAs, the rest of the MFMAs last
    auto schedule = [&](auto reads) {
        constexpr int R = decltype(reads)::value, PER = R > 7 ? (R + 6) / 7 : (R > 0 ? 1 : 0);
        int left = R;
#pragma unroll
        for (int m = 0; m < 8; m++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
#pragma unroll
            for (int q = 0; q < PER; q++)
                if (left > 0) { __builtin_amdgcn_sched_group_barrier(0x100, 1, 0); left--; }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    constexpr int RA = AKIND == CONTIG ? 4 : 8, RB = BKIND == CONTIG ? 8 : 16;   // LDS reads of a unit of A, of a step of B

    const int nbx = gridDim.x / NUM_XCD, slot_x = FROM_END ? nbx - 1 - static_cast<int>(blockIdx.x / NUM_XCD) : static_cast<int>(blockIdx.x / NUM_XCD);
    int total_tiles = p.total_tiles, per = 0, rem = 0, run_lo = 0;
    if (SHARES && p.share) {
        expert_order(p.cum, p.n_experts, tid, lane, order);
        if (wave == 0) build_part_table(p.cum, order, p.n_experts, p.share, xcd, lane, tiles_of, tile_end, part);
        if constexpr (!WGRAD) { if (wave == 1) build_first_tiles<BM>(p.cum, p.n_experts, lane, seg); }
        __syncthreads();
        per = __builtin_amdgcn_readfirstlane(tile_end[p.n_experts - 1]);
    } else {
        if (!WGRAD) {
            if (wave == 0) build_tile_table<BM>(p.cum, p.n_experts, lane, tile_end, seg);
            __syncthreads();
            if (DENSE) {
                if (tid == 0) tile_end[p.n_experts] = tile_end[p.n_experts - 1] + (p.dense.rows + BM - 1) / BM;
                __syncthreads();
            }
            constexpr int BN_OUT = (EPI == EPI_SWIGLU) ? BN / 2 : BN;
            total_tiles = __builtin_amdgcn_readfirstlane(tile_end[p.n_experts - 1 + DENSE]) * ((p.n_cols + BN_OUT - 1) / BN_OUT);
        }
        per = total_tiles / NUM_XCD;
        rem = total_tiles - per * NUM_XCD;
        run_lo = xcd * per;
        if (WGRAD && p.n_experts <= WGRAD_BALANCE_MAX_EXPERTS) {
            int lo, hi;
            wgrad_xcd_run(p.cum, p.n_experts, p.tiles_e, BK, xcd, NUM_XCD, lane, lo, hi);
            run_lo = __builtin_amdgcn_readfirstlane(lo);
            per = __builtin_amdgcn_readfirstlane(hi) - run_lo;
            rem = 0;
        }
    }
    // the block's place in round `it` of its XCD
    auto place = [&](int it) { return SHARES && p.share && (it & 1) ? nbx - 1 - slot_x : slot_x; };
    const int n_mine = per / nbx + (place(per / nbx) < per % nbx ? 1 : 0);
    const int n_all = n_mine + ((xcd < rem && slot_x == per % nbx) ? 1 : 0);
    int it = 0;
    auto next_tile = [&]() -> bool {
        while (it < n_all) {
            const int logical = it < n_mine ? run_lo + place(it) + it * nbx : total_tiles - rem + xcd;
            it++;
            // (nothing to add for an expert without rows)
            if (setup_tile(logical) && !(ACCUM && n_steps == 0)) return true;
        }
        return false;
    };
    constexpr IntC<0> c0_{}; constexpr IntC<1> c1_{}; constexpr IntC<2> c2_{}; constexpr IntC<3> c3_{};
    constexpr IntC<4> c4_{}; constexpr IntC<6> c6_{}; constexpr IntC<8> c8_{};
    // Step 0 of a tile, and (second) of step 1 what does not go where the strips of the epilogue lie (A's last units).
    // EARLY: both are loaded ahead of the epilogue's stores, and the tile's first step does not wait for those: the memory
    // counter runs in order, so before this a tile began when the last one's 128 KB had been accepted.  Weight gradients
    // alone, us: 64 experts of 2048/1024, 512 tokens, uneven 200 -> 180 (the pass 603 -> 599, bound by what memory takes),
    // 16384 tokens 1447 -> 1415; 32 experts of 7168/2048, 400 uneven rows, 1364 -> 1314, added 1814 -> 1783.  The row products,
    // with more steps to a tile, gain nothing by it (1 % slower in gate+up of 512 rows), nor do 128x128 tiles, whose two blocks per CU
    // cover each other's stores: early, with the stores waited for -> not, us: 12 experts of 1000/712, 9003 rows, 74.3 -> 73.8; 64 of
    // 1712/1048, 8192 rows, 309 -> 304; 8 of 256/512, 4096 rows, 25.8 -> 25.5 (with a whole tile's eight stores counted 1.5 % slower than early).
    constexpr int FIRST = 6;                  // loads of step 1 in second()
    constexpr int LAST = TM == 4 ? 2 : 1;     // the unit of A that follows them (TM == 4: and the one behind it, with step 0)
    // 128x128: what a wavefront loads of that unit goes where its own strip lies, so it need not wait for the others' strips, as it does
    // with 256x256 tiles (one barrier later; strips of their own in those units gained nothing there).  With few steps to a tile
    // part of the load's way was waited for.  Behind the barrier -> ahead of the first wait, us: 8 experts of 256/512, 4096 rows, down 13.2
    // -> 12.9; weight gradients of 64 experts of 1712/1048, 8192 rows, 304 -> 300, added ones of 16 of 1304/600, 4096 rows, 62.8 -> 62.1.
    constexpr bool OWN_STRIP = TM == 2;
    constexpr bool EARLY = WGRAD && !EDGE;
    auto second = [&]() {
        if (n_steps == 1) return;
        const int c1 = next_c0(rot * BK);
        const char *qa1 = a_step(c1, 1), *qb1 = b_step(c1, 1);
        issue_b_all(qb1, c1, c1_, src[GATHER_W ? 1 : 0]);
        issue_a(2, qa1, c1, c1_, c0_, src[GATHER_W ? 1 : 0]);
        if constexpr (TM == 4) issue_a(2, qa1, c1, c1_, c1_, src[GATHER_W ? 1 : 0]);
    };
    auto prefetch = [&]() {
        if (n_steps == 0) return;
        const int c0 = rot * BK;
        const char *qa = a_step(c0, 0), *qb = b_step(c0, 0);
        issue_b_all(qb, c0, c0_, src[0]);
        issue_a(2, qa, c0, c0_, c0_, src[0]);
        issue_a(2, qa, c0, c0_, c1_, src[0]);
        if constexpr (TM == 4) { issue_a(2, qa, c0, c0_, c2_, src[0]); issue_a(2, qa, c0, c0_, c3_, src[0]); }
        if (EARLY) second();
    };
    // 16-byte stores that a wavefront makes at least for a tile all of whose rows exist: they follow the next tile's prefetch,
    // and its first step does not wait for them
    constexpr int STORES = EARLY ? 16 : 0;
    bool stores_follow = false;
    bool have = next_tile();
    if (have) prefetch();
    while (have) {
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < 8; j++) acc[i][j >> 2][j & 3] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    if (n_steps > 0) {
        // c0 and operand addresses of the steps t + 1 and t + 2 (t: the step being multiplied)
        const int cs0 = rot * BK;
        int cs1 = next_c0(cs0), cs2 = next_c0(cs1), cst = cs0;
        const char *pa1 = a_step(cs1, 1), *pa2 = a_step(cs2, 2), *pb2 = b_step(cs2, 2);
        // steps that follow step 0, for the wait in its middle: nothing to wait for where all that it needs is here.  Asked for in step 0
        // alone, this makes the compiler copy the loop's first round, with accumulators that need not be zeroed first.  The weight gradients
        // gain by the copy; without it, us: 64 experts of 2048/1024, 512 tokens, uneven, 186 -> 192; added ones of 16 of 1304/600, 4096 rows,
        // 68.5 -> 70.6, of 12 of 1000/712, 9003 rows, 71.0 -> 72.4.  In the row products of 128x128 tiles it is a third of the code for a wait
        // that only a single step can skip; with -> without: 12 of 1000/712, 9003 rows, down 33.8 -> 33.0, 8 of 256/512, 4096 rows, 13.2 -> 12.9, 64 of
        // 2048/1024, 296 rows, 48.0 -> 47.4, others within 1 %.
        const int left0 = __builtin_amdgcn_readfirstlane(stores_follow || n_steps == 1 ? -1 : n_steps - 1);
        // One contraction step of parity P (see the comment above the kernel).  Past the last step nothing is loaded, and
        // what is read for it is not used.
        auto step = [&](auto par, auto full, int t) {
            constexpr int P = decltype(par)::value;
            constexpr bool FULL = decltype(full)::value;
            const int left = __builtin_amdgcn_readfirstlane(n_steps - 1 - t);
            constexpr IntC<P> same{}; constexpr IntC<P ^ 1> other{};
            const int (&s2)[L] = src[GATHER_W ? 2 : 0];
            int src3[L] = {};   // source rows of step t + 3
            const int cs3 = next_c0(cs2);
            constexpr IntC<RA / 2> ra{}; constexpr IntC<RA / 2 + RB / (TM == 2 ? 2 : 4)> rab{};
            if constexpr (TM == 2) {
                issue_b(left, pb2, cs2, same, c0_, s2);
                issue_b(left, pb2, cs2, same, c1_, s2);
                issue_a(left, pa2, cs2, same, c0_, s2);
                read_a(same, c1_, c0_, c1_);
                multiply(same, c0_, c0_);
                schedule(ra);
                read_a(same, c1_, c1_, c2_);
                multiply(same, c0_, c1_);
                schedule(ra);
                wait_step_loads<8, 2>(WGRAD && t == 0 ? left0 : left, lds_addr);
                zero_tail(cs1, other, c0_);
                block_barrier();
                if (GATHER_W && left >= 2) look_up(cs3, src3);
                issue_a(left, pa2, cs2, same, c1_, s2);
                read_a(other, c0_, c0_, c1_);
                read_b(other, c0_, c4_);
                if (FULL || active > 1) multiply(same, c1_, c0_);
                schedule(rab);
                read_a(other, c0_, c1_, c2_);
                read_b(other, c4_, c8_);
                if (FULL || active > 1) multiply(same, c1_, c1_);
                schedule(rab);
                wait_step_loads<8, 0>(left - (left == 0), lds_addr);
                zero_tail(cs1, other, c1_);
                block_barrier();
            } else {
                // phase 0
                issue_a(left + 1, pa1, cs1, other, c3_, src[GATHER_W ? 1 : 0]);
                read_a(same, c1_, c0_, c1_);
                multiply(same, c0_, c0_);
                schedule(ra);
                issue_b(left, pb2, cs2, same, c0_, s2);
                read_a(same, c1_, c1_, c2_);
                multiply(same, c0_, c1_);
                schedule(ra);
                // phase 1
                issue_b(left, pb2, cs2, same, c1_, s2);
                read_a(same, c2_, c0_, c1_);
                if (FULL || active > 1) multiply(same, c1_, c0_);
                schedule(ra);
                issue_b(left, pb2, cs2, same, c2_, s2);
                read_a(same, c2_, c1_, c2_);
                if (FULL || active > 1) multiply(same, c1_, c1_);
                schedule(ra);
                wait_step_loads<6, 3>(WGRAD && t == 0 ? left0 : left, lds_addr);
                zero_tail(cs1, other, c0_);
                zero_tail(cst, same, c3_);
                block_barrier();
                // phase 2
                if (GATHER_W && left >= 2) look_up(cs3, src3);
                issue_b(left, pb2, cs2, same, c3_, s2);
                read_a(same, c3_, c0_, c1_);
                read_b(other, c0_, c2_);
                if (FULL || active > 2) multiply(same, c2_, c0_);
                schedule(rab);
                issue_a(left, pa2, cs2, same, c0_, s2);
                read_a(same, c3_, c1_, c2_);
                read_b(other, c2_, c4_);
                if (FULL || active > 2) multiply(same, c2_, c1_);
                schedule(rab);
                // phase 3
                issue_a(left, pa2, cs2, same, c1_, s2);
                read_a(other, c0_, c0_, c1_);
                read_b(other, c4_, c6_);
                if (FULL || active > 3) multiply(same, c3_, c0_);
                schedule(rab);
                issue_a(left, pa2, cs2, same, c2_, s2);
                read_a(other, c0_, c1_, c2_);
                read_b(other, c6_, c8_);
                if (FULL || active > 3) multiply(same, c3_, c1_);
                schedule(rab);
                wait_step_loads<8, 1>(left - (left == 0), lds_addr);
                zero_tail(cs1, other, c1_);
                zero_tail(cs1, other, c2_);
                block_barrier();
            }
            if (GATHER_W) {
#pragma unroll
                for (int l = 0; l < L; l++) { src[0][l] = src[GATHER_W ? 1 : 0][l]; src[GATHER_W ? 1 : 0][l] = src[GATHER_W ? 2 : 0][l]; src[GATHER_W ? 2 : 0][l] = src3[l]; }
            }
            cst = cs1;
            cs1 = cs2;
            cs2 = cs3;
            pa1 = pa2;
            pa2 = a_step(cs2, t + 3);
            pb2 = b_step(cs2, t + 3);
        };
        if (!EARLY) second();
        auto last = [&]() { if (n_steps > 1) issue_a(2, pa1, cs1, c1_, IntC<LAST>{}, src[GATHER_W ? 1 : 0]); };
        if (OWN_STRIP) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (the strip's reads are back)
            last();
        }
        if (STORES && stores_follow) wait_loads<STORES>(lds_addr);
        else if (n_steps > 1) wait_loads<FIRST + (OWN_STRIP ? L : 0)>(lds_addr);
        else wait_loads<0>(lds_addr);
        zero_tail(cs0, c0_, c0_);
        zero_tail(cs0, c0_, c1_);
        if constexpr (TM == 4) { zero_tail(cs0, c0_, c2_); zero_tail(cs0, c0_, c3_); }
        block_barrier();
        if (!OWN_STRIP) last();   // (the strips are done with)
        set_fragments();
        read_a(c0_, c0_, c0_, c2_);
        read_b(c0_, c0_, c8_);
        block_barrier();   // (their buffers are the first that step 0 loads into)
        auto loop = [&](auto full) {
            for (int t = 0; t < n_steps; t += 2) {
                step(c0_, full, t);
                if (t + 1 < n_steps) step(c1_, full, t + 1);
            }
        };
        if (active == TM) loop(std::true_type{});
        else loop(std::false_type{});
    }
    __syncthreads();

    // ---- epilogue, while the next tile's first steps are loaded --------------------------------------------------------------
    // Each wavefront turns its accumulators around 16 rows at a time in a strip of its own (128-byte rows, 64 columns; in
    // the last units of odd steps' A) and moves 16-byte chunks of 8 neighbouring columns, eight lanes to a row.
    int lane_e = lane, wave_e = wave;
    asm volatile("" : "+v"(lane_e), "+s"(wave_e));
    const int wm_e = wave_e / WAVES_N, wn_e = wave_e % WAVES_N;
    constexpr int COLS = (EPI == EPI_SWIGLU) ? 32 : 64;   // output columns of this wavefront (EPI_SWIGLU: gate and up, side by side)
    static_assert(NW * 2048 == (TM - LAST) * UNIT, "strips are the units that second() leaves out");
    static_assert(!OWN_STRIP || (L * 1024 == 2048 && TM - LAST == 1), "a wavefront's strip is what it loads of that unit");
    const int strip = 2 * A_STAGE - NW * 2048 + wave_e * 2048;   // bytes from lds; 2 KB, its 16-byte chunks XOR-permuted by row
    int put_at[2], get_at[2];   // of blocks 0 and 1 (2 and 3: the other half of the row); of 8 rows and the other 8
    {
        const int row = lane_e & 15, g4 = lane_e >> 4;
#pragma unroll
        for (int j = 0; j < 2; j++) put_at[j] = strip + row * 128 + (((j * 2 + (g4 >> 1)) ^ swz(row)) << 4) + (g4 & 1) * 8;
#pragma unroll
        for (int x = 0; x < 2; x++) get_at[x] = strip + (x * 8 + (lane_e >> 3)) * 128 + (((lane_e & 7) ^ swz(x * 8 + (lane_e >> 3))) << 4);
    }
    auto strip_put = [&](auto block, f32x4 f) {
        constexpr int J = decltype(block)::value;
        *reinterpret_cast<u32x2 *>(lds + (put_at[J & 1] ^ (J >= 2 ? 64 : 0))) = u32x2{pack2_bf16(f[0], f[1]), pack2_bf16(f[2], f[3])};
    };
    auto strip_sync = [&]() {  // LDS operations of one wavefront are performed in order
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    // four blocks side by side: chunks 0 and 1 of the strip's rows
    auto turn = [&](f32x4 b0, f32x4 b1, f32x4 b2, f32x4 b3, u32x4 (&chunk)[2]) {
        strip_put(c0_, b0); strip_put(c1_, b1); strip_put(c2_, b2); strip_put(c3_, b3);
        strip_sync();
#pragma unroll
        for (int x = 0; x < 2; x++) chunk[x] = *reinterpret_cast<const u32x4 *>(lds + get_at[x]);
        strip_sync();
    };
    // SwiGLU backward: the saved g and u (and the weights) of two units are loaded ahead of the next tile's look-ups, those of
    // a further one when its buffer has been used; the fragments' registers are free by now.  Half a unit at a time, behind the next
    // tile's loads, each was waited for.  us: 3001 tokens, hidden 1000, ffn 712, 12 experts, top-3 (128x128) 39.9 -> 37.1; 512 tokens,
    // uneven, 64 experts of 2048/1024 as before (77); 16384 tokens (256x256) 715 -> 660 and less, whole steps of 2048 985 -> 977, 4096
    // 1546 -> 1524, 16384 uneven 5484 -> 5453 (the power limit keeps the rest), 32 experts of 1024/768, 9000 tokens, 709 -> 700.
    constexpr bool GU = EPI == EPI_SWIGLU_BWD;
    const int e_n_cols = n_cols, e_row_begin = row_begin, e_row_end = row_end, e_active = active;
    const int col0 = n0 + wn_e * COLS;   // first output column
    const int chunk_col = (lane_e & (COLS / 8 - 1)) * 8, chunk_row = lane_e >> 3;
    auto chunk_m = [&](int i, int x) { return (2 * i + wm_e) * 32 + x * 8 + chunk_row; };   // row within the tile; x 0 .. 3
    const bool all_rows = !EDGE && (WGRAD || e_row_begin + BM <= e_row_end);
    const int row_lim = EDGE && col0 + chunk_col >= e_n_cols ? 0 : e_row_end;
    const bool e_dense = dense;
    uint16_t *const C = own(p.dense.C, p.C), *const C1 = own(p.dense.C1, p.C1);
    uint16_t *const Cb = GATHER == MERGED ? p.set[product].C + expert * p.set[product].strideC : C + (WGRAD ? expert * p.strideC : 0);
    const int64_t e_ldc = GATHER == MERGED ? n_cols : p.ldc;
    uint16_t *const h_out = own(p.dense.C2, p.C2);
    const uint16_t *const g_saved = own(p.dense.G, p.G), *const u_saved = own(p.dense.U, p.U);
    // a chunk's element: block-uniform, and this lane's part of it
    const int64_t tile_at = uniform64(static_cast<int64_t>(e_row_begin + wm_e * 32) * e_ldc + col0);
    const uint32_t lane_at = static_cast<uint32_t>(chunk_row) * static_cast<uint32_t>(e_ldc) + chunk_col;
    auto chunk_at = [&](auto *base, int i, int x) {
        int64_t ldc = e_ldc;
        asm volatile("" : "+s"(ldc));   // made where it is used: all of a tile's at once spilled up to 51 scalar registers (times within 0.5 %)
        return base + (tile_at + (i * 64 + x * 8) * ldc) + lane_at;
    };
    float weight[ROWW && EPI == EPI_SWIGLU ? TM : 1][2];   // of the rows of this lane's accumulators; here, so that they do not wait for the prefetch
    if (ROWW && EPI == EPI_SWIGLU) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int x = 0; x < 2; x++)
                weight[ROWW && EPI == EPI_SWIGLU ? i : 0][x] = e_dense ? 1.0f :
                    p.row_scale[min(e_row_begin + (2 * i + wm_e) * 32 + x * 16 + (lane_e & 15), e_row_end - 1)];
    }
    u32x4 g_in[GU ? 2 : 1][GU ? 4 : 1], u_in[GU ? 2 : 1][GU ? 4 : 1];   // of even and odd units
    float w_in[GU ? 2 : 1][GU ? 4 : 1];
    auto load_gu = [&](int i) {
#pragma unroll
        for (int x = 0; x < 4; x++) {   // (rows and columns past the tile's: the last ones, not used)
            const int m = min(e_row_begin + chunk_m(i, x), e_row_end - 1), at = GU ? i & 1 : 0, ax = GU ? x : 0;
            const int64_t from = static_cast<int64_t>(m) * e_ldc + (EDGE ? min(col0 + chunk_col, e_n_cols - 8) : col0 + chunk_col);
            // no reader after this one: past the caches (-1 to -3 %)
            g_in[at][ax] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(g_saved + from));
            u_in[at][ax] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(u_saved + from));
            w_in[at][ax] = ROWW && !e_dense ? p.row_scale[m] : 1.0f;
        }
    };
    if (GU) { load_gu(0); load_gu(1); }
    u32x4 old[ACCUM ? TM : 1][ACCUM ? 4 : 1];
    if (ACCUM) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int x = 0; x < 4; x++) {
                // (EDGE: rows and columns past the matrix: its last ones, not used)
                const uint16_t *from = EDGE ? Cb + static_cast<int64_t>(min(e_row_begin + chunk_m(i, x), e_row_end - 1)) * e_ldc + min(col0 + chunk_col, e_n_cols - 8)
                                            : chunk_at(Cb, i, x);
                old[ACCUM ? i : 0][ACCUM ? x : 0] = *reinterpret_cast<const u32x4 *>(from);
            }
    }
    have = next_tile();
    if (ACCUM) {
        // Waited for here, ahead of the direct loads, which the compiler does not count: behind them each of its waits for an old value was one
        // for most of the next tile's first steps, and a path that it saw around them made it wait for the stores too, in each tile.  us,
        // behind -> ahead: 64 experts of 2048/1024, 4096 rows, uneven, 347 -> 328, 131072 rows 1532 -> 1506; 32 of 7168/2048, 12510 rows,
        // uneven, 1780 -> 1681; 12 of 1000/712, 9003 rows, 85.0 -> 83.1
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int x = 0; x < 4; x++) asm volatile("" : "+v"(old[ACCUM ? i : 0][ACCUM ? x : 0]));
    }
    if (have) prefetch();
    // the next tile's first wait counts the stores as younger than its loads: none may move ahead of them
    if (STORES) asm volatile("; stores from here on" ::: "memory");
    stores_follow = all_rows;
    auto rows_out = [&](auto past_caches) {   // (two loops: of a branch at each store the compiler knows less about what is under way)
#pragma unroll
        for (int i = 0; i < TM; i++) {
            if (i >= e_active) break;
            if (EPI == EPI_SWIGLU) {
                f32x4 h[2][2];
                u32x4 chunk[3][2];
                // gate and up of a row in one strip row: the lanes of its first half store to g, the others to u
                uint16_t *const gu = lane_e & 4 ? C1 : C;
                // neither where no backward follows: 128 MB of 32768 rows of 64 experts of 2048/1024, 345 -> 324 us, forward of 4096 tokens 492 -> 477
                const bool keep_gu = C != nullptr;
                // a strip is written again as soon as its reads are issued; what they bring is stored one strip later
                auto store_gu = [&](int x) {
#pragma unroll
                    for (int y = 0; y < 2; y++)
                        if (all_rows || e_row_begin + chunk_m(i, x * 2 + y) < row_lim)
                            *reinterpret_cast<u32x4 *>(chunk_at(gu, i, x * 2 + y)) = chunk[x][y];
                };
#pragma unroll
                for (int x = 0; x < 2; x++) {
#pragma unroll
                    for (int j = 0; j < 2; j++)
#pragma unroll
                        for (int y = 0; y < 4; y++) {
                            const float gv = acc[i][x][j][y], uv = acc[i][x][2 + j][y];
                            h[x][j][y] = (gv * fast_sigmoid(gv)) * uv;
                            if (ROWW) h[x][j][y] *= weight[ROWW ? i : 0][x];   // h = w[row] * silu(g) * u, one rounding
                        }
                    if (keep_gu) turn(acc[i][x][0], acc[i][x][1], acc[i][x][2], acc[i][x][3], chunk[x]);
                }
                if (keep_gu) store_gu(0);
                // h of the unit's upper 16 rows beside that of its lower ones
                turn(h[0][0], h[0][1], h[1][0], h[1][1], chunk[2]);
                if (keep_gu) store_gu(1);
#pragma unroll
                for (int y = 0; y < 2; y++) {
                    const int upper = lane_e & 4 ? 16 : 0;
                    if (all_rows || e_row_begin + chunk_m(i, y) + upper < row_lim)
                        *reinterpret_cast<u32x4 *>(chunk_at(h_out, i, y) + upper * e_ldc) = chunk[2][y];
                }
            } else {
                u32x4 chunk[2];
#pragma unroll
                for (int x = 0; x < 4; x++) {
                    if (x % 2 == 0) turn(acc[i][x >> 1][0], acc[i][x >> 1][1], acc[i][x >> 1][2], acc[i][x >> 1][3], chunk);
                    u32x4 v = chunk[x & 1];
                    const int m = e_row_begin + chunk_m(i, x);
                    if (EPI == EPI_SWIGLU_BWD) {
                        float dot = 0.0f;   // ROWW: this lane's part of sum_i dh[m][i] * silu(g[m][i]) * u[m][i]
                        if (all_rows || m < row_lim) {
                            float dh[8], gv[8], uv[8], dg[8], du[8];
                            Elem<uint16_t>::unpack(v, dh);
                            Elem<uint16_t>::unpack(g_in[GU ? i & 1 : 0][GU ? x : 0], gv);
                            Elem<uint16_t>::unpack(u_in[GU ? i & 1 : 0][GU ? x : 0], uv);
#pragma unroll
                            for (int y = 0; y < 8; y++) {
                                const float sg = fast_sigmoid(gv[y]);
                                const float sl = gv[y] * sg;
                                if (ROWW) {
                                    // acc is the gradient of w * silu(g) * u: the routing weight's gradient
                                    // is its product with silu(g) * u, the activation's gets the factor w
                                    dot += dh[y] * (sl * uv[y]);
                                    dh[y] *= w_in[GU ? i & 1 : 0][GU ? x : 0];
                                }
                                du[y] = dh[y] * sl;
                                dg[y] = (dh[y] * uv[y]) * (sg * (1.0f + gv[y] * (1.0f - sg)));
                            }
                            u32x4 vg, vu;
#pragma unroll
                            for (int y = 0; y < 4; y++) {
                                vg[y] = pack2_bf16(dg[2 * y], dg[2 * y + 1]);
                                vu[y] = pack2_bf16(du[2 * y], du[2 * y + 1]);
                            }
                            *reinterpret_cast<u32x4 *>(chunk_at(C, i, x)) = vg;
                            *reinterpret_cast<u32x4 *>(chunk_at(C1, i, x)) = vu;
                        }
                        if (ROWW) {   // this wavefront's column range of the row: its eight lanes in a fixed order
                            dot = eight_lanes_sum(dot);
                            if ((lane_e & 7) == 0 && m < row_lim && !e_dense) p.row_dot[(col0 / COLS) * p.rows + m] = dot;
                        }
                        if (x & 1) __builtin_amdgcn_sched_barrier(0);
                    } else if (all_rows || m < row_lim) {   // (all_rows: known to the compiler where old values are waited for)
                        if (ACCUM) {
                            float fresh[8], prev[8];
                            Elem<uint16_t>::unpack(v, fresh);
                            Elem<uint16_t>::unpack(old[ACCUM ? i : 0][ACCUM ? x : 0], prev);
#pragma unroll
                            for (int y = 0; y < 4; y++)
                                v[y] = pack2_bf16(prev[2 * y] + fresh[2 * y], prev[2 * y + 1] + fresh[2 * y + 1]);
                        }
                        u32x4 *to = reinterpret_cast<u32x4 *>(chunk_at(Cb, i, x));
                        if (decltype(past_caches)::value && !ACCUM)
                            store_past_caches(Cb + tile_at, (lane_at + static_cast<uint32_t>(i * 64 + x * 8) * static_cast<uint32_t>(e_ldc)) * 2, v);
                        else if (decltype(past_caches)::value) __builtin_nontemporal_store(v, to);
                        else *to = v;
                        if (ACCUM) __builtin_amdgcn_sched_barrier(0);   // (all of them at once spill registers)
                    }
                }
                if (GU && i + 2 < TM) load_gu(i + 2);
            }
        }
    };
    if (WGRAD && !EDGE && p.stream) rows_out(std::true_type{});
    else rows_out(std::false_type{});
    }  // tile loop
}

template <int BM, int AKIND, int BKIND, int EPI, int GATHER = GATHER_NONE, bool ROWW = false, bool ACCUM = false,
          bool EDGE = false, bool ONCE = false, bool DENSE = false>
__global__ __launch_bounds__(BM == 256 ? 512 : 256, BM == 128 ? 2 : 1) void ggemm_kernel(const GemmParams p) {
    using D = Tables<BM, EPI, GATHER, EDGE>;
    __shared__ __attribute__((aligned(1024))) char lds[D::LDS];
    __shared__ int idx_cache[D::IDX_CACHE];
    __shared__ int order[D::PARTS];
    __shared__ __attribute__((aligned(16))) Part part[D::PARTS];
    __shared__ int tile_end[D::ENDS];
    __shared__ int seg[D::SEGS];
    ggemm_tiles<BM, AKIND, BKIND, EPI, GATHER, ROWW, ACCUM, EDGE, ONCE, DENSE>(p, lds, idx_cache, order, part, tile_end, seg);
}


// The input gradient of gate and up and the three weight gradients of experts whose tiles are 128x128: independent of each other, so that
// the tiles of both share the rounds.  A block works through its row tiles and then, counted from the other end of its XCD's blocks,
// through its tiles of the weight gradients.
template <bool ACCUM> __global__ __launch_bounds__(256, 2) void ggemm_backward_kernel(const GemmParams rows, const GemmParams w) {
    using R = Tables<128, EPI_STORE, GATHER_NONE, true>;
    using W = Tables<128, EPI_WGRAD, MERGED, true>;
    static_assert(R::LDS == W::LDS, "the stages of one are the other's");
    __shared__ __attribute__((aligned(1024))) char lds[R::LDS];
    // the tables of one where the other's were
    struct RowTables { Part part[R::PARTS]; int order[R::PARTS], tile_end[R::ENDS], seg[R::SEGS]; };
    static_assert(sizeof(int[W::IDX_CACHE]) <= sizeof(RowTables), "as many blocks on a CU as of either kernel alone");
    __shared__ __attribute__((aligned(16))) char tables[sizeof(RowTables)];
    __shared__ Part no_part[1];
    __shared__ int none[1];
    RowTables &t = *reinterpret_cast<RowTables *>(tables);
    ggemm_tiles<128, CONTIG, STRIDED, EPI_STORE, GATHER_NONE, false, false, true, false, false>(rows, lds, none, t.order, t.part, t.tile_end, t.seg);
    __syncthreads();
    ggemm_tiles<128, STRIDED, STRIDED, EPI_WGRAD, MERGED, false, ACCUM, true, false, false, true>(
        w, lds, *reinterpret_cast<int (*)[W::IDX_CACHE]>(tables), none, no_part, none, none);
}

// ---- host side ---------------------------------------------------------------------------------

// Two tile shapes: 256x256 (8 wavefronts of 128x64) for the training shapes, 128x128 (4 wavefronts
// of 64x64) when an extent is not a multiple of 256 or experts hold few rows each.

inline bool mult(int64_t v, int m) { return v > 0 && v % m == 0; }
// Operands are addressed as a 64-bit block-uniform base plus a 32-bit lane offset, so their size is
// only bounded by int64 arithmetic on element counts (2^40 here, far beyond device memory); a source
// whose rows are fetched through an index has index * pitch in the lane offset and must span
// < 2^31 elements.  Per-expert pitches are multiples of 8 elements (16-byte vectors need that).
inline bool fits_span(int64_t elems) { return elems >= 0 && elems < (1LL << 40); }
inline bool fits_gather(int64_t elems) { return elems >= 0 && elems < (1LL << 31); }
inline bool pitch_ok(int64_t stride) { return stride >= 0 && stride % 8 == 0; }

// Blocks of a launch: one resident set (a multiple of the 8 XCDs), or fewer when there are few
// tiles.  The 256x256 tile's 128 KB of LDS leave room for one block per CU, the 128x128 tile's
// 64 KB for two.
// Compute units of the current device (256 on an MI355X in its default partition mode), asked from
// the runtime once per device.
inline int device_cu_count() {
    static int cached[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (cached[dev] == 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < NUM_XCD)
            n = 256;
        cached[dev] = n;
    }
    return cached[dev];
}
template <int BM> unsigned persistent_blocks(int64_t tiles) {
    const int64_t per_xcd_max = (device_cu_count() / NUM_XCD) * (BM == 256 ? 1 : 2);
    int64_t per_xcd = (tiles + NUM_XCD - 1) / NUM_XCD;
    if (per_xcd > per_xcd_max) per_xcd = per_xcd_max;
    if (per_xcd < 1) per_xcd = 1;
    return static_cast<unsigned>(per_xcd * NUM_XCD);
}


// CACHED_WEIGHTS: the caches hold 256 MB, and more than a launch's weights passes through them.  From there on (gate and up: 64 M
// elements each) the weights are kept out of them: the 128x128 row products load those of an expert with one row tile without
// leaving them there (rows of whole lines: om_weights_pass_caches), the 256x256 weight gradients are stored past them; what the caches held instead was written back or fetched again under
// the next products.  us, 64 experts of 1024/2048: 37 tokens gate+up 104 -> 93 (5.8 TB/s of weights), down 50 -> 44;
// 512 tokens, uneven, gate/up input gradient behind the weight gradients 167 -> 104, those 209 -> 214; 32 experts of 2048/7168, 64
// rows in all, 146 -> 133 and 84 -> 75.  Around the line, whole forward of 37 tokens, 64 experts, ffn 1024, nothing -> all three
// matrices past the caches: hidden 512 54 -> 58, 768 80 -> 76, 1280 119 -> 108, 1536 136 -> 116, 2048 169 -> 147, 3072 238 -> 206 (1280
// with the line 109); training steps of 512 tokens, gradients written: hidden 256 (48 M in all three) 171 -> 169, 512 239 -> 204 (the line
// leaves that out), 1024 377 -> 325, 1792 624 -> 542; added, within 1.5 %.  What loses by it are weights
// that a second row tile reads (12 experts of 712/1000, 750 rows each: gate+up 51 -> 82 when all were
// loaded so) and the saved g and u of the forward (prefill of 4096 tokens, gate+up 344 -> 354).

// XCDs that share an expert's row products: from 8 M weights a matrix on, four, or all eight with few experts, which two
// groups of XCDs could not divide evenly.  One expert alone needs no sharing: its tiles are alike.
inline int rows_share(const GemmParams &p, int64_t expected) {
    if (p.n_experts < 2 || p.n_experts > SHARE_MAX_EXPERTS || static_cast<int64_t>(p.n_cols) * p.kc < (8 << 20)) return 0;
    if (expected < 32 * static_cast<int64_t>(p.n_experts)) return 0;
    return p.n_experts >= 16 ? 4 : NUM_XCD;
}

template <int BM, int AKIND, int BKIND, int EPI, int GATHER = GATHER_NONE, bool ROWW = false>
int launch_rows(GemmParams &p, int64_t rows, int64_t expected, hipStream_t st) {  // fwd / dgrad family
    constexpr int BN_OUT = (EPI == EPI_SWIGLU) ? BM / 2 : BM;
    if (p.n_experts > MAX_EXPERTS) return OM_ERR_SHAPE;   // the tile table lives in LDS
    p.share = rows_share(p, expected);
    const int64_t m_tiles_max = (rows + BM - 1) / BM + p.n_experts;
    const int64_t tiles = m_tiles_max * ((p.n_cols + BN_OUT - 1) / BN_OUT);
    if (tiles > 0x7fffffffLL) return OM_ERR_SHAPE;
    const dim3 grid(persistent_blocks<BM>(tiles)), block(THREADS<BM>);
    const int64_t weights = static_cast<int64_t>(p.n_experts) * p.n_cols * p.kc * (EPI == EPI_SWIGLU ? 2 : p.phases);
    if (BM == 128 && om_weights_pass_caches(p.B[0], weights, p.ldb, p.strideB) &&
        om_weights_pass_caches(p.B[1], weights, p.ldb, p.strideB))   // (one matrix: a null B[1], nothing to check)
        ggemm_kernel<BM, AKIND, BKIND, EPI, GATHER, ROWW, false, BM == 128, BM == 128><<<grid, block, 0, st>>>(p);
    else
        ggemm_kernel<BM, AKIND, BKIND, EPI, GATHER, ROWW, false, BM == 128><<<grid, block, 0, st>>>(p);
    return om_launch_status();
}

// The tile shape launch_rows_auto picks: 256x256 when the output columns are a whole number of such
// tiles, the contraction a whole number of steps, the experts hold enough rows to fill them, and there are enough of them for at least half
// the CUs (a tiny problem is spread over more CUs by the 128x128 tile).  The 128x128 tile takes any
// extents and contraction lengths that are multiples of 8: its last column tile and its last
// contraction step may be partial.
//
// "Enough rows" per expert on average: 160, for the SwiGLU backward, which suffers most from uneven rows, 192; where an
// expert's matrix has 4 M weights or more, which the 128x128 tile reads once per 128 rows, 128 for gate+up and 112
// for the plain store.  (Gate+up of smaller experts loses against uneven rows when launched alone, below; in whole
// passes of 64 experts of 2048/1024 the 256x256 kernel is the better one at 160 to 175 rows: forward of 1330 tokens with
// popularity as rank^-0.6 2.3 % faster, training steps of 1400 tokens even 0.9 %, of 1330 as rank^-1.2 0.2 %.)
// Launches alone, us, 128x128 -> 256x256, even routing / rows spread
// as exp(0.8 N(0,1)).  32 experts of 7168/2048: gate+up at 112 rows 450 -> 399 / 531 -> 569, 144 rows 710 -> 450 /
// 642 -> 596, SwiGLU backward at 144 rows 348 -> 213 / 329 -> 357, gate/up input gradient at 80 rows 396 -> 420 /
// 486 -> 446, 112 rows 446 -> 430 / 603 -> 462, down 214 -> 210 / 258 -> 228.  64 experts of 2048/1024 at 176 rows:
// gate+up 186 -> 169 / 176 -> 199, SwiGLU backward 101 -> 80 / 99 -> 124, down 89 -> 73 / 86 -> 85, gate/up input
// gradient 179 -> 130 / 183 -> 169; at 112 rows down 64 -> 60 / 65 -> 77.
template <int EPI> bool uses_big_tile(int n_cols, int kc, int n_experts, int64_t rows) {
    constexpr int div = (EPI == EPI_SWIGLU) ? 2 : 1;
    const bool large = static_cast<int64_t>(n_cols) * kc >= (4 << 20);
    const int enough = EPI == EPI_SWIGLU_BWD ? 192 : !large ? 160 : EPI == EPI_SWIGLU ? 128 : 112;
    if (n_cols % (256 / div) != 0 || kc % BK != 0 || rows < static_cast<int64_t>(n_experts) * enough) return false;
    const int64_t tiles = ((rows + 255) / 256) * (n_cols / (256 / div));
    return tiles * 2 >= device_cu_count();
}

// Whether a dense expert rides in the launch of the routed ones: where both would be 128x128 tiles.  A shared expert with few
// rows is a launch of few blocks that each walk all of a long contraction (64 rows of 7168/2048: gate+up 42 us, down 15, in
// the streaming kernels; 128x128 tiles 65 and 21); beside the routed experts' tiles it costs what its weights take to arrive.
// Whole passes of 32 of 256 experts and the shared one, us, on its own -> riding.  7168/2048, forward of 16 tokens 211 -> 190, 64
// 279 -> 231, 128 361 -> 304, 315 431 -> 363; training steps of 16 1225 -> 1097, 128 1795 -> 1670, 400 2233 -> 2175, 1000 2938 ->
// 2843.  3000/1000, forward of 200 190 -> 154; 1024/256 of 600 94 -> 85, of 100 as before; steps of 3000/1000, 700 tokens 888 -> 810.
// Not where its own tiles fill the chip: 1200/1000, forward of 5000 267 -> 275.
template <int EPI> bool dense_rides(const GemmParams &p, int64_t expected, int64_t dense_rows) {
    constexpr int BN_OUT = (EPI == EPI_SWIGLU) ? 64 : 128;
    return p.n_experts < MAX_EXPERTS && rows_share(p, expected) == 0 && !uses_big_tile<EPI>(p.n_cols, p.kc, p.n_experts, expected) &&
           !uses_big_tile<EPI>(p.n_cols, p.kc, 1, dense_rows) &&
           (dense_rows + 127) / 128 * ((p.n_cols + BN_OUT - 1) / BN_OUT) < 2 * device_cu_count();
}
template <int AKIND, int BKIND, int EPI, int GATHER, bool ROWW>
int launch_rows_dense(GemmParams &p, int64_t rows, hipStream_t st) {
    constexpr int BN_OUT = (EPI == EPI_SWIGLU) ? 64 : 128;
    p.share = 0;
    const int64_t tiles = ((rows + 127) / 128 + p.n_experts + (p.dense.rows + 127) / 128) * ((p.n_cols + BN_OUT - 1) / BN_OUT);
    if (tiles > 0x7fffffffLL) return OM_ERR_SHAPE;
    const dim3 grid(persistent_blocks<128>(tiles)), block(THREADS<128>);
    const int64_t weights = static_cast<int64_t>(p.n_experts) * p.n_cols * p.kc * (EPI == EPI_SWIGLU ? 2 : p.phases);
    bool once = true;   // (one matrix: null second pointers, nothing to check)
    for (int i = 0; i < 2; i++)
        once &= om_weights_pass_caches(p.B[i], weights, p.ldb, p.strideB) && om_weights_pass_caches(p.dense.B[i], weights, p.ldb, 0);
    if (once) ggemm_kernel<128, AKIND, BKIND, EPI, GATHER, ROWW, false, true, true, true><<<grid, block, 0, st>>>(p);
    else ggemm_kernel<128, AKIND, BKIND, EPI, GATHER, ROWW, false, true, false, true><<<grid, block, 0, st>>>(p);
    return om_launch_status();
}

// The dense expert of an entry point's arguments; its operands are checked by the launch of its own where it does not ride.
bool dense_operands(GemmParams &p, const om_dense_expert *d) {
    for (const void *q : {d->a[0], d->a[1], d->w[0], d->w[1], static_cast<const void *>(d->c[0]), static_cast<const void *>(d->c[1]),
                          static_cast<const void *>(d->c[2]), d->g, d->u})
        if (!om_aligned16(q)) return false;
    p.dense = {{static_cast<const uint16_t *>(d->a[0]), static_cast<const uint16_t *>(d->a[1])},
               {static_cast<const uint16_t *>(d->w[0]), static_cast<const uint16_t *>(d->w[1])},
               static_cast<uint16_t *>(d->c[0]), static_cast<uint16_t *>(d->c[1]), static_cast<uint16_t *>(d->c[2]),
               static_cast<const uint16_t *>(d->g), static_cast<const uint16_t *>(d->u), static_cast<int>(d->rows)};
    return true;
}

// `rows` sizes the launch, `expected` (rows, or fewer where rows is a bound) selects the kernel.
template <int AKIND, int BKIND, int EPI, int GATHER = GATHER_NONE, bool ROWW = false>
int launch_rows_auto(GemmParams &p, int64_t rows, int64_t expected, hipStream_t st) {
    if (uses_big_tile<EPI>(p.n_cols, p.kc, p.n_experts, expected))
        return launch_rows<256, AKIND, BKIND, EPI, GATHER, ROWW>(p, rows, expected, st);
    if (p.n_cols % 8 != 0 || p.kc % 8 != 0) return OM_ERR_SHAPE;
    return launch_rows<128, AKIND, BKIND, EPI, GATHER, ROWW>(p, rows, expected, st);
}

}  // namespace

extern "C" int om_grouped_gemm_fwd(const void *input, const void *weight, void *output,
                                   const int32_t *cum_token_counts, int64_t rows, int G, int N, int K,
                                   int64_t w_stride, void *stream) {
    return om_grouped_gemm_fwd_bound(input, weight, output, cum_token_counts, rows, rows, G, N, K, w_stride, stream);
}

namespace {
int grouped_fwd_launch(const void *input, const void *weight, void *output, const int32_t *cum_token_counts, int64_t rows,
                       int64_t expected_rows, int G, int N, int K, int64_t w_stride, const om_dense_expert *dense, void *stream) {
    if (rows < 0 || expected_rows < 0 || expected_rows > rows || G < 1 || !mult(N, 8) || !mult(K, 8)) return OM_ERR_SHAPE;
    if (dense && (dense->rows < 1 || !fits_gather(dense->rows))) return OM_ERR_SHAPE;
    if (dense && (!dense->a[0] || !dense->w[0] || !dense->c[0] || !dense->cum)) return OM_ERR_NULL;
    auto dense_alone = [&]() {
        return grouped_fwd_launch(dense->a[0], dense->w[0], dense->c[0], dense->cum, dense->rows, dense->rows, 1, N, K, 0, nullptr, stream);
    };
    if (rows == 0) return dense ? dense_alone() : OM_OK;
    if (!input || !weight || !output || !cum_token_counts) return OM_ERR_NULL;
    if (!om_aligned16(input) || !om_aligned16(weight) || !om_aligned16(output)) return OM_ERR_ALIGN;
    GemmParams p = {};
    p.A[0] = static_cast<const uint16_t *>(input);
    p.B[0] = static_cast<const uint16_t *>(weight);
    p.C = static_cast<uint16_t *>(output);
    p.cum = cum_token_counts;
    p.lda = K; p.ldb = K; p.ldc = N;
    p.strideB = w_stride ? w_stride : static_cast<int64_t>(N) * K;
    if (!pitch_ok(p.strideB)) return OM_ERR_ALIGN;
    if (!fits_span(rows * K) || !fits_span(rows * N) || !fits_span(p.strideB * G)) return OM_ERR_SHAPE;
    const bool past_caches = om_weights_pass_caches(weight, static_cast<int64_t>(G) * N * K, K, p.strideB);
    const bool streams = G <= MAX_EXPERTS && om_ggemm_streams(expected_rows, G, N, past_caches);
    p.rows = rows; p.n_experts = G; p.n_cols = N; p.kc = K; p.phases = 1;
    if (dense && !streams && dense_rides<EPI_STORE>(p, expected_rows, dense->rows)) {
        if (!dense_operands(p, dense)) return OM_ERR_ALIGN;
        return launch_rows_dense<CONTIG, CONTIG, EPI_STORE, GATHER_NONE, false>(p, rows, om_stream(stream));
    }
    if (dense) {
        const int code = dense_alone();
        if (code != OM_OK) return code;
    }
    if (streams)
        return om_ggemm_stream_fwd(input, weight, output, cum_token_counts, rows, expected_rows, G, N, K, p.strideB,
                                   om_stream(stream));
    return launch_rows_auto<CONTIG, CONTIG, EPI_STORE>(p, rows, expected_rows, om_stream(stream));
}
}  // namespace

extern "C" int om_grouped_gemm_fwd_bound(const void *input, const void *weight, void *output,
                                         const int32_t *cum_token_counts, int64_t rows, int64_t expected_rows, int G,
                                         int N, int K, int64_t w_stride, void *stream) {
    return grouped_fwd_launch(input, weight, output, cum_token_counts, rows, expected_rows, G, N, K, w_stride, nullptr, stream);
}

extern "C" int om_grouped_gemm_fwd_dense(const void *input, const void *weight, void *output,
                                         const int32_t *cum_token_counts, int64_t rows, int64_t expected_rows, int G,
                                         int N, int K, int64_t w_stride, const om_dense_expert *dense, void *stream) {
    if (!dense) return OM_ERR_NULL;
    return grouped_fwd_launch(input, weight, output, cum_token_counts, rows, expected_rows, G, N, K, w_stride, dense, stream);
}

extern "C" int om_grouped_gemm_dgrad(const void *output_grad, const void *weight, void *input_grad,
                                     const int32_t *cum_token_counts, int64_t rows, int G, int N, int K,
                                     int64_t w_stride, void *stream) {
    if (rows < 0 || G < 1 || !mult(N, 8) || !mult(K, 8)) return OM_ERR_SHAPE;
    if (rows == 0) return OM_OK;
    if (!output_grad || !weight || !input_grad || !cum_token_counts) return OM_ERR_NULL;
    if (!om_aligned16(output_grad) || !om_aligned16(weight) || !om_aligned16(input_grad)) return OM_ERR_ALIGN;
    GemmParams p = {};
    p.A[0] = static_cast<const uint16_t *>(output_grad);
    p.B[0] = static_cast<const uint16_t *>(weight);
    p.C = static_cast<uint16_t *>(input_grad);
    p.cum = cum_token_counts;
    p.lda = N; p.ldb = K; p.ldc = K;
    p.strideB = w_stride ? w_stride : static_cast<int64_t>(N) * K;
    if (!pitch_ok(p.strideB)) return OM_ERR_ALIGN;
    if (!fits_span(rows * K) || !fits_span(rows * N) || !fits_span(p.strideB * G)) return OM_ERR_SHAPE;
    p.rows = rows; p.n_experts = G; p.n_cols = K; p.kc = N; p.phases = 1;
    return launch_rows_auto<CONTIG, STRIDED, EPI_STORE>(p, rows, rows, om_stream(stream));
}

namespace {
// 256x256 tiles for the weight gradients unless the `matrices` of [n, k] have too few to occupy half the CUs
bool wgrad_big_tile(int n, int k, int64_t matrices) {
    return n % 256 == 0 && k % 256 == 0 && matrices * (n / 256) * (k / 256) * 2 >= device_cu_count();
}

// XCDs that share an expert's weight gradient: all, where an eighth of its tiles is about a third of a round or more.  With few
// rows the writing form is stores alone, which whole experts per XCD do better; the accumulating form leaves out the experts
// without rows, and the rest has to be shared.  The three of 32 experts of 2048/7168 in one launch, us, shared -> not, rows even /
// as 1 / rank^1.2, writing: 8 rows in all 538 -> 483 / 531 -> 505, 128 rows 540 -> 524 / 531 -> 524, 512 rows 541 -> 523 / 550 -> 583,
// 2048 rows 625 -> 634 / 632 -> 684; accumulating: 1 row 114 -> 254, 64 rows 913 -> 1043 / 667 -> 768.  64 experts of 1024/2048,
// writing: 64 rows 161 -> 148 / 159 -> 132, 512 rows 162 -> 158 / 156 -> 161, 2048 rows 166 -> 164 / 177 -> 175.
// Around 12 tiles per XCD the two are near each other, even rows a little better alone and uneven ones shared: 64 rows an expert,
// not shared -> shared, even / uneven, writing: 48 tiles (64 experts of 1024/1024) 97 -> 100 / 110 -> 115, 72 149 -> 145 / 161 -> 152, 84 172 ->
// 168 / 175 -> 173, 96 199 -> 187 / 193 -> 195, 120 239 -> 231 / 245 -> 243, 144 275 -> 284 / 293 -> 284.
int wgrad_share(bool big, int tiles_e, int n_experts, int64_t rows, bool accumulate) {
    if (!accumulate && rows < 16 * static_cast<int64_t>(n_experts)) return 0;
    return big && tiles_e >= 12 * NUM_XCD && n_experts <= SHARE_MAX_EXPERTS ? NUM_XCD : 0;
}

constexpr int STREAM_MAX_PITCH = 1 << 21;   // elements; 256 rows of a tile span less than the 2^31 bytes of store_past_caches

// weight gradient; gather == GATHER_B: contraction row c of `input` is row index[c] of a
// [src_rows, K] matrix; gather == GATHER_WA: contraction row c of `output_grad` is row index[c] of a
// [src_rows, N] matrix (the token gather folded into the loads)
int wgrad_launch(const void *output_grad, const void *input, const int32_t *index, int gather,
                 int64_t src_rows, void *weight_grad, const int32_t *cum_token_counts, int64_t rows, int G,
                 int N, int K, int64_t w_stride, void *stream, bool accumulate = false, int64_t expected = -1) {
    if (rows < 0 || G < 1 || !mult(N, 8) || !mult(K, 8)) return OM_ERR_SHAPE;
    // rows == 0 (nothing routed to these experts): the activations may be empty tensors without
    // storage; the launch then only writes zeros
    if (!weight_grad || !cum_token_counts || (rows > 0 && (!output_grad || !input))) return OM_ERR_NULL;
    if (!om_aligned16(output_grad) || !om_aligned16(input) || !om_aligned16(weight_grad)) return OM_ERR_ALIGN;
    GemmParams p = {};
    p.A[0] = static_cast<const uint16_t *>(output_grad);  // [rows, N]: operand rows = n, c = row
    p.B[0] = static_cast<const uint16_t *>(input);        // [rows, K] (or [src_rows, K] through input_rows)
    p.C = static_cast<uint16_t *>(weight_grad);           // [G, N, K]
    p.cum = cum_token_counts;
    p.row_index = index;
    p.lda = N; p.ldb = K; p.ldc = K;
    p.strideC = w_stride ? w_stride : static_cast<int64_t>(N) * K;
    if (!pitch_ok(p.strideC)) return OM_ERR_ALIGN;
    if (!fits_span(rows * K) || !fits_span(rows * N) || !fits_span(p.strideC * G) ||
        !fits_gather(src_rows * (gather == GATHER_WA ? N : K)))
        return OM_ERR_SHAPE;
    p.rows = rows; p.n_experts = G; p.n_cols = K; p.kc = N; p.phases = 1;
    hipStream_t st = om_stream(stream);
    const bool big = wgrad_big_tile(N, K, G);
    p.tiles_e = big ? (N / 256) * (K / 256) : ((N + 127) / 128) * ((K + 127) / 128);
    p.share = wgrad_share(big, p.tiles_e, G, expected < 0 ? rows : expected, accumulate);
    p.stream = K <= STREAM_MAX_PITCH && om_weights_pass_caches(weight_grad, static_cast<int64_t>(G) * N * K, K, p.strideC);
    const int64_t tiles = static_cast<int64_t>(p.tiles_e) * G;
    if (tiles > 0x7fffffffLL) return OM_ERR_SHAPE;
    p.total_tiles = static_cast<int>(tiles);
    // ACCUM (C[g] = bf16(float(C[g]) + float(bf16(acc))) instead of C[g] = acc) is a template
    // parameter: the plain kernels carry none of it
#define OM_WGRAD(GATHER_KIND, ACC)                                                                               \
    do {                                                                                                         \
        if (big)                                                                                                 \
            ggemm_kernel<256, STRIDED, STRIDED, EPI_WGRAD, GATHER_KIND, false, ACC>                              \
                <<<dim3(persistent_blocks<256>(tiles)), dim3(THREADS<256>), 0, st>>>(p);                         \
        else                                                                                                     \
            ggemm_kernel<128, STRIDED, STRIDED, EPI_WGRAD, GATHER_KIND, false, ACC, true>                        \
                <<<dim3(persistent_blocks<128>(tiles)), dim3(THREADS<128>), 0, st>>>(p);                         \
    } while (0)
    if (accumulate) {
        if (gather == GATHER_NONE) OM_WGRAD(GATHER_NONE, true);
        else if (gather == GATHER_B) OM_WGRAD(GATHER_B, true);
        else OM_WGRAD(GATHER_WA, true);
    } else {
        if (gather == GATHER_NONE) OM_WGRAD(GATHER_NONE, false);
        else if (gather == GATHER_B) OM_WGRAD(GATHER_B, false);
        else OM_WGRAD(GATHER_WA, false);
    }
#undef OM_WGRAD
    return om_launch_status();
}
}  // namespace

extern "C" int om_grouped_gemm_wgrad(const void *output_grad, const void *input, void *weight_grad,
                                     const int32_t *cum_token_counts, int64_t rows, int G, int N, int K,
                                     int64_t w_stride, void *stream) {
    return wgrad_launch(output_grad, input, nullptr, GATHER_NONE, 0, weight_grad, cum_token_counts, rows, G,
                        N, K, w_stride, stream);
}

extern "C" int om_grouped_gemm_wgrad_gathered(const void *output_grad, const void *input,
                                              const int32_t *input_rows, int64_t src_rows,
                                              void *weight_grad, const int32_t *cum_token_counts,
                                              int64_t rows, int G, int N, int K, int64_t w_stride,
                                              void *stream) {
    if (!input_rows) return OM_ERR_NULL;
    if (src_rows < 1) return OM_ERR_SHAPE;
    return wgrad_launch(output_grad, input, input_rows, GATHER_B, src_rows, weight_grad, cum_token_counts,
                        rows, G, N, K, w_stride, stream);
}

extern "C" int om_grouped_gemm_wgrad_gathered_out(const void *output_grad, const int32_t *output_grad_rows,
                                                  int64_t src_rows, const void *input, void *weight_grad,
                                                  const int32_t *cum_token_counts, int64_t rows, int G,
                                                  int N, int K, int64_t w_stride, void *stream) {
    if (!output_grad_rows) return OM_ERR_NULL;
    if (src_rows < 1) return OM_ERR_SHAPE;
    return wgrad_launch(output_grad, input, output_grad_rows, GATHER_WA, src_rows, weight_grad,
                        cum_token_counts, rows, G, N, K, w_stride, stream);
}

// The accumulating forms: weight_grad += dW in the gradient's dtype, inside the epilogue.
extern "C" int om_grouped_gemm_wgrad_accumulate(const void *output_grad, const void *input, void *weight_grad,
                                                const int32_t *cum_token_counts, int64_t rows, int G, int N,
                                                int K, int64_t w_stride, void *stream) {
    return wgrad_launch(output_grad, input, nullptr, GATHER_NONE, 0, weight_grad, cum_token_counts, rows, G,
                        N, K, w_stride, stream, true);
}

extern "C" int om_grouped_gemm_wgrad_gathered_accumulate(const void *output_grad, const void *input,
                                                         const int32_t *input_rows, int64_t src_rows,
                                                         void *weight_grad, const int32_t *cum_token_counts,
                                                         int64_t rows, int G, int N, int K, int64_t w_stride,
                                                         void *stream) {
    if (!input_rows) return OM_ERR_NULL;
    if (src_rows < 1) return OM_ERR_SHAPE;
    return wgrad_launch(output_grad, input, input_rows, GATHER_B, src_rows, weight_grad, cum_token_counts,
                        rows, G, N, K, w_stride, stream, true);
}

extern "C" int om_grouped_gemm_wgrad_gathered_out_accumulate(const void *output_grad,
                                                             const int32_t *output_grad_rows, int64_t src_rows,
                                                             const void *input, void *weight_grad,
                                                             const int32_t *cum_token_counts, int64_t rows,
                                                             int G, int N, int K, int64_t w_stride,
                                                             void *stream) {
    if (!output_grad_rows) return OM_ERR_NULL;
    if (src_rows < 1) return OM_ERR_SHAPE;
    return wgrad_launch(output_grad, input, output_grad_rows, GATHER_WA, src_rows, weight_grad,
                        cum_token_counts, rows, G, N, K, w_stride, stream, true);
}

namespace {
// dW_down (+)= dout^T h, dW_gate (+)= dg^T x, dW_up (+)= du^T x, in one launch where that saves rounds of tiles: those of an
// expert's three gradients come one after the other.
// `beside`: the gate/up input gradient, whose tiles join the launch where it is one of 128x128 tiles; *joined says whether they did.
int wgrad_merged_launch(const void *dout, const int32_t *dout_rows, const void *h, const void *dg, const void *du, const void *x,
                        const int32_t *x_rows, int64_t src_rows, void *dw_down, void *dw_gate, void *dw_up,
                        const int32_t *cum_token_counts, int64_t rows, int64_t expected, int G, int I, int H, int64_t down_stride,
                        int64_t gate_stride, int64_t up_stride, bool accumulate, void *stream, const GemmParams *beside = nullptr,
                        bool *joined = nullptr) {
    if (rows < 0 || expected < 0 || expected > rows || G < 1 || !mult(I, 8) || !mult(H, 8)) return OM_ERR_SHAPE;
    if (!dw_down || !dw_gate || !dw_up || !cum_token_counts || (rows > 0 && (!dout || !h || !dg || !du || !x))) return OM_ERR_NULL;
    if ((dout_rows || x_rows) && src_rows < 1) return OM_ERR_SHAPE;
    GemmParams p = {};
    const int64_t packed = static_cast<int64_t>(I) * H;
    auto set = [&](int i, const void *a, const int32_t *a_rows, const void *b, const int32_t *b_rows, void *c, int64_t stride, int m, int n) {
        p.set[i] = {static_cast<const uint16_t *>(a), static_cast<const uint16_t *>(b), static_cast<uint16_t *>(c), a_rows, b_rows,
                    stride ? stride : packed, m, n};
        return om_aligned16(a) && om_aligned16(b) && om_aligned16(c) && pitch_ok(p.set[i].strideC);
    };
    if (!set(0, dout, dout_rows, h, nullptr, dw_down, down_stride, H, I) || !set(1, dg, nullptr, x, x_rows, dw_gate, gate_stride, I, H) ||
        !set(2, du, nullptr, x, x_rows, dw_up, up_stride, I, H))
        return OM_ERR_ALIGN;
    if (!fits_span(rows * H) || !fits_span(rows * I) || ((dout_rows || x_rows) && !fits_gather(src_rows * H))) return OM_ERR_SHAPE;
    for (const WgradSet &s : p.set)
        if (!fits_span(s.strideC * G)) return OM_ERR_SHAPE;
    p.cum = cum_token_counts;
    p.rows = rows; p.n_experts = G; p.phases = 1;
    const bool big = wgrad_big_tile(H, I, 3 * static_cast<int64_t>(G));
    const int tile = big ? 256 : 128;
    const int64_t each = static_cast<int64_t>((H + tile - 1) / tile) * ((I + tile - 1) / tile), tiles = 3 * each * G;
    if (tiles > 0x7fffffffLL) return OM_ERR_SHAPE;
    // One launch where it saves rounds of tiles, and more of them than the tenth that its kernel is slower by (its operands
    // are chosen per tile): 12 experts of 1000x712, 576 tiles a product on 512 blocks, 103 -> 72 us; 8 of 256x512, 64
    // tiles, 38 -> 16.  One of 7168x2048, 224 tiles on 256 blocks and as many rounds either way, 698 -> 774; 64 of
    // 2048x1024 with 2048 rows, 2048 tiles, 1620 -> 1701.  With few rows an expert, where a launch is stores and its ends
    // weigh more, one launch as well: those 64 experts with 64 rows each on average, a step of 512 tokens 717 -> 696.  But not with
    // many rounds of 128x128 tiles, beside which the ends weigh little.  One -> three launches, us: 64 experts of 1048x1712, 48 rounds,
    // writing 64 rows in all 219 -> 204, 2048 rows 251 -> 244, 8192 rows 361 -> 330, accumulating 299 -> 290, 354 -> 357, 440 -> 415; 16 of
    // 1104x3736, 26 rounds, writing 64 rows 132 -> 118, 2048 203 -> 179, accumulating 193 -> 210, 253 -> 244; 16 of 688x2304, 11 rounds, writing
    // 50 -> 53, 72 -> 67; 48 of 520x1400, 16 rounds (18 in three), writing 67 -> 69, 70 -> 70, accumulating 95 -> 104, 97 -> 111.
    // Nor from 128 rows an expert on with many rounds of 256x256 tiles that are written, of experts that the XCDs share in each launch
    // (those that they share in one launch only, 128 of 1024x2048, gain by that: uneven 256 rows 992 -> 750).  One -> three, even rows
    // / as 1 / rank^1.2: 32 of 2048x7168, 84 rounds, 64 rows 583 -> 605 / 662 -> 645, 128 rows 771 -> 755 / 788 -> 753, 256 rows 1171 -> 1058 /
    // 1198 -> 1060; 16 of them, 42 rounds, 64 rows 296 -> 308 / 329 -> 323, 128 rows 390 -> 380 / 415 -> 395, 256 rows 560 -> 525 / 561 ->
    // 541; 64 of 2048x4096, 96 rounds, 128 rows 880 -> 870 / 914 -> 912, 256 rows 1322 -> 1245 / 1392 -> 1315; 32 of 1536x5120, 45 rounds,
    // 128 rows 408 -> 407 / 428 -> 428, 256 rows 605 -> 581 / 603 -> 602; 8 of 2048x7168, 21 rounds, 256 rows 282 -> 307 / 309 -> 308.
    // Adding, 32 of 2048x7168, 128 rows 1213 -> 1208 / 1276 -> 1272, others slower in three.
    const int64_t blocks = static_cast<int64_t>(device_cu_count()) * (big ? 1 : 2);
    auto rounds = [](int64_t t, int64_t b) { return (t + b - 1) / b; };
    const bool big_alone = wgrad_big_tile(H, I, G);
    const int64_t alone = static_cast<int64_t>((H + (big_alone ? 255 : 127)) / (big_alone ? 256 : 128)) *
                          ((I + (big_alone ? 255 : 127)) / (big_alone ? 256 : 128)) * G;
    const int64_t blocks_alone = static_cast<int64_t>(device_cu_count()) * (big_alone ? 1 : 2);
    // Gradients with memory in common (two of the weights are one parameter) are written, or added to, one after another.
    bool overlap = false;
    for (int i = 0; i < 3; i++) {
        const WgradSet &a = p.set[i], &b = p.set[(i + 1) % 3];
        overlap |= om_blocks_overlap(a.C, a.strideC * 2, packed * 2, b.C, b.strideC * 2, packed * 2, G);
    }
    const bool no_fewer_rounds = big == big_alone && 11 * rounds(tiles, blocks) >= 10 * 3 * rounds(alone, blocks_alone);
    const bool many_rounds = !big && rounds(tiles, blocks) > (accumulate ? 32 : 16);
    const bool large = big && !accumulate && rounds(tiles, blocks) > 32 && each >= 12 * NUM_XCD;
    if (overlap || (no_fewer_rounds && (many_rounds || expected > 256 * static_cast<int64_t>(G) || (large && expected >= 128 * static_cast<int64_t>(G))))) {
        const int gather_d = dout_rows ? GATHER_WA : GATHER_NONE, gather_x = x_rows ? GATHER_B : GATHER_NONE;
        int code = wgrad_launch(dout, h, dout_rows, gather_d, dout_rows ? src_rows : 0, dw_down, cum_token_counts, rows, G, H, I,
                                down_stride, stream, accumulate, expected);
        if (code == OM_OK)
            code = wgrad_launch(dg, x, x_rows, gather_x, x_rows ? src_rows : 0, dw_gate, cum_token_counts, rows, G, I, H,
                                gate_stride, stream, accumulate, expected);
        if (code == OM_OK)
            code = wgrad_launch(du, x, x_rows, gather_x, x_rows ? src_rows : 0, dw_up, cum_token_counts, rows, G, I, H,
                                up_stride, stream, accumulate, expected);
        return code;
    }
    p.tiles_e = static_cast<int>(3 * each);
    p.share = wgrad_share(big, p.tiles_e, G, expected, accumulate);
    p.stream = true;
    for (const WgradSet &s : p.set) p.stream &= s.n <= STREAM_MAX_PITCH && om_weights_pass_caches(s.C, 3 * packed * G, s.n, s.strideC);
    p.total_tiles = static_cast<int>(tiles);
    hipStream_t st = om_stream(stream);
    if (beside && !big) {
        const int64_t row_tiles = ((rows + 127) / 128 + G) * ((H + 127) / 128);
        const dim3 both(persistent_blocks<128>(tiles + row_tiles));
        *joined = true;
        if (accumulate) ggemm_backward_kernel<true><<<both, dim3(THREADS<128>), 0, st>>>(*beside, p);
        else ggemm_backward_kernel<false><<<both, dim3(THREADS<128>), 0, st>>>(*beside, p);
        return om_launch_status();
    }
    const dim3 grid(big ? persistent_blocks<256>(tiles) : persistent_blocks<128>(tiles)), block(big ? THREADS<256> : THREADS<128>);
    if (big && accumulate) ggemm_kernel<256, STRIDED, STRIDED, EPI_WGRAD, MERGED, false, true><<<grid, block, 0, st>>>(p);
    else if (big) ggemm_kernel<256, STRIDED, STRIDED, EPI_WGRAD, MERGED><<<grid, block, 0, st>>>(p);
    else if (accumulate) ggemm_kernel<128, STRIDED, STRIDED, EPI_WGRAD, MERGED, false, true, true><<<grid, block, 0, st>>>(p);
    else ggemm_kernel<128, STRIDED, STRIDED, EPI_WGRAD, MERGED, false, false, true><<<grid, block, 0, st>>>(p);
    return om_launch_status();
}
}  // namespace

extern "C" int om_grouped_gemm_wgrad_merged(const void *dout, const int32_t *dout_rows, const void *h, const void *dg,
                                            const void *du, const void *x, const int32_t *x_rows, int64_t src_rows,
                                            void *dw_down, void *dw_gate, void *dw_up, const int32_t *cum_token_counts,
                                            int64_t rows, int G, int I, int H, int64_t down_stride,
                                            int64_t gate_stride, int64_t up_stride, void *stream) {
    return wgrad_merged_launch(dout, dout_rows, h, dg, du, x, x_rows, src_rows, dw_down, dw_gate, dw_up,
                               cum_token_counts, rows, rows, G, I, H, down_stride, gate_stride, up_stride, false, stream);
}

extern "C" int om_grouped_gemm_wgrad_merged_accumulate(const void *dout, const int32_t *dout_rows, const void *h,
                                                       const void *dg, const void *du, const void *x,
                                                       const int32_t *x_rows, int64_t src_rows, void *dw_down,
                                                       void *dw_gate, void *dw_up, const int32_t *cum_token_counts,
                                                       int64_t rows, int G, int I, int H, int64_t down_stride,
                                                       int64_t gate_stride, int64_t up_stride, void *stream) {
    return wgrad_merged_launch(dout, dout_rows, h, dg, du, x, x_rows, src_rows, dw_down, dw_gate, dw_up,
                               cum_token_counts, rows, rows, G, I, H, down_stride, gate_stride, up_stride, true, stream);
}

extern "C" int om_grouped_gemm_wgrad_merged_bound(const void *dout, const int32_t *dout_rows, const void *h, const void *dg,
                                            const void *du, const void *x, const int32_t *x_rows, int64_t src_rows,
                                            void *dw_down, void *dw_gate, void *dw_up, const int32_t *cum_token_counts,
                                            int64_t rows, int64_t expected_rows, int G, int I, int H, int64_t down_stride,
                                            int64_t gate_stride, int64_t up_stride, void *stream) {
    return wgrad_merged_launch(dout, dout_rows, h, dg, du, x, x_rows, src_rows, dw_down, dw_gate, dw_up,
                               cum_token_counts, rows, expected_rows, G, I, H, down_stride, gate_stride, up_stride, false, stream);
}

extern "C" int om_grouped_gemm_wgrad_merged_accumulate_bound(const void *dout, const int32_t *dout_rows, const void *h,
                                                       const void *dg, const void *du, const void *x,
                                                       const int32_t *x_rows, int64_t src_rows, void *dw_down,
                                                       void *dw_gate, void *dw_up, const int32_t *cum_token_counts,
                                                       int64_t rows, int64_t expected_rows, int G, int I, int H, int64_t down_stride,
                                                       int64_t gate_stride, int64_t up_stride, void *stream) {
    return wgrad_merged_launch(dout, dout_rows, h, dg, du, x, x_rows, src_rows, dw_down, dw_gate, dw_up,
                               cum_token_counts, rows, expected_rows, G, I, H, down_stride, gate_stride, up_stride, true, stream);
}

namespace {
// `x_rows` != null: sorted row r of the activations is row x_rows[r] of x [src_rows, H]
// `row_weights` != null (needs x_rows): h = row_weights[r] * silu(g) * u
int gate_up_fwd_launch(const void *x, const int32_t *x_rows, int64_t src_rows, const void *w_gate,
                       const void *w_up, const float *row_weights, void *g, void *u, void *h,
                       const int32_t *cum_token_counts, int64_t rows, int64_t expected, int G, int I, int H,
                       int64_t w_stride, void *stream, const om_dense_expert *dense = nullptr, bool hidden_only = false) {
    if (rows < 0 || expected < 0 || expected > rows || G < 1 || !mult(I, 8) || !mult(H, 8)) return OM_ERR_SHAPE;
    if (dense && (dense->rows < 1 || !fits_gather(dense->rows * H))) return OM_ERR_SHAPE;
    if (dense && (!dense->a[0] || !dense->w[0] || !dense->w[1] || !dense->c[2] || !dense->cum)) return OM_ERR_NULL;
    if (dense && !hidden_only && (!dense->c[0] || !dense->c[1])) return OM_ERR_NULL;
    auto dense_alone = [&]() {
        return gate_up_fwd_launch(dense->a[0], nullptr, 0, dense->w[0], dense->w[1], nullptr, dense->c[0], dense->c[1], dense->c[2],
                                  dense->cum, dense->rows, dense->rows, 1, I, H, 0, stream, nullptr, hidden_only);
    };
    if (rows == 0) return dense ? dense_alone() : OM_OK;
    if (!x || !w_gate || !w_up || (!hidden_only && (!g || !u)) || !h || !cum_token_counts) return OM_ERR_NULL;
    if (!om_aligned16(x) || !om_aligned16(w_gate) || !om_aligned16(w_up) || !om_aligned16(g) ||
        !om_aligned16(u) || !om_aligned16(h))
        return OM_ERR_ALIGN;
    GemmParams p = {};
    p.A[0] = static_cast<const uint16_t *>(x);
    p.B[0] = static_cast<const uint16_t *>(w_gate);
    p.B[1] = static_cast<const uint16_t *>(w_up);
    p.C = static_cast<uint16_t *>(g);
    p.C1 = static_cast<uint16_t *>(u);
    p.C2 = static_cast<uint16_t *>(h);
    p.cum = cum_token_counts;
    p.row_index = x_rows;
    p.row_scale = row_weights;
    p.lda = H; p.ldb = H; p.ldc = I;
    p.strideB = w_stride ? w_stride : static_cast<int64_t>(I) * H;
    if (!pitch_ok(p.strideB)) return OM_ERR_ALIGN;
    if (!fits_span(rows * H) || !fits_span(rows * I) || !fits_span(p.strideB * G) || !fits_gather(src_rows * H))
        return OM_ERR_SHAPE;
    const int64_t weights = 2 * static_cast<int64_t>(G) * I * H;
    const bool past_caches = om_weights_pass_caches(w_gate, weights, H, p.strideB) && om_weights_pass_caches(w_up, weights, H, p.strideB);
    const bool streams = G <= MAX_EXPERTS && om_ggemm_streams(expected, G, 2 * I, past_caches);
    if (dense) {
        p.n_experts = G; p.n_cols = I; p.kc = H; p.phases = 1; p.rows = rows;
        if (!streams && dense_rides<EPI_SWIGLU>(p, expected, dense->rows)) {
            if (!dense_operands(p, dense)) return OM_ERR_ALIGN;
            return launch_rows_dense<CONTIG, CONTIG, EPI_SWIGLU, GATHER_A, true>(p, rows, om_stream(stream));
        }
        const int code = dense_alone();
        if (code != OM_OK) return code;
    }
    if (streams)
        return om_ggemm_stream_gate_up(x, x_rows, w_gate, w_up, row_weights, g, u, h, cum_token_counts, rows, expected, G, I,
                                       H, p.strideB, om_stream(stream));
    p.rows = rows; p.n_experts = G; p.n_cols = I; p.kc = H; p.phases = 1;
    if (row_weights)
        return launch_rows_auto<CONTIG, CONTIG, EPI_SWIGLU, GATHER_A, true>(p, rows, expected, om_stream(stream));
    if (x_rows) return launch_rows_auto<CONTIG, CONTIG, EPI_SWIGLU, GATHER_A>(p, rows, expected, om_stream(stream));
    return launch_rows_auto<CONTIG, CONTIG, EPI_SWIGLU>(p, rows, expected, om_stream(stream));
}
}  // namespace

extern "C" int om_merged_mlp_gate_up_fwd(const void *x, const void *w_gate, const void *w_up, void *g,
                                         void *u, void *h, const int32_t *cum_token_counts,
                                         int64_t rows, int G, int I, int H, int64_t w_stride,
                                         void *stream) {
    return gate_up_fwd_launch(x, nullptr, 0, w_gate, w_up, nullptr, g, u, h, cum_token_counts, rows, rows, G, I,
                              H, w_stride, stream);
}

extern "C" int om_merged_mlp_gate_up_fwd_gathered(const void *x, const int32_t *x_rows, int64_t src_rows,
                                                  const void *w_gate, const void *w_up, void *g, void *u,
                                                  void *h, const int32_t *cum_token_counts,
                                                  int64_t rows, int G, int I, int H, int64_t w_stride,
                                                  void *stream) {
    if (rows > 0 && !x_rows) return OM_ERR_NULL;
    if (src_rows < 1 && rows > 0) return OM_ERR_SHAPE;
    return gate_up_fwd_launch(x, x_rows, src_rows, w_gate, w_up, nullptr, g, u, h, cum_token_counts, rows,
                              rows, G, I, H, w_stride, stream);
}

extern "C" int om_merged_mlp_gate_up_fwd_weighted(const void *x, const int32_t *x_rows, int64_t src_rows,
                                                  const void *w_gate, const void *w_up,
                                                  const float *row_weights, void *g, void *u, void *h,
                                                  const int32_t *cum_token_counts, int64_t rows, int G,
                                                  int I, int H, int64_t w_stride, void *stream) {
    return om_merged_mlp_gate_up_fwd_weighted_bound(x, x_rows, src_rows, w_gate, w_up, row_weights, g, u, h,
                                                    cum_token_counts, rows, rows, G, I, H, w_stride, stream);
}

extern "C" int om_merged_mlp_gate_up_fwd_weighted_bound(const void *x, const int32_t *x_rows, int64_t src_rows,
                                                        const void *w_gate, const void *w_up,
                                                        const float *row_weights, void *g, void *u, void *h,
                                                        const int32_t *cum_token_counts, int64_t rows,
                                                        int64_t expected_rows, int G, int I, int H, int64_t w_stride,
                                                        void *stream) {
    if (rows > 0 && (!x_rows || !row_weights)) return OM_ERR_NULL;
    if (src_rows < 1 && rows > 0) return OM_ERR_SHAPE;
    return gate_up_fwd_launch(x, x_rows, src_rows, w_gate, w_up, row_weights, g, u, h, cum_token_counts,
                              rows, expected_rows, G, I, H, w_stride, stream);
}

extern "C" int om_merged_mlp_gate_up_fwd_weighted_dense(const void *x, const int32_t *x_rows, int64_t src_rows,
                                                        const void *w_gate, const void *w_up,
                                                        const float *row_weights, void *g, void *u, void *h,
                                                        const int32_t *cum_token_counts, int64_t rows,
                                                        int64_t expected_rows, int G, int I, int H, int64_t w_stride,
                                                        const om_dense_expert *dense, void *stream) {
    if (!dense || (rows > 0 && (!x_rows || !row_weights))) return OM_ERR_NULL;
    if (src_rows < 1 && rows > 0) return OM_ERR_SHAPE;
    return gate_up_fwd_launch(x, x_rows, src_rows, w_gate, w_up, row_weights, g, u, h, cum_token_counts,
                              rows, expected_rows, G, I, H, w_stride, stream, dense);
}

extern "C" int om_merged_mlp_hidden_fwd(const void *x, const int32_t *x_rows, int64_t src_rows, const void *w_gate,
                                        const void *w_up, const float *row_weights, void *h,
                                        const int32_t *cum_token_counts, int64_t rows, int64_t expected_rows, int G, int I,
                                        int H, int64_t w_stride, const om_dense_expert *dense, void *stream) {
    if ((row_weights || dense) && rows > 0 && (!x_rows || !row_weights)) return OM_ERR_NULL;
    if (x_rows && src_rows < 1 && rows > 0) return OM_ERR_SHAPE;
    om_dense_expert hidden = {};
    if (dense) {
        hidden = *dense;
        hidden.c[0] = hidden.c[1] = nullptr;
    }
    return gate_up_fwd_launch(x, x_rows, x_rows ? src_rows : 0, w_gate, w_up, row_weights, nullptr, nullptr, h, cum_token_counts,
                              rows, expected_rows, G, I, H, w_stride, stream, dense ? &hidden : nullptr, true);
}

extern "C" int om_merged_mlp_dense_products(int64_t expected_rows, int G, int I, int H, int64_t dense_rows) {
    if (expected_rows < 0 || G < 1 || !mult(I, 8) || !mult(H, 8) || dense_rows < 1) return OM_ERR_SHAPE;
    GemmParams up = {}, down = {};   // of extents [I] x H and [H] x I
    up.n_experts = down.n_experts = G;
    up.n_cols = down.kc = I; up.kc = down.n_cols = H;
    const int64_t weights = static_cast<int64_t>(G) * I * H;     // (whether they pass the caches: as far as sizes say)
    const bool up_streams = om_ggemm_streams(expected_rows, G, 2 * I, 2 * weights >= CACHED_WEIGHTS && H % 64 == 0);
    const bool down_streams = om_ggemm_streams(expected_rows, G, H, weights >= CACHED_WEIGHTS && I % 64 == 0);
    return (!up_streams && dense_rides<EPI_SWIGLU>(up, expected_rows, dense_rows) ? OM_DENSE_GATE_UP : 0) |
           (!down_streams && dense_rides<EPI_STORE>(down, expected_rows, dense_rows) ? OM_DENSE_DOWN : 0) |
           (dense_rides<EPI_SWIGLU_BWD>(up, expected_rows, dense_rows) ? OM_DENSE_DOWN_DGRAD : 0) |
           (dense_rides<EPI_STORE>(down, expected_rows, dense_rows) ? OM_DENSE_GATE_UP_DGRAD : 0);
}

extern "C" int om_merged_mlp_dense_rides(int64_t expected_rows, int G, int I, int H, int64_t dense_rows) {
    const int products = om_merged_mlp_dense_products(expected_rows, G, I, H, dense_rows);
    return products < 0 ? products : products & OM_DENSE_GATE_UP ? 1 : 0;
}

namespace {
// columns of the intermediate size that one wavefront's epilogue covers (both tile shapes): the
// granularity of the row_dot partial sums
constexpr int ROW_DOT_COLS = 64;
static_assert(256 / WAVES_N<256> == ROW_DOT_COLS && 128 / WAVES_N<128> == ROW_DOT_COLS, "row_dot layout");

// `dy_rows` != null: sorted row r of dy is row dy_rows[r] of a [src_rows, H] matrix, the result is
// scaled by row_weights[r] and row_dot receives the partial sums of (dy W) * silu(g) * u
int down_dgrad_launch(const void *dy, const int32_t *dy_rows, int64_t src_rows, const void *w_down,
                      const void *g, const void *u, const float *row_weights, void *dg, void *du,
                      float *row_dot, const int32_t *cum_token_counts, int64_t rows, int64_t expected, int G, int I,
                      int H, int64_t w_stride, void *stream, const om_dense_expert *dense = nullptr) {
    if (rows < 0 || expected < 0 || expected > rows || G < 1 || !mult(I, 8) || !mult(H, 8)) return OM_ERR_SHAPE;
    if (dense && (dense->rows < 1 || !fits_gather(dense->rows * H))) return OM_ERR_SHAPE;
    if (dense && (!dense->a[0] || !dense->w[0] || !dense->c[0] || !dense->c[1] || !dense->g || !dense->u || !dense->cum)) return OM_ERR_NULL;
    auto dense_alone = [&]() {
        return down_dgrad_launch(dense->a[0], nullptr, 0, dense->w[0], dense->g, dense->u, nullptr, dense->c[0], dense->c[1], nullptr,
                                 dense->cum, dense->rows, dense->rows, 1, I, H, 0, stream);
    };
    if (rows == 0) return dense ? dense_alone() : OM_OK;
    if (!dy || !w_down || !g || !u || !dg || !du || !cum_token_counts) return OM_ERR_NULL;
    if (!om_aligned16(dy) || !om_aligned16(w_down) || !om_aligned16(g) || !om_aligned16(u) ||
        !om_aligned16(dg) || !om_aligned16(du))
        return OM_ERR_ALIGN;
    GemmParams p = {};
    p.A[0] = static_cast<const uint16_t *>(dy);      // [rows, H]
    p.B[0] = static_cast<const uint16_t *>(w_down);  // [G, H, I]: c = h, operand row = i
    p.C = static_cast<uint16_t *>(dg);
    p.C1 = static_cast<uint16_t *>(du);
    p.G = static_cast<const uint16_t *>(g);
    p.U = static_cast<const uint16_t *>(u);
    p.cum = cum_token_counts;
    p.row_index = dy_rows;
    p.row_scale = row_weights;
    p.row_dot = row_dot;
    p.lda = H; p.ldb = I; p.ldc = I;
    p.strideB = w_stride ? w_stride : static_cast<int64_t>(H) * I;
    if (!pitch_ok(p.strideB)) return OM_ERR_ALIGN;
    if (!fits_span(rows * H) || !fits_span(rows * I) || !fits_span(p.strideB * G) || !fits_gather(src_rows * H))
        return OM_ERR_SHAPE;
    p.rows = rows; p.n_experts = G; p.n_cols = I; p.kc = H; p.phases = 1;
    if (dense) {
        if (dense_rides<EPI_SWIGLU_BWD>(p, expected, dense->rows)) {
            if (!dense_operands(p, dense)) return OM_ERR_ALIGN;
            return launch_rows_dense<CONTIG, STRIDED, EPI_SWIGLU_BWD, GATHER_A, true>(p, rows, om_stream(stream));
        }
        const int code = dense_alone();
        if (code != OM_OK) return code;
    }
    if (dy_rows)
        return launch_rows_auto<CONTIG, STRIDED, EPI_SWIGLU_BWD, GATHER_A, true>(p, rows, expected, om_stream(stream));
    return launch_rows_auto<CONTIG, STRIDED, EPI_SWIGLU_BWD>(p, rows, expected, om_stream(stream));
}
}  // namespace

extern "C" int om_merged_mlp_down_dgrad(const void *dy, const void *w_down, const void *g, const void *u,
                                        void *dg, void *du, const int32_t *cum_token_counts,
                                        int64_t rows, int G, int I, int H, int64_t w_stride,
                                        void *stream) {
    return down_dgrad_launch(dy, nullptr, 0, w_down, g, u, nullptr, dg, du, nullptr, cum_token_counts, rows,
                             rows, G, I, H, w_stride, stream);
}

extern "C" int om_merged_mlp_row_dot_parts(int I) {
    if (I < 8 || I % 8 != 0) return OM_ERR_SHAPE;
    return (I + ROW_DOT_COLS - 1) / ROW_DOT_COLS;
}

extern "C" int om_merged_mlp_down_dgrad_weighted(const void *dy, const int32_t *dy_rows, int64_t src_rows,
                                                 const void *w_down, const void *g, const void *u,
                                                 const float *row_weights, void *dg, void *du,
                                                 float *row_dot, const int32_t *cum_token_counts,
                                                 int64_t rows, int G, int I, int H, int64_t w_stride,
                                                 void *stream) {
    return om_merged_mlp_down_dgrad_weighted_bound(dy, dy_rows, src_rows, w_down, g, u, row_weights, dg, du, row_dot,
                                                   cum_token_counts, rows, rows, G, I, H, w_stride, stream);
}

extern "C" int om_merged_mlp_down_dgrad_weighted_bound(const void *dy, const int32_t *dy_rows, int64_t src_rows,
                                                       const void *w_down, const void *g, const void *u,
                                                       const float *row_weights, void *dg, void *du,
                                                       float *row_dot, const int32_t *cum_token_counts,
                                                       int64_t rows, int64_t expected_rows, int G, int I, int H,
                                                       int64_t w_stride, void *stream) {
    if (rows > 0 && (!dy_rows || !row_weights || !row_dot)) return OM_ERR_NULL;
    if (src_rows < 1 && rows > 0) return OM_ERR_SHAPE;
    return down_dgrad_launch(dy, dy_rows, src_rows, w_down, g, u, row_weights, dg, du, row_dot,
                             cum_token_counts, rows, expected_rows, G, I, H, w_stride, stream);
}

extern "C" int om_merged_mlp_down_dgrad_weighted_dense(const void *dy, const int32_t *dy_rows, int64_t src_rows,
                                                       const void *w_down, const void *g, const void *u,
                                                       const float *row_weights, void *dg, void *du,
                                                       float *row_dot, const int32_t *cum_token_counts,
                                                       int64_t rows, int64_t expected_rows, int G, int I, int H,
                                                       int64_t w_stride, const om_dense_expert *dense, void *stream) {
    if (!dense || (rows > 0 && (!dy_rows || !row_weights || !row_dot))) return OM_ERR_NULL;
    if (src_rows < 1 && rows > 0) return OM_ERR_SHAPE;
    return down_dgrad_launch(dy, dy_rows, src_rows, w_down, g, u, row_weights, dg, du, row_dot,
                             cum_token_counts, rows, expected_rows, G, I, H, w_stride, stream, dense);
}

extern "C" int om_merged_mlp_gate_up_dgrad(const void *dg, const void *du, const void *w_gate,
                                           const void *w_up, void *dx, const int32_t *cum_token_counts,
                                           int64_t rows, int G, int I, int H, int64_t w_stride,
                                           void *stream) {
    return om_merged_mlp_gate_up_dgrad_bound(dg, du, w_gate, w_up, dx, cum_token_counts, rows, rows, G, I, H, w_stride,
                                             stream);
}

namespace {
// The product's operands, checked; rows > 0.
int gate_up_dgrad_params(const void *dg, const void *du, const void *w_gate, const void *w_up, void *dx, const int32_t *cum_token_counts,
                         int64_t rows, int G, int I, int H, int64_t w_stride, GemmParams &p) {
    if (!dg || !du || !w_gate || !w_up || !dx || !cum_token_counts) return OM_ERR_NULL;
    if (!om_aligned16(dg) || !om_aligned16(du) || !om_aligned16(w_gate) || !om_aligned16(w_up) ||
        !om_aligned16(dx))
        return OM_ERR_ALIGN;
    p.A[0] = static_cast<const uint16_t *>(dg);
    p.A[1] = static_cast<const uint16_t *>(du);
    p.B[0] = static_cast<const uint16_t *>(w_gate);  // [G, I, H]: c = i, operand row = h
    p.B[1] = static_cast<const uint16_t *>(w_up);
    p.C = static_cast<uint16_t *>(dx);
    p.cum = cum_token_counts;
    p.lda = I; p.ldb = H; p.ldc = H;
    p.strideB = w_stride ? w_stride : static_cast<int64_t>(I) * H;
    if (!pitch_ok(p.strideB)) return OM_ERR_ALIGN;
    if (!fits_span(rows * H) || !fits_span(rows * I) || !fits_span(p.strideB * G)) return OM_ERR_SHAPE;
    p.rows = rows; p.n_experts = G; p.n_cols = H; p.kc = I; p.phases = 2;
    return OM_OK;
}
int gate_up_dgrad_launch(const void *dg, const void *du, const void *w_gate, const void *w_up, void *dx,
                         const int32_t *cum_token_counts, int64_t rows, int64_t expected_rows, int G, int I, int H,
                         int64_t w_stride, const om_dense_expert *dense, void *stream) {
    if (rows < 0 || expected_rows < 0 || expected_rows > rows || G < 1 || !mult(I, 8) || !mult(H, 8)) return OM_ERR_SHAPE;
    if (dense && (dense->rows < 1 || !fits_gather(dense->rows))) return OM_ERR_SHAPE;
    if (dense && (!dense->a[0] || !dense->a[1] || !dense->w[0] || !dense->w[1] || !dense->c[0] || !dense->cum)) return OM_ERR_NULL;
    auto dense_alone = [&]() {
        return gate_up_dgrad_launch(dense->a[0], dense->a[1], dense->w[0], dense->w[1], dense->c[0], dense->cum, dense->rows,
                                    dense->rows, 1, I, H, 0, nullptr, stream);
    };
    if (rows == 0) return dense ? dense_alone() : OM_OK;
    GemmParams p = {};
    const int params = gate_up_dgrad_params(dg, du, w_gate, w_up, dx, cum_token_counts, rows, G, I, H, w_stride, p);
    if (params != OM_OK) return params;
    if (dense) {
        if (dense_rides<EPI_STORE>(p, expected_rows, dense->rows)) {
            if (!dense_operands(p, dense)) return OM_ERR_ALIGN;
            return launch_rows_dense<CONTIG, STRIDED, EPI_STORE, GATHER_NONE, false>(p, rows, om_stream(stream));
        }
        const int code = dense_alone();
        if (code != OM_OK) return code;
    }
    return launch_rows_auto<CONTIG, STRIDED, EPI_STORE>(p, rows, expected_rows, om_stream(stream));
}
}  // namespace

extern "C" int om_merged_mlp_gate_up_dgrad_bound(const void *dg, const void *du, const void *w_gate,
                                                 const void *w_up, void *dx, const int32_t *cum_token_counts,
                                                 int64_t rows, int64_t expected_rows, int G, int I, int H,
                                                 int64_t w_stride, void *stream) {
    return gate_up_dgrad_launch(dg, du, w_gate, w_up, dx, cum_token_counts, rows, expected_rows, G, I, H, w_stride, nullptr, stream);
}

// Where the tiles of both are 128x128 and no more than 8 rounds of two blocks a CU: the last round of either launch is then a good part of it, and
// with few tiles either leaves most of the chip idle.  Two launches -> one, us, caches full of written data, gradients written / added: 8
// experts of 256/512, 4096 rows (0.5 rounds in all) 34.4 -> 26.2 / 36.2 -> 27.5; 16 of 512/256, 1200 rows 24.2 -> 17.4 / 28.2 -> 19.4; 12 of 1000/712,
// 9003 rows (4.6) 130 -> 122 / 140 -> 133, uneven 157 -> 142 / 164 -> 151, 900 rows 56.5 -> 53.3 / 66.9 -> 60.4; 16 of 1304/600, 4096 rows (6.0) 97 ->
// 92 / 114 -> 110; 8 of 2000/1000, 8000 rows (8.1) 259 -> 259 / 282 -> 283; 32 of 1000/1000, 32000 rows (16) 533 -> 534 / 557 -> 555.
extern "C" int om_merged_mlp_backward_joins(int64_t expected_rows, int G, int I, int H) {
    if (expected_rows < 0 || G < 1 || !mult(I, 8) || !mult(H, 8)) return OM_ERR_SHAPE;
    GemmParams p = {};
    p.n_experts = G; p.n_cols = H; p.kc = I;
    if (expected_rows < 1 || G > MAX_EXPERTS || rows_share(p, expected_rows) || uses_big_tile<EPI_STORE>(H, I, G, expected_rows) ||
        2 * static_cast<int64_t>(G) * I * H >= CACHED_WEIGHTS || wgrad_big_tile(H, I, 3 * static_cast<int64_t>(G)))
        return 0;
    const int64_t across = (H + 127) / 128, weight_tiles = 3 * across * ((I + 127) / 128) * G, row_tiles = (expected_rows / 128 + (G + 1) / 2) * across;
    return weight_tiles + row_tiles <= 8 * 2 * static_cast<int64_t>(device_cu_count()) ? 1 : 0;
}

namespace {
int backward_launch(const void *dout, const int32_t *dout_rows, const void *h, const void *dg, const void *du,
                    const void *x, const int32_t *x_rows, int64_t src_rows, const void *w_gate,
                    const void *w_up, void *dx, void *dw_down, void *dw_gate, void *dw_up,
                    const int32_t *cum_token_counts, int64_t rows, int64_t expected_rows, int G, int I,
                    int H, int64_t w_stride, int64_t down_stride, int64_t gate_stride, int64_t up_stride,
                    bool accumulate, void *stream) {
    if (rows < 1 || expected_rows < 0 || expected_rows > rows || G < 1 || !mult(I, 8) || !mult(H, 8)) return OM_ERR_SHAPE;
    GemmParams p = {};
    int code = gate_up_dgrad_params(dg, du, w_gate, w_up, dx, cum_token_counts, rows, G, I, H, w_stride, p);
    if (code != OM_OK) return code;
    bool joined = false;
    const bool may = om_merged_mlp_backward_joins(expected_rows, G, I, H) == 1;
    code = wgrad_merged_launch(dout, dout_rows, h, dg, du, x, x_rows, src_rows, dw_down, dw_gate, dw_up, cum_token_counts, rows,
                               expected_rows, G, I, H, down_stride, gate_stride, up_stride, accumulate, stream, may ? &p : nullptr, &joined);
    if (code != OM_OK || joined) return code;
    return launch_rows_auto<CONTIG, STRIDED, EPI_STORE>(p, rows, expected_rows, om_stream(stream));
}
}  // namespace

extern "C" int om_grouped_gemm_wgrad_merged_dgrad(const void *dout, const int32_t *dout_rows, const void *h, const void *dg, const void *du, const void *x, const int32_t *x_rows,
    int64_t src_rows, const void *w_gate, const void *w_up, void *dx, void *dw_down, void *dw_gate, void *dw_up,
    const int32_t *cum_token_counts, int64_t rows, int64_t expected_rows, int G, int I, int H, int64_t w_stride, int64_t down_stride,
    int64_t gate_stride, int64_t up_stride, void *stream) {
    return backward_launch(dout, dout_rows, h, dg, du, x, x_rows, src_rows, w_gate, w_up, dx, dw_down, dw_gate, dw_up, cum_token_counts, rows,
                           expected_rows, G, I, H, w_stride, down_stride, gate_stride, up_stride, false, stream);
}

extern "C" int om_grouped_gemm_wgrad_merged_dgrad_accumulate(const void *dout, const int32_t *dout_rows, const void *h, const void *dg, const void *du, const void *x, const int32_t *x_rows,
    int64_t src_rows, const void *w_gate, const void *w_up, void *dx, void *dw_down, void *dw_gate, void *dw_up,
    const int32_t *cum_token_counts, int64_t rows, int64_t expected_rows, int G, int I, int H, int64_t w_stride, int64_t down_stride,
    int64_t gate_stride, int64_t up_stride, void *stream) {
    return backward_launch(dout, dout_rows, h, dg, du, x, x_rows, src_rows, w_gate, w_up, dx, dw_down, dw_gate, dw_up, cum_token_counts, rows,
                           expected_rows, G, I, H, w_stride, down_stride, gate_stride, up_stride, true, stream);
}

extern "C" int om_merged_mlp_gate_up_dgrad_dense(const void *dg, const void *du, const void *w_gate,
                                                 const void *w_up, void *dx, const int32_t *cum_token_counts,
                                                 int64_t rows, int64_t expected_rows, int G, int I, int H,
                                                 int64_t w_stride, const om_dense_expert *dense, void *stream) {
    if (!dense) return OM_ERR_NULL;
    return gate_up_dgrad_launch(dg, du, w_gate, w_up, dx, cum_token_counts, rows, expected_rows, G, I, H, w_stride, dense, stream);
}

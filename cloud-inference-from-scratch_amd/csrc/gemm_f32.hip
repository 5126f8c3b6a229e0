// True float32 matrix product for the 32-bit path: C = A * W^T (+ bias), or the gated unit of its two halves.
//   A [M, K] row-major (row stride lda), W [N, K] row-major (a Linear's weight), C [M, N] (row stride ldc);
//   with the gate: C [M, N / 2] = silu(first half of the columns) * (second half).
// Float32 matrix instructions (v_mfma_f32_16x16x4_f32: float32 products and sums, no reduced-precision mode).
//
// Every output element is the same sum in the same order in every form below, so a row's result does not depend on
// how many other rows are in the batch: K in blocks of 256, the sum of two chains of 128 in which
// k ascends (an instruction takes four neighbouring k); the sums of four blocks are added one after the other, and so are the sums of these stretches of 1,024 k
// (the rounding error grows with 128 + 1 + 4 + K/1024 terms, not with K).
//
// Two forms:
//
// * gemm_f32_rows_kernel, few rows: bound by the stream of W and, in a decode layer, by its launches (some 4.8 us each before
//   one streams anything).  It can take its neighbours' work with it, all of it in the bits that their own kernels give: the
//   RMS norm in front of it (every workgroup sums the few rows' squares while its first pieces of W are on their way), the add
//   into the stream behind it, the rotation and the cache write of q/k/v.  A decode layer has six kernels so, not nine.  A workgroup owns 8 to 32 columns and 8 to 32 rows and
//   goes on to the next columns until none are left; its waves take the blocks of K in turn, each wave fetching W and
//   A as 128-byte row segments (8 lanes to a segment: a load in which every lane reads another row keeps the address
//   unit busy four times as long), four 32-wide pieces ahead in registers and across the end of a tile, and turning
//   them into operand order in 2 KB of LDS per 16 rows of its own.  The blocks' sums meet in LDS and are added in
//   order.
// * gemm_f32_tile_kernel, more rows: bound by the matrix cores (256 flops a cycle and unit; 157 TFLOP/s).  Four waves
//   share a tile of 64 x 64 through two stages of LDS in 32-wide slices, the four following slices on their way in
//   registers (one slice ahead a tile alone on its unit took twice as long: 89 -> 45 us at 256 rows, N = K = 2,048).
//   Where the tiles leave units idle a workgroup takes one stretch of K and leaves its sum in a workspace, and
//   gemm_f32_join_kernel adds the stretches in order.
//   gemm_f32_direct_kernel: the same tiles, loaded straight into LDS, where a unit takes five and more (goes_direct); the
//   matrix cores are busy 77 % of its time, with zeros for numbers too, so it is not the power.
//
// Measured (MI355X, us): 4 rows: N 22,016, K 2,048 42 (4.3 TB/s), N 2,048, K 11,008 27 (3.4 TB/s), N = K = 2,048 10;
// 517 rows: 460 (101 TFLOP/s), 256 with K in stretches (91 TFLOP/s; 359 without), 68; 2,048 rows: 1,555 (119 TFLOP/s),
// 753, 150.  Plain fused multiply-adds in tiles of 64 x 64, whatever the rows, took 370 for the median product of a step
// of 4 rows and 833 of one of 517 (23 TFLOP/s).
#include "common.h"

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_pointer;

constexpr int kBlockK = 256;   // a block of K: its sum joins the total
constexpr int kPiece = 32;     // k of a piece: 128 bytes of a row
constexpr int kPiecesPerBlock = kBlockK / kPiece;
constexpr int kPiecesPerChain = kPiecesPerBlock / 2;
constexpr int kBlocksPerStretch = 4;
constexpr int kStretch = kBlockK * kBlocksPerStretch;
constexpr int kTileFloats = 16 * kPiece;  // 16 rows of a piece

// 16-byte chunk `c` (0..7) of row `row` in a tile whose rows are 128 bytes: the chunks of 16 rows that a quarter wave
// reads at one time lie in different banks.
__device__ __forceinline__ int chunk_at(int row, int c) { return row * kPiece + 4 * (c ^ ((row >> 1) & 7)); }

// The numbers k = 16 g + 4 t + q of a row for t = 0..3, where q is the lane's quarter: what four instructions in turn take
// of 16 k.  (Four 4-byte reads; one 16-byte read and a transposition over the quarters with row swaps made the products
// of many rows 20 % slower, and one 16-byte read with the k in another order 2 % faster.)
__device__ __forceinline__ floatx4 operand(const float* tile, int row, int g, int q) {
    floatx4 v;
#pragma unroll
    for (int t = 0; t < 4; ++t) v[t] = tile[chunk_at(row, 4 * g + t) + q];
    return v;
}

// Four values of a row from k on; what lies past K is 0 (`inside`).  kVec: K and the row's start are multiples of
// four numbers.  The load stands under no condition (a piece past the end reads the row's start again), so that the
// compiler can count the loads that are under way.
template <bool kVec>
__device__ __forceinline__ floatx4 load4(const float* __restrict__ row, int k, int K) {
    if constexpr (kVec) {
        return *reinterpret_cast<const floatx4*>(row + (k < K ? k : 0));
    } else {
        floatx4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = row[k + j < K ? k + j : 0];
        return v;
    }
}

template <bool kVec>
__device__ __forceinline__ floatx4 inside(floatx4 v, int k, int K) {
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = (kVec ? k : k + j) < K ? v[j] : 0.f;
    return v;
}

__device__ __forceinline__ float gated(float g, float u) { return (g / (1.0f + expf(-g))) * u; }

// What the rows kernel does beside the product: nothing; the norm of its rows; that, the rotation and the cache write; the add
// into C; nothing, into a C whose address lies on the device (a captured launch writes where its replay says).
enum { kPlain = 0, kNormed = 1, kRotated = 2, kAdded = 3, kPointed = 4 };
constexpr bool norms_rows(int beside) { return beside == kNormed || beside == kRotated; }

struct RowsBeside {
    const float* norm_weight;  // kNormed, kRotated: A is the stream, its rows' norm is multiplied
    float eps;
    // kRotated: W stacks the rows of q, k and v heads; queries go to C, keys and values to the cache
    const float *cos_table, *sin_table;  // [positions, rotary_dim / 2]
    const int *positions, *seq_of_token, *seq_slot, *block_table;
    int table_width;
    float *k_pool, *v_pool;    // [pages, Hkv, page_size, D], [pages, Hkv, D, page_size]
    int q_heads, kv_heads, head_dim, rotary_dim, page_size, rotate, write_kv;
    float* const* c_at;  // kPointed
};

// Where pair i (0..7) of group j (0..head_dim / 16 - 1) of a head lies: its first dimension, and how far on its partner is.  The
// first rotary_dim / 16 groups are dimensions of the rotated part's first half, the others of what does not rotate.
struct HeadPair {
    int first, apart;
    bool rotates;
};
__device__ __forceinline__ HeadPair head_pair(const RowsBeside& b, int j, int i) {
    const int turning = b.rotary_dim / 16;
    if (j < turning) return {j * 8 + i, b.rotary_dim / 2, b.rotate != 0};
    return {b.rotary_dim + (j - turning) * 8 + i, (b.head_dim - b.rotary_dim) / 2, false};
}

constexpr int kSegment = 8 * kWave;      // of a row: what a wave of the norm's own kernel sums
constexpr int kNormSegments = 16;        // rows of up to this many segments ...
constexpr int kNormTasks = 32;           // ... and so many segments in all: what 64 KB of LDS hold

// kRows rows (8, 16 or 32) by kColumns columns (8, 16 or 32; with the gate kColumns / 2 of each half), in tiles of 16
// of which the last may be half empty.  kWaves waves share K.  Workgroup x takes the columns' tiles x, x + gridDim.x, ...
// kHalves: 2, or 1 for a K of up to one chain's, which has no second chain (K 64 at 8 rows 4.2 -> 3.4 us).  Both this and kAdded are
// known when the kernel is compiled: as numbers of the launch they cost every product 0.3 to 2 us (4 rows, 2,048 columns, K
// 11,008 28.0 -> 25.8; 16 rows, 896 columns, K 4,864 19.4 -> 18.9), the loop over the chains no longer
// being unrolled and the waits in it being for what the add might have asked for.
template <int kRows, int kColumns, int kWaves, bool kGate, bool kVec, int kBeside, int kHalves>
__global__ void __launch_bounds__(kWaves * kWave)
gemm_f32_rows_kernel(const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                     float* __restrict__ C, int M, int N, int K, int lda, int ldc, RowsBeside beside) {
    constexpr int kRowTiles = (kRows + 15) / 16, kColumnTiles = (kColumns + 15) / 16;
    constexpr bool kOwnRows = norms_rows(kBeside);  // the normed rows lie in LDS, whole
    constexpr int kTiles = kRowTiles + kColumnTiles, kStaged = kOwnRows ? kColumnTiles : kTiles;
    constexpr int kSums = kRowTiles * kColumnTiles * 256;
    constexpr int kAhead = kPiecesPerChain;  // pieces on their way
    constexpr int kThreads = kWaves * kWave;
    constexpr int kOwned = (kSums + kThreads - 1) / kThreads;
    constexpr int kStep = kGate ? kColumns / 2 : kColumns;  // output columns of a tile
    static_assert(!kGate || kColumns == 32 || kColumns == 16, "a gate's tile holds as many columns of either half");
    static_assert(!kOwnRows || (kVec && kRows == 8), "a few rows in 16-byte pieces");
    static_assert(kBeside != kRotated || (!kGate && kColumns == 16 && kRows * 8 <= kThreads), "8 dimensions and their partners");
    __shared__ float stage_all[kWaves * kStaged * kTileFloats];
    __shared__ float sums[2][kWaves * kSums];
    if constexpr (kBeside == kPointed) C = *beside.c_at;
    const int lane = threadIdx.x % kWave;
    const int wave = threadIdx.x / kWave;
    float* stage = stage_all + wave * kStaged * kTileFloats;
    const int m0 = blockIdx.y * kRows;
    const int width = kGate ? N / 2 : N;  // output columns
    const int column_tiles = (width + kStep - 1) / kStep;
    const int blocks = (K + kBlockK - 1) / kBlockK;
    const int rounds = (blocks + kWaves - 1) / kWaves;

    // kRotated: tile t takes the eight pairs of group j of head h, t = h * D / 16 + j
    const int per_head = kBeside == kRotated ? beside.head_dim / 16 : 1;
    // row r (0..kColumns - 1) of a tile of W
    auto weight_row = [&](int tile, int r) {
        if constexpr (kBeside == kRotated) {
            const int head = tile / per_head;
            const HeadPair pair = head_pair(beside, tile - head * per_head, r % 8);
            return W + static_cast<size_t>(head * beside.head_dim + pair.first + r / 8 * pair.apart) * K;
        }
        const int n = kGate ? min(tile * kStep + r % kStep, width - 1) + (r / kStep) * width : min(tile * kStep + r, N - 1);
        return W + static_cast<size_t>(n) * K;
    };
    constexpr int kWLoads = kColumns / 8, kALoads = kRows / 8;
    const int chunk = lane % 8;
    const float* a_row[kALoads];
#pragma unroll
    for (int i = 0; i < kALoads; ++i) a_row[i] = A + static_cast<size_t>(min(m0 + 8 * i + lane / 8, M - 1)) * lda;

    constexpr int pieces = kHalves * kPiecesPerChain;
    // the piece that is fetched next: its place in the block, the round and the tile
    int f_piece = 0, f_round = 0, f_tile = blockIdx.x;
    const float* w_row[kWLoads];
#pragma unroll
    for (int i = 0; i < kWLoads; ++i) w_row[i] = weight_row(f_tile, 8 * i + lane / 8);
    floatx4 w_ahead[kAhead][kWLoads], a_ahead[kAhead][kALoads];
    auto fetch = [&](floatx4 (&w)[kWLoads], floatx4 (&a)[kALoads]) {
        const int k = (wave + f_round * kWaves) * kBlockK + f_piece * kPiece + 4 * chunk;
#pragma unroll
        for (int i = 0; i < kWLoads; ++i) w[i] = load4<kVec>(w_row[i], k, K);
        if constexpr (!kOwnRows)
#pragma unroll
            for (int i = 0; i < kALoads; ++i) a[i] = load4<kVec>(a_row[i], k, K);
        if (++f_piece == pieces) {
            f_piece = 0;
            if (++f_round == rounds) {
                f_round = 0;
                f_tile = min(f_tile + static_cast<int>(gridDim.x), column_tiles - 1);
#pragma unroll
                for (int i = 0; i < kWLoads; ++i) w_row[i] = weight_row(f_tile, 8 * i + lane / 8);
            }
        }
    };
    // where the token of this thread's result (row threadIdx.x / 8, pair threadIdx.x % 8 of a tile) sits: three loads, each of
    // which needs the one before, between what else is on its way
    const int place_row = min(m0 + static_cast<int>(threadIdx.x) / 8 % kRows, M - 1);
    int pos = 0, page = -1;
    if constexpr (kBeside == kRotated) {
        pos = beside.positions[place_row];
        if (beside.write_kv) page = beside.seq_of_token[place_row];
    }
    // The norm's rows: asked for in front of the first pieces of W (behind them they would wait for all of these), summed
    // segment by segment as the norm's kernel sums them, and left in LDS, where the product takes its operand from: rows
    // `apart` numbers apart, zeros behind K up to the last block's end.
    __shared__ __attribute__((aligned(16))) float own_rows[kOwnRows ? kNormTasks * kSegment + 4 * kRows : 1];
    const int apart = blocks * kBlockK + 4;
    constexpr int kTogether = kNormTasks / kWaves;
    const int segments = (K + kSegment - 1) / kSegment, tasks = min(kRows, M - m0) * segments;
    eight_t own[kTogether] = {}, gain[kTogether] = {};
    if constexpr (kOwnRows) {
        const int first = __builtin_amdgcn_readfirstlane(wave);
#pragma unroll
        for (int i = 0; i < kTogether; ++i) {
            if (first + i * kWaves >= tasks) break;
            const int task = first + i * kWaves, row = task / segments;
            const int h = min((task - row * segments) * kSegment + lane * 8, K - 8);
            own[i] = load_eight(A + static_cast<size_t>(m0 + row) * lda + h);
            gain[i] = load_eight(beside.norm_weight + h);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int s = 0; s < kAhead; ++s) fetch(w_ahead[s], a_ahead[s]);
    if constexpr (kOwnRows) {
        __builtin_amdgcn_sched_barrier(0);
        if (kBeside == kRotated && beside.write_kv) page = beside.seq_slot[page];
        __shared__ float segment_sums[kNormTasks];
        const int first = __builtin_amdgcn_readfirstlane(wave);
#pragma unroll
        for (int i = 0; i < kTogether; ++i) {
            const int task = first + i * kWaves, row = task / segments, h = (task - row * segments) * kSegment + lane * 8;
            if (task >= tasks) break;
            const float sum = wave_sum(h < K ? 0.f + sum_of_squares(own[i]) : 0.f);
            if (lane == 0) segment_sums[task] = sum;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kTogether; ++i) {
            const int task = first + i * kWaves, row = task / segments, h = (task - row * segments) * kSegment + lane * 8;
            if (task >= tasks) break;
            float sum = 0.f;
            for (int s = 0; s < segments; ++s) sum += segment_sums[row * segments + s];
            const float inverse = 1.0f / sqrtf(sum / static_cast<float>(K) + beside.eps);
            if (h < blocks * kBlockK) store_eight(own_rows + row * apart + h, h < K ? (own[i] * inverse) * gain[i] : eight_t{});
        }
        if (kBeside == kRotated && beside.write_kv)
            page = beside.block_table[static_cast<size_t>(page) * beside.table_width + pos / beside.page_size];
        __syncthreads();
    }
    const float* own_row[kRowTiles];  // this lane's rows of A (one past the last reads that one again, and is not stored)
#pragma unroll
    for (int rt = 0; rt < kRowTiles; ++rt) own_row[rt] = own_rows + min(16 * rt + lane % 16, min(kRows, M - m0) - 1) * apart;

    int turn = 0;  // two sets of sums take turns: the next block's are written while others still read this one's
    for (int tile = blockIdx.x; tile < column_tiles; tile += gridDim.x) {
        float total[kOwned] = {}, stretch[kOwned] = {};
        // a thread's sum e: tile e / 256 (column tiles outer), column 4 * (place / 16) + e % 4, row place % 16
        auto column_of = [&](int e) { return 16 * (e / 256 / kRowTiles) + 4 * ((e / 4) % kWave / 16) + e % 4; };
        auto row_of = [&](int e) { return 16 * (e / 256 % kRowTiles) + (e / 4) % kWave % 16; };
        float old[kOwned] = {};  // (of a C that is added to: on its way while W streams)
        if constexpr (kBeside == kAdded)
#pragma unroll
            for (int o = 0; o < kOwned; ++o) {
                const int e = min(static_cast<int>(threadIdx.x) + o * kThreads, kSums - 1);
                old[o] = C[static_cast<size_t>(min(m0 + row_of(e), M - 1)) * ldc + min(tile * kStep + column_of(e), N - 1)];
            }
        float c = 1.f, s = 0.f;  // this thread's angle
        if constexpr (kBeside == kRotated) {
            const int head = tile / per_head;
            const HeadPair pair = head_pair(beside, tile - head * per_head, threadIdx.x % 8);
            if (pair.rotates && head < beside.q_heads + beside.kv_heads) {
                const size_t at = static_cast<size_t>(pos) * (beside.rotary_dim / 2) + pair.first;
                c = beside.cos_table[at];
                s = beside.sin_table[at];
            }
        }
        for (int round = 0; round < rounds; ++round) {
            floatx4 block[kColumnTiles][kRowTiles] = {};
            for (int half = 0; half < kHalves; ++half) {
                floatx4 acc[kColumnTiles][kRowTiles] = {};
#pragma unroll
                for (int s = 0; s < kAhead; ++s) {
                    const int k = (wave + round * kWaves) * kBlockK + (half * kAhead + s) * kPiece + 4 * chunk;
                    __builtin_amdgcn_wave_barrier();
#pragma unroll
                    for (int i = 0; i < kWLoads; ++i)
                        *reinterpret_cast<floatx4*>(stage + chunk_at(8 * i + lane / 8, chunk)) = inside<kVec>(w_ahead[s][i], k, K);
                    if constexpr (!kOwnRows)
#pragma unroll
                        for (int i = 0; i < kALoads; ++i)
                            *reinterpret_cast<floatx4*>(stage + kColumnTiles * kTileFloats + chunk_at(8 * i + lane / 8, chunk)) =
                                inside<kVec>(a_ahead[s][i], k, K);
                    fetch(w_ahead[s], a_ahead[s]);
                    __builtin_amdgcn_wave_barrier();
#pragma unroll
                    for (int g = 0; g < kPiece / 16; ++g) {
                        floatx4 f[kTiles];
#pragma unroll
                        for (int t = 0; t < kStaged; ++t) {
                            // (a half empty tile reads its 8 rows twice; what comes of the copies is not stored)
                            const int r = (t < kColumnTiles ? kColumns : kRows) == 8 ? lane % 8 : lane % 16;
                            f[t] = operand(stage + t * kTileFloats, r, g, lane / 16);
                        }
                        if constexpr (kOwnRows)
#pragma unroll
                            for (int rt = 0; rt < kRowTiles; ++rt)
#pragma unroll
                                for (int t = 0; t < 4; ++t)  // (a block past the last reads that one, and is not summed)
                                    f[kColumnTiles + rt][t] = own_row[rt][min(wave + round * kWaves, blocks - 1) * kBlockK + (half * kAhead + s) * kPiece + 16 * g + 4 * t + lane / 16];
#pragma unroll
                        for (int j = 0; j < 4; ++j)
#pragma unroll
                            for (int ct = 0; ct < kColumnTiles; ++ct)
#pragma unroll
                                for (int rt = 0; rt < kRowTiles; ++rt)
                                    acc[ct][rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[ct][j], f[kColumnTiles + rt][j],
                                                                                       acc[ct][rt], 0, 0, 0);
                    }
                }
#pragma unroll
                for (int ct = 0; ct < kColumnTiles; ++ct)
#pragma unroll
                    for (int rt = 0; rt < kRowTiles; ++rt) block[ct][rt] += acc[ct][rt];
            }
            float* all = sums[turn];
            turn ^= 1;
#pragma unroll
            for (int ct = 0; ct < kColumnTiles; ++ct)
#pragma unroll
                for (int rt = 0; rt < kRowTiles; ++rt)
                    *reinterpret_cast<floatx4*>(all + wave * kSums + ((ct * kRowTiles + rt) * kWave + lane) * 4) = block[ct][rt];
            __syncthreads();
            const int here = min(kWaves, blocks - round * kWaves);
#pragma unroll
            for (int o = 0; o < kOwned; ++o) {
                const int e = threadIdx.x + o * kThreads;
                if (e < kSums)
                    for (int w = 0; w < here; ++w) {
                        stretch[o] += all[w * kSums + e];
                        const int block = round * kWaves + w;
                        if (block % kBlocksPerStretch == kBlocksPerStretch - 1 || block == blocks - 1) {
                            total[o] += stretch[o];
                            stretch[o] = 0.f;
                        }
                    }
            }
        }
        if constexpr (kGate || kBeside == kRotated) {
            // the two halves of a column belong to two threads (or to one thread's two sums): they meet in LDS
            float* all = sums[turn];
            turn ^= 1;
#pragma unroll
            for (int o = 0; o < kOwned; ++o) {
                const int e = threadIdx.x + o * kThreads;
                if (e < kSums) all[e] = total[o];
            }
            __syncthreads();
            auto sum_of = [&](int r, int column) {
                return all[(column / 16 * kRowTiles + r / 16) * 256 + ((column % 16) / 4 * 16 + r % 16) * 4 + column % 4];
            };
            if constexpr (kBeside == kRotated) {
                const int r = threadIdx.x / 8, i = threadIdx.x % 8, m = m0 + r;
                if (r < kRows && m < M) {
                    const int head = tile / per_head, D = beside.head_dim;
                    const HeadPair pair = head_pair(beside, tile - head * per_head, i);
                    const int d = pair.first, half = pair.apart, n = head * D + d;
                    const float x1 = sum_of(r, i) + (bias ? bias[n] : 0.f), x2 = sum_of(r, 8 + i) + (bias ? bias[n + half] : 0.f);
                    const bool turns = pair.rotates && head < beside.q_heads + beside.kv_heads;
                    const float y1 = turns ? __builtin_fmaf(x1, c, -(x2 * s)) : x1;  // (rounded as the rotation's kernel does)
                    const float y2 = turns ? __builtin_fmaf(x2, c, x1 * s) : x2;
                    if (head < beside.q_heads) {
                        C[static_cast<size_t>(m) * ldc + n] = y1;
                        C[static_cast<size_t>(m) * ldc + n + half] = y2;
                    } else if (page >= 0) {  // (no page: nothing is to be written)
                        const int in_page = pos % beside.page_size;
                        const size_t head_base = (static_cast<size_t>(page) * beside.kv_heads + (head - beside.q_heads) % beside.kv_heads) * beside.page_size * D;
                        if (head < beside.q_heads + beside.kv_heads) {
                            beside.k_pool[head_base + static_cast<size_t>(in_page) * D + d] = y1;
                            beside.k_pool[head_base + static_cast<size_t>(in_page) * D + d + half] = y2;
                        } else {  // element d of the token goes to [d, in_page]
                            beside.v_pool[head_base + static_cast<size_t>(d) * beside.page_size + in_page] = y1;
                            beside.v_pool[head_base + static_cast<size_t>(d + half) * beside.page_size + in_page] = y2;
                        }
                    }
                }
            } else {
                for (int at = threadIdx.x; at < kRows * kStep; at += kThreads) {
                    const int n = tile * kStep + at % kStep, m = m0 + at / kStep;
                    if (m < M && n < width)
                        C[static_cast<size_t>(m) * ldc + n] = gated(sum_of(at / kStep, at % kStep), sum_of(at / kStep, kStep + at % kStep));
                }
            }
        } else {
#pragma unroll
            for (int o = 0; o < kOwned; ++o) {
                const int e = threadIdx.x + o * kThreads;
                const int n = tile * kStep + column_of(e), m = m0 + row_of(e);
                if (e < kSums && column_of(e) < kColumns && row_of(e) < kRows && m < M && n < N) {
                    const float sum = total[o] + (bias ? bias[n] : 0.f);
                    C[static_cast<size_t>(m) * ldc + n] = kBeside == kAdded ? old[o] + sum : sum;
                }
            }
        }
    }
}

// kN x kM tiles of 16 per wave, two by two waves: 32 * kN columns (with the gate half of them of each half, one tile of
// either in turn), 32 * kM rows per workgroup; kAhead slices on their way.
template <int kN, int kM, int kAhead, bool kGate, bool kVec>
__global__ void __launch_bounds__(256, 2)
gemm_f32_tile_kernel(const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                     float* __restrict__ C, int M, int N, int K, int lda, int ldc, int row_blocks, int tiles,
                     float* __restrict__ parts) {
    constexpr int kRows = 32 * (kN + kM);  // of W, then of A, in a stage
    constexpr int kStep = kGate ? 16 * kN : 32 * kN;
    static_assert(kN % 2 == 0 && kAhead % 2 == 0 && kPiecesPerBlock % kAhead == 0, "");
    __shared__ float stage[2][kRows * kPiece];
    const int lane = threadIdx.x % kWave;
    const int wave = threadIdx.x / kWave;
    // workgroups come to the 8 XCDs in turn: each XCD takes a run of neighbouring tiles, row blocks first, so that
    // the tiles that read the same rows of W share an L2
    const int per = (tiles + 7) / 8;
    const int tile = (blockIdx.x % 8) * per + blockIdx.x / 8;
    if (blockIdx.x / 8 >= per || tile >= tiles) return;
    const int m0 = (tile % row_blocks) * 32 * kM;
    const int n0 = (tile / row_blocks) * kStep;
    const int width = kGate ? N / 2 : N;
    // with `parts` workgroup y takes stretch y of K and leaves its sum in parts[y] [M, N]
    const int k_first = parts ? blockIdx.y * kStretch : 0;
    const int k_end = parts ? min(K, k_first + kStretch) : K;

    const int chunk = threadIdx.x % 8;
    const float* row_of[kN + kM];
#pragma unroll
    for (int i = 0; i < kN + kM; ++i) {
        const int r = threadIdx.x / 8 + 32 * i;
        const int n = kGate ? min(n0 + r / 32 * 16 + r % 16, width - 1) + (r / 16 % 2) * width : min(n0 + r, N - 1);
        row_of[i] = i < kN ? W + static_cast<size_t>(n) * K : A + static_cast<size_t>(min(m0 + r - 32 * kN, M - 1)) * lda;
    }
    floatx4 ahead[kAhead][kN + kM];
    auto fetch = [&](floatx4 (&to)[kN + kM], int slice) {
#pragma unroll
        for (int i = 0; i < kN + kM; ++i) to[i] = load4<kVec>(row_of[i], k_first + slice * kPiece + 4 * chunk, k_end);
    };
    auto put = [&](const floatx4 (&from)[kN + kM], int slice, float* to) {
#pragma unroll
        for (int i = 0; i < kN + kM; ++i)
            *reinterpret_cast<floatx4*>(to + chunk_at(threadIdx.x / 8 + 32 * i, chunk)) =
                inside<kVec>(from[i], k_first + slice * kPiece + 4 * chunk, k_end);
    };

    auto join = [](floatx4 (&to)[kN][kM], floatx4 (&from)[kN][kM]) {
#pragma unroll
        for (int in = 0; in < kN; ++in)
#pragma unroll
            for (int im = 0; im < kM; ++im) {
                to[in][im] += from[in][im];
                from[in][im] = floatx4{0.f, 0.f, 0.f, 0.f};
            }
    };
    const int slices = (k_end - k_first + kPiece - 1) / kPiece;
    floatx4 acc[kN][kM] = {}, block[kN][kM] = {}, stretch[kN][kM] = {}, total[kN][kM] = {};
#pragma unroll
    for (int a = 0; a < kAhead; ++a) fetch(ahead[a], a);
    const int wn = (wave % 2) * 16 * kN, wm = 32 * kN + (wave / 2) * 16 * kM;  // this wave's rows in a stage
    for (int first = 0; first < slices; first += kAhead) {
#pragma unroll
        for (int a = 0; a < kAhead; ++a) {
            const int slice = first + a;
            float* here = stage[a % 2];
            // (this stage was read two slices ago, and all waves have passed the barrier since)
            put(ahead[a], slice, here);
            fetch(ahead[a], slice + kAhead);
            __syncthreads();
#pragma unroll
            for (int g = 0; g < kPiece / 16; ++g) {
                floatx4 w[kN], x[kM];
#pragma unroll
                for (int i = 0; i < kN; ++i)
                    w[i] = operand(here, wn + 16 * i + lane % 16, g, lane / 16);
#pragma unroll
                for (int i = 0; i < kM; ++i)
                    x[i] = operand(here, wm + 16 * i + lane % 16, g, lane / 16);
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int in = 0; in < kN; ++in)
#pragma unroll
                        for (int im = 0; im < kM; ++im)
                            acc[in][im] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[in][j], x[im][j], acc[in][im], 0, 0, 0);
            }
        }
        // (what stands behind the last slice adds zeros)
        const int past = first + kAhead;
        const bool end = past >= slices;
        if (end || past % kPiecesPerChain == 0) join(block, acc);
        if (end || past % kPiecesPerBlock == 0) join(stretch, block);
        if (end || past % (kPiecesPerBlock * kBlocksPerStretch) == 0) join(total, stretch);
    }
    if (parts) C = parts + static_cast<size_t>(blockIdx.y) * M * N;
    const bool wide = ldc % 4 == 0 && reinterpret_cast<uintptr_t>(C) % 16 == 0;
#pragma unroll
    for (int in = 0; in < kN; in += kGate ? 2 : 1) {
        const int n = n0 + (kGate ? wn / 2 + 8 * in : wn + 16 * in) + 4 * (lane / 16);
        floatx4 b = {0.f, 0.f, 0.f, 0.f};
        if (bias)
#pragma unroll
            for (int i = 0; i < 4; ++i) b[i] = bias[min(n + i, N - 1)];
#pragma unroll
        for (int im = 0; im < kM; ++im) {
            const int m = m0 + (wm - 32 * kN) + 16 * im + lane % 16;
            if (m >= M) continue;
            floatx4 v = total[in][im];
            if constexpr (kGate) {
                const floatx4 u = total[in + 1][im];
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = gated(v[i], u[i]);
            } else {
                v += b;
            }
            float* to = C + static_cast<size_t>(m) * ldc + n;
            if (wide && n + 3 < width) {
                *reinterpret_cast<floatx4*>(to) = v;
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (n + i < width) to[i] = v[i];
            }
        }
    }
}

// The tiles of gemm_f32_direct_kernel: those whose 64 rows are all there, and the last row block's where they are not.
struct DirectGrid {
    int whole_blocks, whole, ragged, whole_each, ragged_each;  // (..._each: of an XCD)
    __host__ __device__ DirectGrid(int M, int row_blocks, int tiles) {
        const bool ends_early = M % 64 != 0 && row_blocks > 1;
        const int columns = tiles / row_blocks;
        whole_blocks = row_blocks - (ends_early ? 1 : 0);
        whole = columns * whole_blocks;
        ragged = ends_early ? columns : 0;
        whole_each = (whole + 7) / 8;
        ragged_each = (ragged + 7) / 8;
    }
    __host__ __device__ int workgroups() const { return 8 * (whole_each + ragged_each); }
};

// Tiles of 64 x 64 by four waves, two by two, whose operands go straight into LDS: K a multiple of 32.  Four stages of 32 k
// (16 KB), so that three slices are under way and two workgroups share a unit; one barrier a slice, between its halves of 16
// k, as in gemm_direct.hip.  A wave whose rows lie partly past M leaves those products out.
template <bool kGate>
__global__ void __launch_bounds__(256, 2)
gemm_f32_direct_kernel(const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                       float* __restrict__ C, int M, int N, int K, int lda, int ldc, int row_blocks, int tiles,
                       float* __restrict__ parts) {
#if defined(__HIP_DEVICE_COMPILE__)  // (the host's pass has no type for a buffer's description)
    constexpr int kN = 2, kM = 2, kStages = 4, kWaves = 4;
    constexpr int kRows = 32 * (kN + kM), kStageFloats = kRows * kPiece;
    constexpr int kLoads = kRows / 8 / kWaves;      // of 8 rows, a wave and slice: half of them W's, half A's
    constexpr int kStep = kGate ? 16 * kN : 32 * kN;
    static_assert(kPiecesPerChain == kStages, "the loop takes a chain at a time");
    __shared__ __attribute__((aligned(1024))) float stages[kStages * kStageFloats];
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    // each XCD takes a run of neighbouring whole tiles, row blocks first, and behind them its share of those whose rows end
    // early (less work: what is left to do when the last turn is short)
    const DirectGrid grid(M, row_blocks, tiles);
    const int xcd = blockIdx.x % 8, local = blockIdx.x / 8;
    const bool ragged = local >= grid.whole_each;
    const int at = ragged ? xcd * grid.ragged_each + local - grid.whole_each : xcd * grid.whole_each + local;
    if (at >= (ragged ? grid.ragged : grid.whole)) return;
    const int m0 = (ragged ? row_blocks - 1 : at % grid.whole_blocks) * 32 * kM;
    const int n0 = (ragged ? at : at / grid.whole_blocks) * kStep;
    const int width = kGate ? N / 2 : N;
    const int k_first = parts ? blockIdx.y * kStretch : 0;
    const int slices = ((parts ? min(K, k_first + kStretch) : K) - k_first) / kPiece;

    unsigned from[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int r = (wave + kWaves * i) * 8 + lane / 8;
        const int chunk = (lane % 8) ^ ((r >> 1) & 7);
        const int n = kGate ? min(n0 + r / 32 * 16 + r % 16, width - 1) + (r / 16 % 2) * width : min(n0 + r, N - 1);
        const int m = min(m0 + r - 32 * kN, M - 1);
        from[i] = 4u * (r < 32 * kN ? static_cast<unsigned>(n) * K + k_first + 4 * chunk : static_cast<unsigned>(m) * lda + k_first + 4 * chunk);
    }
    const __amdgpu_buffer_rsrc_t of_w = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(W), 0, 0xffffffffu, 0x00027000);
    const __amdgpu_buffer_rsrc_t of_a = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(A), 0, 0xffffffffu, 0x00027000);
    auto fetch = [&](int slice, int stage) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(i < kLoads / 2 ? of_w : of_a,
                                                     (lds_pointer)(stages + stage * kStageFloats + (wave + kWaves * i) * 8 * kPiece), 16,
                                                     from[i], slice * kPiece * 4, 0, 0);
    };

    const int wn = (wave % 2) * 16 * kN, wm = 32 * kN + (wave / 2) * 16 * kM;  // this wave's rows in a stage
    const int row_tiles = max(0, min(kM, (M - m0 - (wm - 32 * kN) + 15) / 16));  // ... of which so many hold rows
    floatx4 acc[kN][kM] = {}, block[kN][kM] = {}, stretch[kN][kM] = {}, total[kN][kM] = {};
    auto join = [](floatx4 (&to)[kN][kM], floatx4 (&from)[kN][kM]) __attribute__((always_inline)) {
#pragma unroll
        for (int in = 0; in < kN; ++in)
#pragma unroll
            for (int im = 0; im < kM; ++im) {
                to[in][im] += from[in][im];
                from[in][im] = floatx4{0.f, 0.f, 0.f, 0.f};
            }
    };
    struct Operands {
        floatx4 w[kN], x[kM];
    };
    auto read = [&](Operands& to, const float* at, int g) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kN; ++i) to.w[i] = operand(at, wn + 16 * i + lane % 16, g, lane / 16);
#pragma unroll
        for (int i = 0; i < kM; ++i) to.x[i] = operand(at, wm + 16 * i + lane % 16, g, lane / 16);
    };
    auto products = [&](const Operands& o, int im) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int in = 0; in < kN; ++in)
                acc[in][im] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.w[in][j], o.x[im][j], acc[in][im], 0, 0, 0);
    };
    auto multiply = [&](const Operands& o) __attribute__((always_inline)) {
        if (row_tiles == kM) {  // (the same for the wave)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int in = 0; in < kN; ++in)
#pragma unroll
                    for (int im = 0; im < kM; ++im)
                        acc[in][im] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.w[in][j], o.x[im][j], acc[in][im], 0, 0, 0);
        } else if (row_tiles == 1) {
            products(o, 0);
        }
    };
    // A product's sums are read (join) only when it has finished: the wait states between the two are written here, for
    // every way that leads from a product to a join.
    auto settle = [] __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    Operands even, odd;
    auto meet = [&](bool more) __attribute__((always_inline)) {
        if (more) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((kStages - 2) * kLoads) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        asm volatile("s_barrier" ::: "memory");
    };
#pragma unroll
    for (int s = 0; s < kStages; ++s)
        if (s < slices) fetch(s, s);
    if (slices >= kStages) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kStages - 1) * kLoads) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    asm volatile("s_barrier" ::: "memory");
    read(even, stages, 0);
    for (int first = 0; first < slices; first += kStages) {
#pragma unroll
        for (int j = 0; j < kStages; ++j) {
            const int slice = first + j;
            if (slice < slices) {  // (the same for all)
                read(odd, stages + j * kStageFloats, 1);
                __builtin_amdgcn_sched_barrier(0);
                multiply(even);
                __builtin_amdgcn_sched_barrier(0);
                meet(slice + kStages <= slices);  // the next slice is there, and nobody reads this one any more
                if (slice + kStages < slices) fetch(slice + kStages, j);
                read(even, stages + (j + 1) % kStages * kStageFloats, 0);  // (past the last slice: read and dropped)
                __builtin_amdgcn_sched_barrier(0);
                multiply(odd);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        const int past = first + kStages;
        const bool end = past >= slices;
        settle();
        join(block, acc);
        if (end || past % kPiecesPerBlock == 0) join(stretch, block);
        if (end || past % (kPiecesPerBlock * kBlocksPerStretch) == 0) join(total, stretch);
    }
    if (parts) C = parts + static_cast<size_t>(blockIdx.y) * M * N;
    const bool wide = ldc % 4 == 0 && reinterpret_cast<uintptr_t>(C) % 16 == 0;
#pragma unroll
    for (int in = 0; in < kN; in += kGate ? 2 : 1) {
        const int n = n0 + (kGate ? wn / 2 + 8 * in : wn + 16 * in) + 4 * (lane / 16);
        floatx4 b = {0.f, 0.f, 0.f, 0.f};
        if (bias)
#pragma unroll
            for (int i = 0; i < 4; ++i) b[i] = bias[min(n + i, N - 1)];
#pragma unroll
        for (int im = 0; im < kM; ++im) {
            const int m = m0 + (wm - 32 * kN) + 16 * im + lane % 16;
            if (m >= M) continue;
            floatx4 v = total[in][im];
            if constexpr (kGate) {
                const floatx4 u = total[in + 1][im];
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = gated(v[i], u[i]);
            } else {
                v += b;
            }
            float* to = C + static_cast<size_t>(m) * ldc + n;
            if (wide && n + 3 < width) {
                *reinterpret_cast<floatx4*>(to) = v;
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (n + i < width) to[i] = v[i];
            }
        }
    }
#endif
}

// C = the sums of `stretches` parts [M, N] in order (+ bias), or the gated unit of their halves; a thread an output number.
template <bool kGate>
__global__ void __launch_bounds__(256)
gemm_f32_join_kernel(const float* __restrict__ parts, int stretches, const float* __restrict__ bias, float* __restrict__ C,
                     int M, int N, int ldc) {
    const int width = kGate ? N / 2 : N;
    const int n = blockIdx.x * 256 + threadIdx.x, m = blockIdx.y;
    if (n >= width) return;
    const size_t apart = static_cast<size_t>(M) * N;
    const float* from = parts + static_cast<size_t>(m) * N + n;
    float total = 0.f, up = 0.f;
    for (int first = 0; first < stretches; first += 4) {
        float v[4], u[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {  // (a part past the last is read again and dropped)
            v[i] = from[min(first + i, stretches - 1) * apart];
            if constexpr (kGate) u[i] = from[min(first + i, stretches - 1) * apart + width];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (first + i >= stretches) break;
            total += v[i];
            if constexpr (kGate) up += u[i];
        }
    }
    C[static_cast<size_t>(m) * ldc + n] = kGate ? gated(total, up) : total + (bias ? bias[n] : 0.f);
}

struct Product {
    const float *A, *W, *bias;
    float *C, *parts;
    int M, N, K, lda, ldc, units;
    RowsBeside beside;
};

// Whether `workgroups` tiles load straight into LDS: whole slices of K, places in the operands in 32 bits of bytes, and so many
// tiles to a unit: five and more over all of K (N 22,016, K 2,048 with the gate, us, before and so: 100 rows, 2.7 to a unit,
// 129, 133; 256 rows, 5.4, 228, 229; 264 rows 269, 253; 448 rows 377, 361; 517 rows 486, 460; N 2,560,
// K 2,048: 800 rows, 4 to a unit, 106, 110), twelve in stretches (N 2,048, K 11,008: 288 rows, 6.9 to a unit, 147, 150; 384 rows,
// 8.3, 176, 182; 448 rows, 9.6, 196, 197; 517 rows, 12.4, 264, 256; 2,048 rows 821, 753).
constexpr long kDirectTiles = 5, kDirectStretches = 12;

bool goes_direct(const Product& p, long workgroups, long per_unit) {
    return workgroups >= per_unit * p.units && p.K % kPiece == 0 && static_cast<long>(p.N) * p.K < (1L << 30) &&
           static_cast<long>(p.M) * p.lda < (1L << 30);
}

template <int kRows, int kColumns, int kWaves, bool kGate, bool kVec, int kBeside = kPlain>
void run_rows(hipStream_t s, const Product& p) {
    static_assert(kBeside != kAdded || !kGate, "a product's own result is added");
    const int step = kGate ? kColumns / 2 : kColumns;
    const int tiles = ((kGate ? p.N / 2 : p.N) + step - 1) / step;
    // as many workgroups as the units hold at a time by their LDS (2 KB a wave for each staged tile and each tile of sums):
    // further ones would start cold behind them instead of fetching across the end of a tile (N 22,016, K 2,048 with the
    // gate at 32 rows 54.3 -> 49.3 us, N 3,584, K 18,944 at 16 rows 88 -> 83).  Not for 16 columns of up to 16 rows, three to
    // a unit, whose columns never exceed four a unit: all at once (N 14,000, K 2,048 at 4 rows 25.9; by their LDS 27.4)
    constexpr int kRowTiles = (kRows + 15) / 16, kColumnTiles = (kColumns + 15) / 16;
    constexpr int kLds = kWaves * 2048 * (kRowTiles + kColumnTiles + kRowTiles * kColumnTiles);
    const int most = p.units * (norms_rows(kBeside) ? 1 : kRows <= 16 && kColumns == 16 ? 32 / kWaves : 160 * 1024 / kLds);
    dim3 grid(tiles < most ? tiles : most, (p.M + kRows - 1) / kRows);
    if constexpr (kWaves == 4) {  // (a K that short has four waves, but for operands off 16 bytes)
        if (p.K <= kBlockK / 2) {
            gemm_f32_rows_kernel<kRows, kColumns, kWaves, kGate, kVec, kBeside, 1><<<grid, kWaves * kWave, 0, s>>>(p.A, p.W, p.bias, p.C, p.M, p.N, p.K, p.lda, p.ldc, p.beside);
            return;
        }
    }
    gemm_f32_rows_kernel<kRows, kColumns, kWaves, kGate, kVec, kBeside, 2><<<grid, kWaves * kWave, 0, s>>>(p.A, p.W, p.bias, p.C, p.M, p.N, p.K, p.lda, p.ldc, p.beside);
}

template <bool kGate, bool kVec>
void run_tiles(hipStream_t s, const Product& p) {
    const int step = kGate ? 32 : 64;
    const int row_blocks = (p.M + 63) / 64;
    const int tiles = row_blocks * (((kGate ? p.N / 2 : p.N) + step - 1) / step);
    if (kVec && goes_direct(p, tiles, kDirectTiles)) gemm_f32_direct_kernel<kGate><<<DirectGrid(p.M, row_blocks, tiles).workgroups(), 256, 0, s>>>(p.A, p.W, p.bias, p.C, p.M, p.N, p.K, p.lda, p.ldc, row_blocks, tiles, nullptr);
    else gemm_f32_tile_kernel<2, 2, kVec ? 4 : 2, kGate, kVec><<<(tiles + 7) / 8 * 8, 256, 0, s>>>(p.A, p.W, p.bias, p.C, p.M, p.N, p.K, p.lda, p.ldc, row_blocks, tiles, nullptr);
}

template <bool kVec>
void run_stretches(hipStream_t s, const Product& p, bool gate) {
    const int row_blocks = (p.M + 63) / 64;
    const int tiles = row_blocks * ((p.N + 63) / 64);
    const int stretches = (p.K + kStretch - 1) / kStretch;
    dim3 grid((tiles + 7) / 8 * 8, stretches);
    if (kVec && goes_direct(p, static_cast<long>(tiles) * stretches, kDirectStretches)) gemm_f32_direct_kernel<false><<<dim3(DirectGrid(p.M, row_blocks, tiles).workgroups(), stretches), 256, 0, s>>>(p.A, p.W, nullptr, nullptr, p.M, p.N, p.K, p.lda, p.N, row_blocks, tiles, p.parts);
    else gemm_f32_tile_kernel<2, 2, kVec ? 4 : 2, false, kVec><<<grid, 256, 0, s>>>(p.A, p.W, nullptr, nullptr, p.M, p.N, p.K, p.lda, p.N, row_blocks, tiles, p.parts);
    dim3 join(((gate ? p.N / 2 : p.N) + 255) / 256, p.M);
    if (gate) gemm_f32_join_kernel<true><<<join, 256, 0, s>>>(p.parts, stretches, nullptr, p.C, p.M, p.N, p.ldc);
    else gemm_f32_join_kernel<false><<<join, 256, 0, s>>>(p.parts, stretches, p.bias, p.C, p.M, p.N, p.ldc);
}

// (kAdded: up to 8 rows)
template <bool kGate, int kBeside = kPlain>
void run_few(hipStream_t s, const Product& p, bool vec) {
    if (!vec) return run_rows<16, 16, 8, kGate, false, kBeside>(s, p);
    // columns enough for two workgroups of 32 on every unit; a short K has blocks for four waves only
    const bool wide = p.N >= 64 * p.units, shallow = p.K <= 4 * kBlockK;
    // a long K and too few columns for a workgroup of 16 on every unit: 8 columns (a unit streams some 30 GB/s
    // however many loads it has under way: N 2,048, K 11,008 at 4 rows 32 -> 26 us; K 2,048 is as fast with 16)
    const bool narrow = !kGate && p.K > 8 * kBlockK && p.N < 16 * p.units;
    if constexpr (kBeside == kPlain) {
        if (p.M > 16) {
            if (shallow) wide ? run_rows<32, 32, 4, kGate, true>(s, p) : run_rows<32, 16, 4, kGate, true>(s, p);
            else wide ? run_rows<32, 32, 8, kGate, true>(s, p) : run_rows<32, 16, 8, kGate, true>(s, p);
            return;
        }
        if (p.M > 8) {
            if (wide) return shallow ? run_rows<16, 32, 4, kGate, true>(s, p) : run_rows<16, 32, 8, kGate, true>(s, p);
            if constexpr (!kGate)
                if (narrow) return run_rows<16, 8, 16, false, true>(s, p);
            return shallow ? run_rows<16, 16, 4, kGate, true>(s, p) : run_rows<16, 16, 8, kGate, true>(s, p);
        }
    }
    if (wide) return shallow ? run_rows<8, 32, 4, kGate, true, kBeside>(s, p) : run_rows<8, 32, 8, kGate, true, kBeside>(s, p);
    if constexpr (!kGate)
        if (narrow) return run_rows<8, 8, 16, false, true, kBeside>(s, p);
    shallow ? run_rows<8, 16, 4, kGate, true, kBeside>(s, p) : run_rows<8, 16, 8, kGate, true, kBeside>(s, p);
}

// The same choice for up to 8 rows with their norm beside the gated product, or beside that of q/k/v; no width takes 8 columns here.
void run_normed_gate(hipStream_t s, const Product& p) {
    const bool wide = p.N >= 64 * p.units, shallow = p.K <= 4 * kBlockK;
    if (wide) shallow ? run_rows<8, 32, 4, true, true, kNormed>(s, p) : run_rows<8, 32, 8, true, true, kNormed>(s, p);
    else shallow ? run_rows<8, 16, 4, true, true, kNormed>(s, p) : run_rows<8, 16, 8, true, true, kNormed>(s, p);
}
void run_normed_rope(hipStream_t s, const Product& p) {
    p.K <= 4 * kBlockK ? run_rows<8, 16, 4, false, true, kRotated>(s, p) : run_rows<8, 16, 8, false, true, kRotated>(s, p);
}

bool on_16_bytes(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

// Up to 8 rows of a float32 stream whose norm the product makes itself.
bool takes_norm(const float* stream, const float* W, const float* norm_weight, float eps, int M, int K) {
    return M >= 1 && M <= 8 && K >= 8 && K % 8 == 0 && K <= kNormSegments * kSegment &&
           M * ((K + kSegment - 1) / kSegment) <= kNormTasks && eps > 0.f && stream && W && norm_weight &&
           on_16_bytes(stream) && on_16_bytes(W) && on_16_bytes(norm_weight);
}

template <bool kGate>
void run_form(hipStream_t s, const Product& p, int form, bool vec) {
    if (form == 0) run_few<kGate>(s, p, vec);
    else if (form == 1) vec ? run_tiles<kGate, true>(s, p) : run_tiles<kGate, false>(s, p);
    else vec ? run_stretches<true>(s, p, kGate) : run_stretches<false>(s, p, kGate);
}

}  // namespace

// `form`: 0 = few rows, 1 = tiles, 2 = tiles with a stretch of K each, and with
// `parts` a workspace of ceil(K / 1024) * M * N numbers.  `gate`: the gated unit of the product's halves (N even, no
// bias).  `units`: compute units of the device.
CIE_API int cie_gemm_f32(void* stream, const float* A, const float* W, const float* bias, float* C, float* parts,
                         int M, int N, int K, int lda, int ldc, int gate, int form, int units) {
    if (M < 0 || N <= 0 || K <= 0 || lda < K || ldc < (gate ? N / 2 : N) || form < 0 || form > 2 || units < 1) return CIE_BAD_ARGUMENT;
    if ((gate && (N % 2 || bias)) || (form == 2 && !parts)) return CIE_BAD_ARGUMENT;
    if (M == 0) return CIE_OK;
    if (static_cast<long>((M + 63) / 64) * ((N + 31) / 32) > (1L << 30)) return CIE_BAD_ARGUMENT;
    if ((form == 0 && M > 8 * 65535) || (form == 2 && (M > 65535 || K > 65535 * kStretch))) return CIE_BAD_ARGUMENT;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool vec = K % 4 == 0 && lda % 4 == 0 && reinterpret_cast<uintptr_t>(A) % 16 == 0 && reinterpret_cast<uintptr_t>(W) % 16 == 0;
    const Product p{A, W, bias, C, parts, M, N, K, lda, ldc, units, {}};
    if (gate) run_form<true>(s, p, form, vec);
    else run_form<false>(s, p, form, vec);
    return cie_after_launch();
}

// Up to 8 rows: C [M, N] (rows ldc apart) += A W^T (+ bias), added to as the norm's kernel would add the product to its stream.
CIE_API int cie_gemm_f32_into(void* stream, const float* A, const float* W, const float* bias, float* C, int M, int N, int K,
                              int lda, int ldc, int units) {
    if (M < 0 || M > 8 || N <= 0 || K <= 0 || lda < K || ldc < N || units < 1) return CIE_BAD_ARGUMENT;
    if (M == 0) return CIE_OK;
    const bool vec = K % 4 == 0 && lda % 4 == 0 && on_16_bytes(A) && on_16_bytes(W);
    const Product p{A, W, bias, C, nullptr, M, N, K, lda, ldc, units, {}};
    run_few<false, kAdded>(static_cast<hipStream_t>(stream), p, vec);
    return cie_after_launch();
}

// Up to 8 rows: the contiguous [M, N] whose address is *c_at (on the device) = A W^T.
CIE_API int cie_gemm_f32_at(void* stream, const float* A, const float* W, float* const* c_at, int M, int N, int K, int lda, int units) {
    if (M < 0 || M > 8 || N <= 0 || K <= 0 || lda < K || units < 1 || !c_at) return CIE_BAD_ARGUMENT;
    if (M == 0) return CIE_OK;
    const bool vec = K % 4 == 0 && lda % 4 == 0 && on_16_bytes(A) && on_16_bytes(W);
    Product p{A, W, nullptr, nullptr, nullptr, M, N, K, lda, N, units, {}};
    p.beside.c_at = c_at;
    run_few<false, kPointed>(static_cast<hipStream_t>(stream), p, vec);
    return cie_after_launch();
}

// Up to 8 rows, and rows * ceil(K / 512) up to 32: C [M, N / 2] = the gated unit of norm(rows of the stream [M, K], contiguous) W^T.
// K a multiple of 8, up to 8,192; stream, W and the norm's weight at multiples of 16 bytes.
CIE_API int cie_gemm_f32_normed(void* stream, const float* rows, const float* norm_weight, float eps, const float* W, float* C, int M,
                                int N, int K, int ldc, int units) {
    if (!takes_norm(rows, W, norm_weight, eps, M, K) || N <= 0 || N % 2 || ldc < N / 2 || units < 1 || !C) return CIE_BAD_ARGUMENT;
    Product p{rows, W, nullptr, C, nullptr, M, N, K, K, ldc, units, {}};
    p.beside.norm_weight = norm_weight;
    p.beside.eps = eps;
    run_normed_gate(static_cast<hipStream_t>(stream), p);
    return cie_after_launch();
}

// The same for a q/k/v weight (heads of head_dim dimensions, of which the first rotary_dim rotate, multiples of 16): rotated queries go to C [M, N], rotated keys
// and values to the cache.
CIE_API int cie_gemm_f32_normed_rope(void* stream, const float* rows, const float* norm_weight, float eps, const float* W, const float* bias,
                                     float* C, int M, int N, int K, const float* cos_table, const float* sin_table,
                                     const int* positions, const int* seq_of_token, const int* seq_slot, const int* block_table,
                                     int table_width, float* k_pool, float* v_pool, int q_heads, int kv_heads, int head_dim,
                                     int rotary_dim, int page_size, int rotate, int write_kv, int units) {
    if (!takes_norm(rows, W, norm_weight, eps, M, K) || units < 1 || !C) return CIE_BAD_ARGUMENT;
    if (q_heads <= 0 || kv_heads <= 0 || head_dim <= 0 || head_dim % 16 || rotary_dim <= 0 || rotary_dim % 16 ||
        rotary_dim > head_dim || page_size <= 0 || table_width <= 0 ||
        N != (q_heads + 2 * kv_heads) * head_dim)
        return CIE_BAD_ARGUMENT;
    if (!positions || (rotate && (!cos_table || !sin_table)) ||
        (write_kv && (!seq_of_token || !seq_slot || !block_table || !k_pool || !v_pool)))
        return CIE_BAD_ARGUMENT;
    const Product p{rows, W, bias, C, nullptr, M, N, K, K, N, units,
                    {norm_weight, eps, cos_table, sin_table, positions, seq_of_token, seq_slot, block_table, table_width, k_pool,
                     v_pool, q_heads, kv_heads, head_dim, rotary_dim, page_size, rotate, write_kv, nullptr}};
    run_normed_rope(static_cast<hipStream_t>(stream), p);
    return cie_after_launch();
}

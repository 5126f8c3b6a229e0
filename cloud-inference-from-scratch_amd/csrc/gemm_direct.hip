// bfloat16 products of some dozens of rows and more on the matrix cores, operands loaded straight into LDS: C = A * W^T with
// A [M, K], W [N, K] bf16, K a multiple of 64, and float32 sums.  Epilogues: those of gemm_tiles.hip, which is left with the
// other K.
//
// Eight waves share a tile; a stage of LDS holds 64 k of the tile's rows of W and A, and as many stages as fit wait for their
// turn.  Every wave loads 1 KB of a stage (8 rows) at a time with the loads that write LDS themselves, so that nothing waits
// in registers: the tile may be 256 x 256, and the slices under way are as many as LDS holds.  One barrier a slice: it
// stands between the slice's halves of 32 k, when the second half's operands are in registers; behind it the next slice is
// in LDS and the stage that was just read takes the loads of the slice kStages ahead.  The reads of the next half and the
// loads stand between the products of this one, pinned there: left alone the compiler collects the reads behind the products.
//
// What bounds it (MI355X, 3B gate/up, 2,048 rows, 256 x 256, us): the products alone 107 (random numbers hold the matrix
// cores to 1.8 PFLOP/s by the power they draw), the loads alone 100 to 120 (the lines of W from memory, A from beyond an
// XCD's L2 every turn), the reads of LDS alone 24; together 147 to 170, and a start and an end of 8 a turn that nothing hides.
// Where the loads stand between the products, how far the reads run ahead and which waves load which operand changed nothing
// (within 3 %); touching the lines of W and A a slice or two early, by the workgroups of an XCD in shares, cost 2 to 10 %.
// At fewer rows it is the weight's way from memory, which each unit takes its own lines of at some 20 bytes a cycle, and the
// turns: parts/linear.py picks the tile whose turns come out best.
//
// A lane stores 16 bytes whose neighbours are its neighbours' (64 bytes a row and instruction): sums of K in parts, 3B down
// at 2,048 rows, 101 -> 92 us.  Where the result's rows lie no multiple of that apart, in pieces of 8 or 4 bytes (bf16, 777 rows, K
// 2,048, 4,098 columns, which are stored two at a time, 18.9 us; one at a time 24.8; 768 rows, K 768, 10,508 columns, four at a
// time, 18.0 and 32.5).  The q/k/v epilogue asks for its rows' places between the last slices: 256 rows 14.8 -> 14.1; at 256 x 256
// it spills 14 registers (60 bytes a lane), no other form any.
//
// The gate's quotient (gate_of) has the division's bits in fewer instructions than the compiler's division: a wave makes 64
// of them a lane, and the matrix cores wait.  3B gate/up 2,048 rows 161 -> 158 (three turns of it), 613 rows 66.1 -> 64.6, 256
// rows 33.1 -> 32.8.  (The reciprocal instruction's alone, 1 unit in the last place and 0 beyond 2^126: 154, 64.1, 32.6.)
//
// Measured (MI355X, us, weights from memory; before: the library with the kernel behind its product, or gemm_tiles.hip):
// 3B: gate/up 256 rows 40 -> 33, 613 rows 72 -> 61, 777 81 -> 72, 2,048 186 -> 157; down 256 rows 27 -> 23, 613 47 -> 36, 2,048
// 100 -> 91; 7B: gate/up 777 rows 272 -> 175, 2,048 541 -> 445; down 777 167 -> 98, 1,024 163 -> 119.  Whole prompts: 777 tokens
// of the 7B shape behind 4,000 (8 layers, 4 steps of decoding in it) 9.66 -> 8.33 ms, 2,048 of 3B (12 layers) 4.92 -> 4.65.
#include "common.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_pointer;

enum { DIRECT_BF16 = 0, DIRECT_SILU = 1, DIRECT_RESID = 2, DIRECT_PARTS = 3, DIRECT_ROPE = 4, DIRECT_ATOMIC = 5, DIRECT_SCALED = 6 };
constexpr bool gates(int epilogue) { return epilogue == DIRECT_SILU || epilogue == DIRECT_SCALED; }

constexpr int kSlice = 64;                   // k of a stage: 128 bytes of a row
constexpr int kLdsBytes = 160 * 1024;

// What the ROPE epilogue needs beside the product: where each row's token sits, and the cache.
struct DirectRope {
    const float *cos_table, *sin_table;  // [max_position, D/2]
    const int *positions, *seq_of_token; // [M]
    const int* seq_slot;                 // [sequences]
    const int* block_table;              // [slots, table_width]
    int table_width;
    bf16_t* k_pool;                      // [pages, Hkv, page_size, D]
    bf16_t* v_pool;                      // [pages, Hkv, D, page_size]
    int q_heads, kv_heads, head_dim, page_size, rotate, write_kv;
};

struct DirectArgs {
    const bf16_t *a, *w, *bias;
    void* c;            // BF16, SILU, SCALED: bf16 [M, ldc]; RESID, ATOMIC: the float32 stream; PARTS: float32 [parts, M, N]
    int M, N, K, lda, ldc;
    int k_per_part;     // a multiple of kSlice
    int row_blocks, tiles;
    DirectRope rope;    // ROPE only
    // SCALED only: partial sums of squares [M, sumsq_parts] of the rows of the stream whose 1/rms A lacks
    const float* row_sumsq;
    int sumsq_parts;
    float eps;
};

// 16-byte chunk `c` (0..7) of row `row` of a stage: the chunks of 16 rows that are read at one time lie in different banks
__device__ __forceinline__ int chunk_at(int row, int c) { return row * 128 + 16 * (c ^ ((row >> 1) & 7)); }

// Where, among its wave's output columns, row i of the wave's tile t of W lies: bf16 results in pairs of tiles, so that a
// lane ends with eight neighbouring columns and four lanes with 32.
template <int EPI, int kN>
__device__ __forceinline__ int column_of(int t, int i) {
    constexpr int kOut = gates(EPI) ? kN / 2 : kN;
    if (gates(EPI)) t /= 2;
    if ((EPI == DIRECT_BF16 || gates(EPI)) && kOut % 2 == 0) return t / 2 * 32 + i / 4 * 8 + t % 2 * 4 + i % 4;
    return 16 * t + i;
}

// Where the token of each of a lane's rows sits: three loads, each of which needs the one before.  They are asked for one at
// a time between the last slices, when no more loads of operands are counted.
template <int kM>
struct RowPlaces {
    int pos[kM], page[kM];
    int known = 0;

    __device__ __forceinline__ void step(const DirectArgs& p, int m_first, int lane) {
        const DirectRope& t = p.rope;
        if (known == 0) {
#pragma unroll
            for (int im = 0; im < kM; ++im) {
                const int m = min(m_first + 16 * im + lane % 16, p.M - 1);
                pos[im] = t.positions[m];
                page[im] = t.write_kv ? t.seq_of_token[m] : 0;
            }
        } else if (known == 1) {
#pragma unroll
            for (int im = 0; im < kM; ++im) page[im] = t.write_kv ? t.seq_slot[page[im]] : 0;
        } else if (known == 2) {
#pragma unroll
            for (int im = 0; im < kM; ++im)
                page[im] = t.write_kv ? t.block_table[static_cast<size_t>(page[im]) * t.table_width + pos[im] / t.page_size] : -1;
        }
        ++known;
    }
};

// The ROPE epilogue of a wave's tiles: pairs `pair`, `pair` + 1, ... of 16 dimensions and the 16 they rotate with.  Values
// are rounded to bf16 before the rotation, so that the results equal those of the plain epilogue followed by the rotation
// kernel.  The angles of all rows of a pair are asked for together.
template <int kN, int kM>
__device__ __forceinline__ void store_rope(const DirectArgs& p, const floatx4 (&acc)[kN][kM], const RowPlaces<kM>& at, int pair, int m_first, int lane) {
    const DirectRope& t = p.rope;
    const int D = t.head_dim, half = D / 2, per_head = D / 32;
#pragma unroll
    for (int in = 0; in < kN; in += 2, ++pair) {
        if (pair >= p.N / 32) return;
        const int head = pair / per_head;
        const int d = pair % per_head * 16 + 4 * (lane / 16);
        const bool is_query = head < t.q_heads, is_value = head >= t.q_heads + t.kv_heads;
        const int kv_head = is_value ? head - t.q_heads - t.kv_heads : head - t.q_heads;
        float bias_lo[4] = {}, bias_hi[4] = {};
        if (p.bias)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                bias_lo[i] = to_float(p.bias[head * D + d + i]);
                bias_hi[i] = to_float(p.bias[head * D + half + d + i]);
            }
        floatx4 c[kM], s[kM];
        if (t.rotate && !is_value) {
#pragma unroll
            for (int im = 0; im < kM; ++im) {
                c[im] = *reinterpret_cast<const floatx4*>(t.cos_table + static_cast<size_t>(at.pos[im]) * half + d);
                s[im] = *reinterpret_cast<const floatx4*>(t.sin_table + static_cast<size_t>(at.pos[im]) * half + d);
            }
        }
#pragma unroll
        for (int im = 0; im < kM; ++im) {
            const int m = m_first + 16 * im + lane % 16;
            if (m >= p.M || (!is_query && at.page[im] < 0)) continue;
            float lo[4], hi[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                lo[i] = to_float(from_float<bf16_t>(acc[in][im][i] + bias_lo[i]));
                hi[i] = to_float(from_float<bf16_t>(acc[in + 1][im][i] + bias_hi[i]));
            }
            const int in_page = at.pos[im] % t.page_size;
            if (is_value) {
                bf16_t* to = t.v_pool + ((static_cast<size_t>(at.page[im]) * t.kv_heads + kv_head) * D + d) * t.page_size + in_page;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    to[static_cast<size_t>(i) * t.page_size] = from_float<bf16_t>(lo[i]);
                    to[static_cast<size_t>(half + i) * t.page_size] = from_float<bf16_t>(hi[i]);
                }
                continue;
            }
            if (t.rotate) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float x1 = lo[i], x2 = hi[i];
                    lo[i] = __builtin_fmaf(x1, c[im][i], -(x2 * s[im][i]));  // (rounded as the rotation's kernel does)
                    hi[i] = __builtin_fmaf(x2, c[im][i], x1 * s[im][i]);
                }
            }
            bf16_t* to = is_query ? static_cast<bf16_t*>(p.c) + static_cast<size_t>(m) * p.ldc + head * D + d
                                  : t.k_pool + ((static_cast<size_t>(at.page[im]) * t.kv_heads + kv_head) * t.page_size + in_page) * D + d;
            *reinterpret_cast<uint2*>(to) = uint2{pack_bf16(lo[0], lo[1]), pack_bf16(lo[2], lo[3])};
            *reinterpret_cast<uint2*>(to + half) = uint2{pack_bf16(hi[0], hi[1]), pack_bf16(hi[2], hi[3])};
        }
    }
}

// x / (1 + e^-x), rounded as the division rounds it.  The reciprocal instruction's quotient is within a unit in the last place, and
// adding what its remainder still gives rounds it right (Markstein, IBM J. Res. Dev. 34, 1990); the instruction's result is 0
// where it lies below the normal numbers, so it is asked for a quarter of the denominator and scaled behind it; the last step
// puts infinities, zeros and NaN right.  Equal to the division for each of the 2^32 floats, which were all compared.
__device__ __forceinline__ float gate_of(float x) {
    const float e = __expf(-x), y = 1.0f + e;
    const float r = 0.25f * __builtin_amdgcn_rcpf(__builtin_fmaf(e, 0.25f, 0.25f)), q = x * r;
    return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-y, q, x), r, q), y, x);
}

// All of this wave's loads but the youngest kYounger are in LDS, and all its reads of LDS in registers.
template <int kYounger>
__device__ __forceinline__ void wait_for_all_but() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kYounger) : "memory");
}

// The stages, and behind them each row's scale.
template <int EPI>
constexpr int lds_bytes(int columns, int rows, int stages) {
    return stages * (columns + rows) * 128 + (EPI == DIRECT_SCALED ? rows * static_cast<int>(sizeof(float)) : 0);
}

// kN x kM tiles of 16 columns x 16 rows per wave, kWN waves side by side along the columns and kWM along the rows.
template <int EPI, int kWN, int kWM, int kN, int kM, int kStages>
__global__ void __launch_bounds__(64 * kWN * kWM, 2) gemm_direct_kernel(DirectArgs p) {
#if defined(__HIP_DEVICE_COMPILE__)  // (the host's pass has no type for a buffer's description)
    constexpr int kWaves = kWN * kWM;
    constexpr int kColumns = 16 * kN * kWN, kTileRows = 16 * kM * kWM;
    constexpr int kStageBytes = (kColumns + kTileRows) * 128;
    constexpr int kPieces = (kColumns + kTileRows) / 8;         // loads of 8 rows that a stage takes
    constexpr int kLoads = (kPieces + kWaves - 1) / kWaves;     // ... of a wave; some waves have one fewer
    constexpr int kUneven = kPieces % kWaves;                   // (the first so many waves have kLoads, if it is not 0)
    constexpr int kStep = gates(EPI) ? kColumns / 2 : kColumns;
    static_assert(kStages >= 2 && lds_bytes<EPI>(kColumns, kTileRows, kStages) <= kLdsBytes && (!gates(EPI) || kN % 2 == 0) && (EPI != DIRECT_ROPE || kN % 2 == 0), "");
    extern __shared__ __attribute__((aligned(1024))) char stages[];
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    // workgroups come to the 8 XCDs in turn: each XCD takes a run of neighbouring tiles, row blocks first, so that the
    // tiles that read the same rows of W share an L2
    const int per = (p.tiles + 7) / 8;
    const int tile = (blockIdx.x % 8) * per + blockIdx.x / 8;
    if (static_cast<int>(blockIdx.x) / 8 >= per || tile >= p.tiles) return;
    const int m0 = (tile % p.row_blocks) * kTileRows;
    const int n0 = (tile / p.row_blocks) * kStep;
    const int width = gates(EPI) ? p.N / 2 : p.N;
    const int k_first = blockIdx.y * p.k_per_part;
    const int slices = (min(p.K, k_first + p.k_per_part) - k_first) / kSlice;

    // what this lane fetches: its place in LDS is given (16 bytes behind its neighbour's), so it picks the chunk that belongs there
    const bool uneven_more = kUneven == 0 || wave < kUneven;
    unsigned from[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int row = (wave + kWaves * i) * 8 + lane / 8;
        const int chunk = (lane % 8) ^ ((row >> 1) & 7);
        if (row < kColumns) {
            const int t = row % (16 * kN) / 16, j = row % 16;
            int n;
            if (gates(EPI)) {
                n = min(n0 + row / (16 * kN) * 8 * kN + column_of<EPI, kN>(t, j), width - 1) + t % 2 * width;
            } else if (EPI == DIRECT_ROPE) {  // 16 dimensions of a head's first half, then the 16 they rotate with
                const int per_head = p.rope.head_dim / 32, pair = min((n0 + row) / 32, p.N / 32 - 1);
                n = pair / per_head * p.rope.head_dim + (row / 16 % 2) * (p.rope.head_dim / 2) + pair % per_head * 16 + j;
            } else {
                n = min(n0 + row / (16 * kN) * 16 * kN + column_of<EPI, kN>(t, j), p.N - 1);
            }
            from[i] = (static_cast<unsigned>(n) * p.K + k_first + 8 * chunk) * 2u;
        } else {
            from[i] = (static_cast<unsigned>(min(m0 + row - kColumns, p.M - 1)) * p.lda + k_first + 8 * chunk) * 2u;
        }
    }
    const __amdgpu_buffer_rsrc_t of_w = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(p.w), 0, 0xffffffffu, 0x00027000);
    const __amdgpu_buffer_rsrc_t of_a = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(p.a), 0, 0xffffffffu, 0x00027000);
    auto fetch_one = [&](int i, int slice, int stage) __attribute__((always_inline)) {
        if (i == kLoads - 1 && !uneven_more) return;
        const int piece = wave + kWaves * i;
        char* to = stages + stage * kStageBytes + piece * 1024;
        const bool all_w = kWaves * (i + 1) * 8 <= kColumns, all_a = kWaves * i * 8 >= kColumns;
        if (all_w || (!all_a && piece * 8 < kColumns))
            __builtin_amdgcn_raw_ptr_buffer_load_lds(of_w, (lds_pointer)to, 16, from[i], slice * kSlice * 2, 0, 0);
        else
            __builtin_amdgcn_raw_ptr_buffer_load_lds(of_a, (lds_pointer)to, 16, from[i], slice * kSlice * 2, 0, 0);
    };

    // The rows' 1/rms: behind the first loads, some lanes to a row, eight pieces each at a time
    float* row_scale = reinterpret_cast<float*>(stages + kStages * kStageBytes);  // (SCALED only)
    auto scale_rows = [&] __attribute__((always_inline)) {
        constexpr int kSpare = 64 * kWaves / kTileRows, kPer = kSpare >= 8 ? 8 : kSpare >= 4 ? 4 : 2, kHeld = 8;
        static_assert(kSpare >= 2, "");
        const int row = threadIdx.x / kPer, sub = threadIdx.x % kPer;
        const float* sums = p.row_sumsq + static_cast<size_t>(min(m0 + min(row, kTileRows - 1), p.M - 1)) * p.sumsq_parts;
        float sum = 0.f;
        if (p.sumsq_parts % 4 == 0) {
            for (int first = sub * 4; first < p.sumsq_parts; first += kHeld * kPer * 4) {
                floatx4 held[kHeld];
#pragma unroll
                for (int i = 0; i < kHeld; ++i) held[i] = *reinterpret_cast<const floatx4*>(sums + min(first + i * kPer * 4, p.sumsq_parts - 4));
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < kHeld; ++i)
                    if (first + i * kPer * 4 < p.sumsq_parts) sum += (held[i][0] + held[i][1]) + (held[i][2] + held[i][3]);
            }
        } else {
            for (int at = sub; at < p.sumsq_parts; at += kPer) sum += sums[at];
        }
#pragma unroll
        for (int apart = 1; apart < kPer; apart *= 2) sum += __shfl_xor(sum, apart, kWave);
        if (sub == 0 && row < kTileRows) row_scale[row] = 1.0f / sqrtf(sum / static_cast<float>(p.K) + p.eps);
    };

    const int wn = (wave % kWN) * 16 * kN, wm = kColumns + (wave / kWN) * 16 * kM;  // this wave's rows in a stage
    RowPlaces<kM> places;
    floatx4 acc[kN][kM] = {};
    struct Operands {
        u32x4 w[kN], x[kM];
    };
    auto read_w = [&](Operands& to, int i, const char* at, int h) __attribute__((always_inline)) {
        to.w[i] = *reinterpret_cast<const u32x4*>(at + chunk_at(wn + 16 * i + lane % 16, 4 * h + lane / 16));
    };
    auto read_x = [&](Operands& to, int i, const char* at, int h) __attribute__((always_inline)) {
        to.x[i] = *reinterpret_cast<const u32x4*>(at + chunk_at(wm + 16 * i + lane % 16, 4 * h + lane / 16));
    };
    // Half a slice: the products of `o`, in kN groups; in front of each group some reads of `next` from `at` (the rows of W
    // one group ahead of the place they take) and its share of the loads l0 .. l1 - 1.
    auto half_slice = [&](const Operands& o, Operands& next, const char* at, int h, int l0, int l1, int slice, int stage) __attribute__((always_inline)) {
        constexpr int kSpan = kN > 1 ? kN - 1 : 1, kXStep = (kM + kSpan - 1) / kSpan;
#pragma unroll
        for (int g = 0; g < kN; ++g) {
#pragma unroll
            for (int i = 0; i < kM; ++i)
                if (i >= g * kXStep && i < (g + 1) * kXStep) read_x(next, i, at, h);
            if (g == 0) read_w(next, 0, at, h);
            if (g + 1 < kN) read_w(next, g + 1, at, h);
#pragma unroll
            for (int i = 0; i < kLoads; ++i)
                if (i >= l0 + (l1 - l0) * g / kN && i < l0 + (l1 - l0) * (g + 1) / kN) fetch_one(i, slice, stage);
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int im = 0; im < kM; ++im)
                acc[g][im] = EPI == DIRECT_ATOMIC  // (there a lane has one column of four rows)
                    ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, o.x[im]), __builtin_bit_cast(bf16x8, o.w[g]), acc[g][im], 0, 0, 0)
                    : __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, o.w[g]), __builtin_bit_cast(bf16x8, o.x[im]), acc[g][im], 0, 0, 0);
            __builtin_amdgcn_s_setprio(0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // a slice's loads: all behind the barrier that frees their stage, or, with slices to spare, half of them a half slice later
    constexpr int kFirst = kStages > 2 ? (kLoads + 1) / 2 : kLoads;
    // ... then the barrier.  A wave with one load fewer a slice counts its own.
    constexpr int kAhead = kStages - 2, kFewer = kLoads - 1;
    auto meet = [&] __attribute__((always_inline)) {
        if (uneven_more) wait_for_all_but<kAhead * kLoads>();
        else wait_for_all_but<kAhead * kFewer>();
        asm volatile("s_barrier" ::: "memory");
    };
    auto meet_with_all = [&] __attribute__((always_inline)) {
        wait_for_all_but<0>();
        asm volatile("s_barrier" ::: "memory");
    };

    Operands even, odd;
    const bool many = slices >= kStages;
#pragma unroll
    for (int s = 0; s < kStages - 1; ++s)
        if (s < slices)
#pragma unroll
            for (int i = 0; i < kLoads; ++i) fetch_one(i, s, s);
    if (many)
#pragma unroll
        for (int i = 0; i < kFirst; ++i) fetch_one(i, kStages - 1, kStages - 1);
    if constexpr (EPI == DIRECT_SCALED) scale_rows();
    if (many) {
        if (uneven_more) wait_for_all_but<kAhead * kLoads + kFirst>();
        else wait_for_all_but<kAhead * kFewer + (kFirst < kFewer ? kFirst : kFewer)>();
        asm volatile("s_barrier" ::: "memory");
    } else {
        meet_with_all();
    }
#pragma unroll
    for (int i = 0; i < kN; ++i) read_w(even, i, stages, 0);
#pragma unroll
    for (int i = 0; i < kM; ++i) read_x(even, i, stages, 0);
    int s = 0;
    for (; s + 2 * kStages <= slices; s += kStages)
#pragma unroll
        for (int j = 0; j < kStages; ++j) {
            half_slice(even, odd, stages + j * kStageBytes, 1, kFirst, kLoads, s + j - 1 + kStages, (j + kStages - 1) % kStages);
            meet();
            half_slice(odd, even, stages + (j + 1) % kStages * kStageBytes, 0, 0, kFirst, s + j + kStages, j);
        }
    if (many)
#pragma unroll
        for (int i = kFirst; i < kLoads; ++i) fetch_one(i, s - 1 + kStages, kStages - 1);
    for (int stage = 0; s < slices; ++s) {  // the last ones, fewer than 2 * kStages
        const int next = stage + 1 == kStages ? 0 : stage + 1;
        half_slice(even, odd, stages + stage * kStageBytes, 1, 0, 0, 0, 0);
        if (s + kStages <= slices) meet();
        else meet_with_all();
        if (s + kStages < slices)
#pragma unroll
            for (int i = 0; i < kLoads; ++i) fetch_one(i, s + kStages, stage);
        else if (EPI == DIRECT_ROPE)
            places.step(p, m0 + (wm - kColumns), lane);
        half_slice(odd, even, stages + next * kStageBytes, 0, 0, 0, 0, 0);  // (past the last slice: read and dropped)
        stage = next;
    }

    if constexpr (EPI == DIRECT_ROPE) {
        while (places.known < 3) places.step(p, m0 + (wm - kColumns), lane);
        store_rope<kN, kM>(p, acc, places, n0 / 32 + wn / 32, m0 + (wm - kColumns), lane);
        return;
    }
    if constexpr (EPI == DIRECT_ATOMIC) {  // every part of K adds its share (the hardware's own float add), 16 neighbours at a time
#pragma unroll
        for (int in = 0; in < kN; ++in) {
            const int n = n0 + wn + 16 * in + lane % 16;
            if (n >= p.N) continue;
            const float add = p.bias && blockIdx.y == 0 ? to_float(p.bias[n]) : 0.f;
#pragma unroll
            for (int im = 0; im < kM; ++im)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int m = m0 + (wm - kColumns) + 16 * im + 4 * (lane / 16) + i;
                    if (m < p.M) unsafeAtomicAdd(static_cast<float*>(p.c) + static_cast<size_t>(m) * p.ldc + n, acc[in][im][i] + add);
                }
        }
        return;
    }
    if constexpr (EPI == DIRECT_SCALED) {
#pragma unroll
        for (int im = 0; im < kM; ++im) {
            const float scale = row_scale[wm - kColumns + 16 * im + lane % 16];
#pragma unroll
            for (int in = 0; in < kN; ++in) acc[in][im] *= scale;
        }
    }
    constexpr int kOut = gates(EPI) ? kN / 2 : kN;
    constexpr int kPair = (EPI == DIRECT_BF16 || gates(EPI)) && kOut % 2 == 0 ? 2 : 1;  // tiles whose columns are neighbours
    const int first = n0 + (gates(EPI) ? wn / 2 : wn);
#pragma unroll
    for (int u = 0; u < kOut; u += kPair) {
        const int n = first + column_of<EPI, kN>(gates(EPI) ? 2 * u : u, lane / 16 * 4);
        const bool whole = n + 4 * kPair <= width;
        float b[4 * kPair] = {};
        if (!gates(EPI) && p.bias && blockIdx.y == 0)
#pragma unroll
            for (int i = 0; i < 4 * kPair; ++i) b[i] = to_float(p.bias[min(n + i, width - 1)]);
#pragma unroll
        for (int im = 0; im < kM; ++im) {
            const int m = m0 + (wm - kColumns) + 16 * im + lane % 16;
            if (m >= p.M) continue;
            float v[4 * kPair];
#pragma unroll
            for (int i = 0; i < 4 * kPair; ++i) {
                if constexpr (gates(EPI)) {
                    v[i] = gate_of(acc[2 * (u + i / 4)][im][i % 4]) * acc[2 * (u + i / 4) + 1][im][i % 4];
                } else {
                    v[i] = acc[u + i / 4][im][i % 4] + b[i];
                }
            }
            if constexpr (EPI == DIRECT_BF16 || gates(EPI)) {
                bf16_t* to = static_cast<bf16_t*>(p.c) + static_cast<size_t>(m) * p.ldc + n;
                if (!whole || p.ldc % 2) {
#pragma unroll
                    for (int i = 0; i < 4 * kPair; ++i)
                        if (n + i < width) to[i] = from_float<bf16_t>(v[i]);
                    continue;
                }
                unsigned packed[2 * kPair];
#pragma unroll
                for (int i = 0; i < 2 * kPair; ++i) packed[i] = pack_bf16(v[2 * i], v[2 * i + 1]);
                if (kPair == 2 && p.ldc % 8 == 0) {
                    *reinterpret_cast<u32x4*>(to) = u32x4{packed[0], packed[1], packed[2 * kPair - 2], packed[2 * kPair - 1]};
                } else if (p.ldc % 4 == 0) {
#pragma unroll
                    for (int i = 0; i < kPair; ++i) reinterpret_cast<uint2*>(to)[i] = uint2{packed[2 * i], packed[2 * i + 1]};
                } else {
#pragma unroll
                    for (int i = 0; i < 2 * kPair; ++i) reinterpret_cast<unsigned*>(to)[i] = packed[i];
                }
            } else {
                float* to = static_cast<float*>(p.c) + (static_cast<size_t>(EPI == DIRECT_PARTS ? blockIdx.y : 0) * p.M + m) * p.ldc + n;
                if (whole && p.ldc % 4 == 0) {
                    floatx4 sum = {v[0], v[1], v[2], v[3]};
                    if (EPI == DIRECT_RESID) sum += *reinterpret_cast<const floatx4*>(to);
                    *reinterpret_cast<floatx4*>(to) = sum;
                } else if (whole && p.ldc % 2 == 0) {
#pragma unroll
                    for (int i = 0; i < 4; i += 2) {
                        float2 sum = {v[i], v[i + 1]};
                        if (EPI == DIRECT_RESID) {
                            const float2 was = *reinterpret_cast<const float2*>(to + i);
                            sum.x += was.x;
                            sum.y += was.y;
                        }
                        *reinterpret_cast<float2*>(to + i) = sum;
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (n + i < width) to[i] = EPI == DIRECT_RESID ? to[i] + v[i] : v[i];
                }
            }
        }
    }
#endif
}

template <int EPI, int kWN, int kWM, int kN, int kM, int kStages>
int run(hipStream_t s, DirectArgs& p, int parts) {
    constexpr int kColumns = 16 * kN * kWN, kTileRows = 16 * kM * kWM;
    constexpr int kBytes = lds_bytes<EPI>(kColumns, kTileRows, kStages);
    if (kBytes > 64 * 1024) {  // more than a kernel gets without asking: once per kernel (and again is harmless)
        static bool asked = false;
        if (!asked) {
            if (hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_direct_kernel<EPI, kWN, kWM, kN, kM, kStages>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, kBytes) != hipSuccess) {
                (void)hipGetLastError();
                return CIE_LAUNCH_FAILED;
            }
            asked = true;
        }
    }
    const int step = gates(EPI) ? kColumns / 2 : kColumns;
    const int width = gates(EPI) ? p.N / 2 : p.N;
    p.row_blocks = (p.M + kTileRows - 1) / kTileRows;
    const long tiles = static_cast<long>(p.row_blocks) * ((width + step - 1) / step);
    if (tiles > (1L << 27)) return CIE_BAD_ARGUMENT;
    p.tiles = static_cast<int>(tiles);
    gemm_direct_kernel<EPI, kWN, kWM, kN, kM, kStages><<<dim3((p.tiles + 7) / 8 * 8, parts), 64 * kWN * kWM, kBytes, s>>>(p);
    return cie_after_launch();
}

// Tiles of up to 128 columns and rows: all there are for parts that add atomically and for rows that are scaled.
template <int EPI>
int run_few_form(hipStream_t s, DirectArgs& p, int parts, int columns, int rows) {
    switch (columns * 1000 + rows) {
        case 128128: return run<EPI, 2, 4, 4, 2, 4>(s, p, parts);
        case 128064: return run<EPI, 4, 2, 2, 2, 3>(s, p, parts);
        case 96128: return run<EPI, 1, 8, 6, 1, 5>(s, p, parts);
        case 96064: return run<EPI, 1, 4, 6, 1, 4>(s, p, parts);
        case 64064: return run<EPI, 2, 2, 2, 2, 4>(s, p, parts);
    }
    return CIE_BAD_ARGUMENT;
}

template <int EPI>
int run_form(hipStream_t s, DirectArgs& p, int parts, int columns, int rows) {
    switch (columns * 1000 + rows) {
        case 256256: return run<EPI, 2, 4, 8, 4, 2>(s, p, parts);
        case 256160: return run<EPI, 4, 2, 4, 5, 3>(s, p, parts);
        case 256128: return run<EPI, 4, 2, 4, 4, 3>(s, p, parts);
        case 192256: return run<EPI, 2, 4, 6, 4, 2>(s, p, parts);
        case 192192: return run<EPI, 2, 4, 6, 3, 3>(s, p, parts);
        case 192128: return run<EPI, 2, 4, 6, 2, 3>(s, p, parts);
        case 128256: return run<EPI, 2, 4, 4, 4, 3>(s, p, parts);
        case 128192: return run<EPI, 2, 4, 4, 3, 3>(s, p, parts);
    }
    return run_few_form<EPI>(s, p, parts, columns, rows);
}

bool fits(const void* a, int lda, const void* w, const void* c, int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0 || K % kSlice || lda < K || lda % 8 || !a || !w || !c) return false;
    // (a lane's place in an operand is a 32-bit number of bytes)
    if (static_cast<long>(N) * K >= (1L << 31) || static_cast<long>(M) * lda >= (1L << 31)) return false;
    return ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(c)) & 15) == 0;
}

}  // namespace

// epilogue: 0 bf16, 1 SiLU-gate (N even, no bias), 2 residual (c float32 [M, N]), 3 parts (c float32 [parts, M, N]), 5 parts
// that add their shares into c (float32 [M, N]) with atomic adds (tiles of up to 128 columns and 128 rows).
// `columns` x `rows`: the workgroup's tile of the product (with the gate: half of the columns of either half).
// K is a multiple of 64, lda of 8; a, w and c lie at multiples of 16 bytes; the operands hold fewer than 2^31 numbers.
CIE_API int cie_gemm_direct(void* stream, const void* a, int lda, const void* w, const void* bias, void* c, int ldc, int M,
                            int N, int K, int epilogue, int columns, int rows, int parts) {
    if (!fits(a, lda, w, c, M, N, K) || parts < 1 || parts > 64) return CIE_BAD_ARGUMENT;
    if ((epilogue == DIRECT_SILU && (N % 2 || bias)) || (epilogue != DIRECT_PARTS && epilogue != DIRECT_ATOMIC && parts != 1)) return CIE_BAD_ARGUMENT;
    if (ldc < (epilogue == DIRECT_SILU ? N / 2 : N)) return CIE_BAD_ARGUMENT;
    DirectArgs p{static_cast<const bf16_t*>(a), static_cast<const bf16_t*>(w), static_cast<const bf16_t*>(bias), c, M, N, K, lda, ldc, 0, 0, 0, {}, nullptr, 0, 0.f};
    p.k_per_part = ((K + parts - 1) / parts + kSlice - 1) / kSlice * kSlice;
    if (static_cast<long>(p.k_per_part) * (parts - 1) >= K) return CIE_BAD_ARGUMENT;  // (a part without k)
    hipStream_t s = static_cast<hipStream_t>(stream);
    switch (epilogue) {
        case DIRECT_BF16: return run_form<DIRECT_BF16>(s, p, parts, columns, rows);
        case DIRECT_SILU: return run_form<DIRECT_SILU>(s, p, parts, columns, rows);
        case DIRECT_RESID: return run_form<DIRECT_RESID>(s, p, parts, columns, rows);
        case DIRECT_PARTS: return run_form<DIRECT_PARTS>(s, p, parts, columns, rows);
        case DIRECT_ATOMIC: return run_few_form<DIRECT_ATOMIC>(s, p, parts, columns, rows);
    }
    return CIE_BAD_ARGUMENT;
}

// The SiLU-gate product of rows `a` = bf16(row of the stream x norm weight), whose 1/rms it applies to its sums: `row_sumsq` [M,
// sumsq_parts] are partial sums of squares of the stream's rows (of K numbers).  Tiles of up to 128 columns and 128 rows.
CIE_API int cie_gemm_direct_silu_scaled(void* stream, const void* a, int lda, const void* w, void* c, int ldc, int M, int N, int K,
                                        int columns, int rows, const float* row_sumsq, int sumsq_parts, float eps) {
    if (!fits(a, lda, w, c, M, N, K) || N % 2 || ldc < N / 2 || !row_sumsq || sumsq_parts < 1 || !(eps > 0.f) ||
        (reinterpret_cast<uintptr_t>(row_sumsq) & 15) != 0)
        return CIE_BAD_ARGUMENT;
    DirectArgs p{static_cast<const bf16_t*>(a), static_cast<const bf16_t*>(w), nullptr, c, M, N, K, lda, ldc, K, 0, 0, {}, row_sumsq, sumsq_parts, eps};
    return run_few_form<DIRECT_SCALED>(static_cast<hipStream_t>(stream), p, 1, columns, rows);
}

// The q/k/v product with the rotation and the cache write in its epilogue: `w` [N, K] stacks the rows of q_heads query
// heads, kv_heads key heads and kv_heads value heads of head_dim dimensions (a multiple of 32); `c` [M, N] receives the
// rotated queries (its key and value columns are left alone).
CIE_API int cie_gemm_direct_rope(void* stream, const void* a, int lda, const void* w, const void* bias, void* c, int M, int N,
                                 int K, int columns, int rows, const float* cos_table, const float* sin_table,
                                 const int* positions, const int* seq_of_token, const int* seq_slot, const int* block_table,
                                 int table_width, void* k_pool, void* v_pool, int q_heads, int kv_heads, int head_dim,
                                 int page_size, int rotate, int write_kv) {
    if (!fits(a, lda, w, c, M, N, K)) return CIE_BAD_ARGUMENT;
    if (q_heads <= 0 || kv_heads <= 0 || head_dim <= 0 || head_dim % 32 || page_size <= 0 || table_width <= 0 ||
        N != (q_heads + 2 * kv_heads) * head_dim)
        return CIE_BAD_ARGUMENT;
    if (!positions || (rotate && (!cos_table || !sin_table)) ||
        (write_kv && (!seq_of_token || !seq_slot || !block_table || !k_pool || !v_pool)))
        return CIE_BAD_ARGUMENT;
    DirectArgs p{static_cast<const bf16_t*>(a), static_cast<const bf16_t*>(w), static_cast<const bf16_t*>(bias), c, M, N, K, lda, N, 0, 0, 0,
                 {cos_table, sin_table, positions, seq_of_token, seq_slot, block_table, table_width, static_cast<bf16_t*>(k_pool),
                  static_cast<bf16_t*>(v_pool), q_heads, kv_heads, head_dim, page_size, rotate, write_kv}, nullptr, 0, 0.f};
    p.k_per_part = K;
    return run_form<DIRECT_ROPE>(static_cast<hipStream_t>(stream), p, 1, columns, rows);
}

// bfloat16 products of some hundred rows on the matrix cores: C = A * W^T with A [M, K], W [N, K] bf16 and float32 sums.
// Products whose K is a multiple of 64 are gemm_direct.hip's (faster at every size measured); this one takes any multiple of 8.
// What is measured below are products of such a K, from when they were its own: another K takes as many slices.
//
// Between the few rows that the streaming kernels take (gemm_fused.hip) and the thousands for which the vendor library
// is tuned such a product has few tiles: its time is how many tiles meet on one unit, and the launches behind it.  The
// epilogues take over what stands behind the product:
//   BF16    C[m, n] = bf16(acc + bias[n])
//   SILU    W stacks gate rows over up rows: C[m, n] = bf16(silu(gate) * up)
//   RESID   residual[m, n] += acc + bias[n]  (float32, in place)
//   ROPE    W stacks the rows of q, k and v heads: bias, rounding, rotation by the row's position, queries to C, keys and
//           values into the paged cache (what rope_kv.hip does to the product's output)
//   PARTS   K is cut into grid.y parts, part y leaves acc (with the bias in part 0) in parts[y, m, n] (float32): the
//           norm that adds the branch to the stream sums them, in order, so the result is the same from run to run
//
// Four waves (eight for 256 rows) share a tile of 64 or 128 columns x 64 to 256 rows through two stages of LDS, 64 k to a
// stage, two further slices of 64 k on their way in registers.  W's rows are the A operand of v_mfma_f32_16x16x32_bf16, so
// that a lane ends with four neighbouring columns of one row.
//
// What bounds it: few tiles, the chain of one tile's slices (0.28 to 0.94 us each); many, the rate at which a unit is fed
// from its L2, some 20 bytes a cycle in every shape of tile (2,048 rows, N 22,016, K 2,048: the matrix cores busy 31 % of
// the time, LDS 31 %, no bank conflicts; 128 x 128 tiles 0.84 PFLOP/s, where the library's tiles of 256 x 256, fed at the
// same rate, reach 1.2: 256 x 256 spills here while its slices wait in registers).  Reading LDS for the next half slice while the matrix cores
// work on this one gave 0-20 % where a unit holds one tile (qkv 128 x 64 22.5 -> 17.5 us) and nothing where it holds many.
//
// Measured (MI355X, 3B shape, us; the library's product, and the kernel behind it, in brackets): 256 rows: down in 4 parts
// 26 (38), o_proj 9 (15), q/k/v with rotation and cache write 15 (16 + 5); 613 rows: down in 3 parts 47 (63), q/k/v 19
// (18 + 5); 1,024 rows: down in 4 parts 56 (74).  Gate/up, with the library's gate kernel in its figure: 256 rows 40 (41),
// 613 rows 77 (72), where it stays the library's; of the 0.5B shape 20.8 (26.4) at 613 rows, 48 (49) at 2,048.
#include "common.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

enum { TILE_BF16 = 0, TILE_SILU = 1, TILE_RESID = 2, TILE_PARTS = 3, TILE_ROPE = 4 };

constexpr int kSlice = 64;     // k of a stage: 128 bytes of a row

// What the ROPE epilogue needs beside the product: where each row's token sits, and the cache.
struct TileRope {
    const float *cos_table, *sin_table;  // [max_position, D/2]
    const int *positions, *seq_of_token; // [M]
    const int* seq_slot;                 // [sequences]
    const int* block_table;              // [slots, table_width]
    int table_width;
    bf16_t* k_pool;                      // [pages, Hkv, page_size, D]
    bf16_t* v_pool;                      // [pages, Hkv, D, page_size]
    int q_heads, kv_heads, head_dim, page_size, rotate, write_kv;
};

struct TileArgs {
    const bf16_t *a, *w, *bias;
    void* c;            // BF16, SILU: bf16 [M, ldc]; RESID: the float32 stream; PARTS: float32 [parts, M, N]
    int M, N, K, lda, ldc;
    int k_per_part;     // a multiple of kSlice
    int row_blocks, tiles;
    TileRope rope;      // ROPE only
};

// 16-byte chunk `c` (0..7) of row `row` of a stage: the chunks of 16 rows that are read at one time lie in different banks
__device__ __forceinline__ int chunk_at(int row, int c) { return row * 128 + 16 * (c ^ ((row >> 1) & 7)); }

// The ROPE epilogue of a wave's tiles: pairs `pair`, `pair` + 1, ... of 16 dimensions and the 16 they rotate with.  Values
// are rounded to bf16 before the rotation, so that the results equal those of the plain epilogue followed by the rotation
// kernel.
template <int kN, int kM>
__device__ __forceinline__ void store_rope(const TileArgs& p, const floatx4 (&acc)[kN][kM], int pair, int m_first, int lane) {
    const TileRope& t = p.rope;
    const int D = t.head_dim, half = D / 2, per_head = D / 32;
    int m[kM], pos[kM], page[kM];
    bool there[kM];
#pragma unroll
    for (int im = 0; im < kM; ++im) {
        m[im] = m_first + 16 * im + lane % 16;
        there[im] = m[im] < p.M;
        m[im] = min(m[im], p.M - 1);
        pos[im] = t.positions[m[im]];
        page[im] = t.write_kv ? t.seq_of_token[m[im]] : 0;
    }
#pragma unroll
    for (int im = 0; im < kM; ++im) page[im] = t.write_kv ? t.seq_slot[page[im]] : 0;
#pragma unroll
    for (int im = 0; im < kM; ++im)
        page[im] = t.write_kv ? t.block_table[static_cast<size_t>(page[im]) * t.table_width + pos[im] / t.page_size] : -1;
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
#pragma unroll
        for (int im = 0; im < kM; ++im) {
            if (!there[im] || (!is_query && page[im] < 0)) continue;
            float lo[4], hi[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                lo[i] = to_float(from_float<bf16_t>(acc[in][im][i] + bias_lo[i]));
                hi[i] = to_float(from_float<bf16_t>(acc[in + 1][im][i] + bias_hi[i]));
            }
            const int in_page = pos[im] % t.page_size;
            if (is_value) {
                bf16_t* to = t.v_pool + ((static_cast<size_t>(page[im]) * t.kv_heads + kv_head) * D + d) * t.page_size + in_page;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    to[static_cast<size_t>(i) * t.page_size] = from_float<bf16_t>(lo[i]);
                    to[static_cast<size_t>(half + i) * t.page_size] = from_float<bf16_t>(hi[i]);
                }
                continue;
            }
            if (t.rotate) {
                const floatx4 c = *reinterpret_cast<const floatx4*>(t.cos_table + static_cast<size_t>(pos[im]) * half + d);
                const floatx4 s = *reinterpret_cast<const floatx4*>(t.sin_table + static_cast<size_t>(pos[im]) * half + d);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float x1 = lo[i], x2 = hi[i];
                    lo[i] = x1 * c[i] - x2 * s[i];
                    hi[i] = x2 * c[i] + x1 * s[i];
                }
            }
            bf16_t* to = is_query ? static_cast<bf16_t*>(p.c) + static_cast<size_t>(m[im]) * p.ldc + head * D + d
                                  : t.k_pool + ((static_cast<size_t>(page[im]) * t.kv_heads + kv_head) * t.page_size + in_page) * D + d;
            *reinterpret_cast<uint2*>(to) = uint2{pack_bf16(lo[0], lo[1]), pack_bf16(lo[2], lo[3])};
            *reinterpret_cast<uint2*>(to + half) = uint2{pack_bf16(hi[0], hi[1]), pack_bf16(hi[2], hi[3])};
        }
    }
}

// kN x kM tiles of 16 columns x 16 rows per wave, two waves side by side along the columns and kWM along the rows.
template <int EPI, int kN, int kM, int kWM>
__global__ void __launch_bounds__(128 * kWM, 2) gemm_tiles_kernel(TileArgs p) {
    constexpr int kThreads = 128 * kWM;
    constexpr int kColumns = 32 * kN, kTileRows = 16 * kM * kWM;
    constexpr int kRows = kColumns + kTileRows;       // of W, then of A, in a stage
    constexpr int kPerLoad = kThreads / 8;            // rows that the threads' 16-byte loads cover at a time
    constexpr int kLoads = kRows / kPerLoad;
    constexpr int kWLoads = kColumns / kPerLoad;
    constexpr int kAhead = 2;
    constexpr int kStep = EPI == TILE_SILU ? kColumns / 2 : kColumns;  // output columns of a tile
    extern __shared__ __attribute__((aligned(16))) char stages[];      // two of kRows * 128 bytes
    const int lane = threadIdx.x % kWave;
    const int wave = threadIdx.x / kWave;
    // workgroups come to the 8 XCDs in turn: each XCD takes a run of neighbouring tiles, row blocks first, so that the
    // tiles that read the same rows of W share an L2
    const int per = (p.tiles + 7) / 8;
    const int tile = (blockIdx.x % 8) * per + blockIdx.x / 8;
    if (static_cast<int>(blockIdx.x) / 8 >= per || tile >= p.tiles) return;
    const int m0 = (tile % p.row_blocks) * kTileRows;
    const int n0 = (tile / p.row_blocks) * kStep;
    const int width = EPI == TILE_SILU ? p.N / 2 : p.N;
    const int k_first = blockIdx.y * p.k_per_part;
    const int k_end = min(p.K, k_first + p.k_per_part);

    const int chunk = threadIdx.x % 8;
    const bf16_t* row_of[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int r = threadIdx.x / 8 + kPerLoad * i;
        int n = min(n0 + r, p.N - 1);
        if (EPI == TILE_SILU) {
            n = min(n0 + r / 32 * 16 + r % 16, width - 1) + (r / 16 % 2) * width;
        } else if (EPI == TILE_ROPE) {  // 16 dimensions of a head's first half, then the 16 they rotate with
            const int per_head = p.rope.head_dim / 32, pair = min(n0 / 32 + r / 32, p.N / 32 - 1);
            n = pair / per_head * p.rope.head_dim + (r / 16 % 2) * (p.rope.head_dim / 2) + pair % per_head * 16 + r % 16;
        }
        row_of[i] = (i < kWLoads ? p.w + static_cast<size_t>(n) * p.K
                                 : p.a + static_cast<size_t>(min(m0 + r - kColumns, p.M - 1)) * p.lda) + 8 * chunk;
    }
    u32x4 ahead[kAhead][kLoads];
    // (a piece past the end reads the part's last piece again: no load stands under a condition)
    auto fetch = [&](u32x4 (&to)[kLoads], int slice) {
        const int k = min(k_first + slice * kSlice, k_end - 8 - 8 * chunk);
#pragma unroll
        for (int i = 0; i < kLoads; ++i) to[i] = *reinterpret_cast<const u32x4*>(row_of[i] + k);
    };
    auto put = [&](u32x4 (&from)[kLoads], int slice, char* to) {
        if (k_first + (slice + 1) * kSlice > k_end) {  // (the same for all: what lies past the end is 0)
            const bool inside = k_first + slice * kSlice + 8 * chunk < k_end;
#pragma unroll
            for (int i = 0; i < kLoads; ++i) from[i] = inside ? from[i] : u32x4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int i = 0; i < kLoads; ++i)
            *reinterpret_cast<u32x4*>(to + chunk_at(threadIdx.x / 8 + kPerLoad * i, chunk)) = from[i];
    };

    const int slices = (k_end - k_first + kSlice - 1) / kSlice;
    const int wn = (wave % 2) * 16 * kN, wm = kColumns + (wave / 2) * 16 * kM;  // this wave's rows in a stage
    floatx4 acc[kN][kM] = {};
    struct Operands {
        u32x4 w[kN], x[kM];
    };
    auto read = [&](Operands& to, const char* from, int s) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kN; ++i) to.w[i] = *reinterpret_cast<const u32x4*>(from + chunk_at(wn + 16 * i + lane % 16, 4 * s + lane / 16));
#pragma unroll
        for (int i = 0; i < kM; ++i) to.x[i] = *reinterpret_cast<const u32x4*>(from + chunk_at(wm + 16 * i + lane % 16, 4 * s + lane / 16));
    };
    auto multiply = [&](const Operands& o) __attribute__((always_inline)) {
#pragma unroll
        for (int in = 0; in < kN; ++in)
#pragma unroll
            for (int im = 0; im < kM; ++im)
                acc[in][im] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, o.w[in]),
                                                                      __builtin_bit_cast(bf16x8, o.x[im]), acc[in][im], 0, 0, 0);
    };
    // What the matrix cores need next is read from LDS, and the next slice written there, while they work: a slice's two
    // halves of 32 k take turns in two sets of operands, and the barrier stands between a slice's halves.
    Operands first_half, second_half;
    fetch(ahead[0], 0);
    put(ahead[0], 0, stages);
#pragma unroll
    for (int a = 0; a < kAhead; ++a) fetch(ahead[(a + 1) % kAhead], a + 1);
    __syncthreads();
    read(first_half, stages, 0);
    for (int first = 0; first < slices; first += 2) {
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            const int slice = first + a;
            char* here = stages + a * kRows * 128;
            char* other = stages + (1 - a) * kRows * 128;
            read(second_half, here, 1);
            // (the other stage was last read in the slice before, and all waves have passed a barrier since)
            put(ahead[(a + 1) % kAhead], slice + 1, other);
            fetch(ahead[(a + 1) % kAhead], slice + 1 + kAhead);
            multiply(first_half);
            __syncthreads();
            read(first_half, other, 0);
            multiply(second_half);
        }
    }

    if constexpr (EPI == TILE_ROPE) {
        store_rope<kN, kM>(p, acc, n0 / 32 + wn / 32, m0 + (wm - kColumns), lane);
        return;
    }
#pragma unroll
    for (int in = 0; in < kN; in += EPI == TILE_SILU ? 2 : 1) {
        const int n = n0 + (EPI == TILE_SILU ? wn / 2 + 8 * in : wn + 16 * in) + 4 * (lane / 16);
        floatx4 b = {0.f, 0.f, 0.f, 0.f};
        if (EPI != TILE_SILU && p.bias && blockIdx.y == 0)
#pragma unroll
            for (int i = 0; i < 4; ++i) b[i] = to_float(p.bias[min(n + i, width - 1)]);
#pragma unroll
        for (int im = 0; im < kM; ++im) {
            const int m = m0 + (wm - kColumns) + 16 * im + lane % 16;
            if (m >= p.M) continue;
            floatx4 v = acc[in][im] + b;
            if constexpr (EPI == TILE_SILU) {
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = (v[i] / (1.0f + __expf(-v[i]))) * acc[in + 1][im][i];
            }
            const bool whole = n + 3 < width && p.ldc % 4 == 0;
            if constexpr (EPI == TILE_BF16 || EPI == TILE_SILU) {
                bf16_t* to = static_cast<bf16_t*>(p.c) + static_cast<size_t>(m) * p.ldc + n;
                if (whole) {
                    *reinterpret_cast<uint2*>(to) = uint2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (n + i < width) to[i] = from_float<bf16_t>(v[i]);
                }
            } else {
                float* to = static_cast<float*>(p.c) + (static_cast<size_t>(EPI == TILE_PARTS ? blockIdx.y : 0) * p.M + m) * p.ldc + n;
                if (whole) {
                    if (EPI == TILE_RESID) v += *reinterpret_cast<const floatx4*>(to);
                    *reinterpret_cast<floatx4*>(to) = v;
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (n + i < width) to[i] = EPI == TILE_RESID ? to[i] + v[i] : v[i];
                }
            }
        }
    }
}

template <int EPI, int kN, int kM, int kWM>
int run(hipStream_t s, TileArgs& p, int parts) {
    constexpr int kBytes = 2 * (32 * kN + 16 * kM * kWM) * 128;
    if (kBytes > 64 * 1024) {  // more than a kernel gets without asking: once per kernel (and again is harmless)
        static bool asked = false;
        if (!asked) {
            if (hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_tiles_kernel<EPI, kN, kM, kWM>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, kBytes) != hipSuccess) {
                (void)hipGetLastError();
                return CIE_LAUNCH_FAILED;
            }
            asked = true;
        }
    }
    const int step = EPI == TILE_SILU ? 16 * kN : 32 * kN;
    const int width = EPI == TILE_SILU ? p.N / 2 : p.N;
    p.row_blocks = (p.M + 16 * kM * kWM - 1) / (16 * kM * kWM);
    const long tiles = static_cast<long>(p.row_blocks) * ((width + step - 1) / step);
    if (tiles > (1L << 30)) return CIE_BAD_ARGUMENT;
    p.tiles = static_cast<int>(tiles);
    gemm_tiles_kernel<EPI, kN, kM, kWM><<<dim3((p.tiles + 7) / 8 * 8, parts), 128 * kWM, kBytes, s>>>(p);
    return cie_after_launch();
}

template <int EPI>
int run_form(hipStream_t s, TileArgs& p, int parts, int columns, int rows) {
    if (columns == 128 && rows == 128) return run<EPI, 4, 4, 2>(s, p, parts);
    if (columns == 128 && rows == 64) return run<EPI, 4, 2, 2>(s, p, parts);
    if (columns == 64 && rows == 64) return run<EPI, 2, 2, 2>(s, p, parts);
    if (columns == 128 && rows == 256) return run<EPI, 4, 4, 4>(s, p, parts);
    return CIE_BAD_ARGUMENT;
}

}  // namespace

// epilogue: 0 bf16, 1 SiLU-gate (N even, no bias), 2 residual (c float32 [M, N]), 3 parts (c float32 [parts, M, N]).
// `columns` x `rows`: the workgroup's tile of the product (with the gate: half of the columns of either half).
// K and lda are multiples of 8; a, w and c lie at multiples of 16 bytes.
CIE_API int cie_gemm_tiles(void* stream, const void* a, int lda, const void* w, const void* bias, void* c, int ldc, int M,
                           int N, int K, int epilogue, int columns, int rows, int parts) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 8 || lda < K || lda % 8 || !a || !w || !c || parts < 1 || parts > 64) return CIE_BAD_ARGUMENT;
    if (((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(c)) & 15) != 0) return CIE_BAD_ARGUMENT;
    if ((epilogue == TILE_SILU && (N % 2 || bias)) || (epilogue != TILE_PARTS && parts != 1)) return CIE_BAD_ARGUMENT;
    if (ldc < (epilogue == TILE_SILU ? N / 2 : N)) return CIE_BAD_ARGUMENT;
    TileArgs p{static_cast<const bf16_t*>(a), static_cast<const bf16_t*>(w), static_cast<const bf16_t*>(bias), c, M, N, K, lda, ldc, 0, 0, 0, {}};
    p.k_per_part = ((K + parts - 1) / parts + kSlice - 1) / kSlice * kSlice;
    if (static_cast<long>(p.k_per_part) * (parts - 1) >= K) return CIE_BAD_ARGUMENT;  // (a part without k)
    hipStream_t s = static_cast<hipStream_t>(stream);
    switch (epilogue) {
        case TILE_BF16: return run_form<TILE_BF16>(s, p, parts, columns, rows);
        case TILE_SILU: return run_form<TILE_SILU>(s, p, parts, columns, rows);
        case TILE_RESID: return run_form<TILE_RESID>(s, p, parts, columns, rows);
        case TILE_PARTS: return run_form<TILE_PARTS>(s, p, parts, columns, rows);
    }
    return CIE_BAD_ARGUMENT;
}

// The q/k/v product with the rotation and the cache write in its epilogue: `w` [N, K] stacks the rows of q_heads query
// heads, kv_heads key heads and kv_heads value heads of head_dim dimensions (a multiple of 32); `c` [M, N] receives the
// rotated queries (its key and value columns are left alone).
CIE_API int cie_gemm_tiles_rope(void* stream, const void* a, int lda, const void* w, const void* bias, void* c, int M, int N,
                                int K, int columns, int rows, const float* cos_table, const float* sin_table,
                                const int* positions, const int* seq_of_token, const int* seq_slot, const int* block_table,
                                int table_width, void* k_pool, void* v_pool, int q_heads, int kv_heads, int head_dim,
                                int page_size, int rotate, int write_kv) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 8 || lda < K || lda % 8 || !a || !w || !c) return CIE_BAD_ARGUMENT;
    if (((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(c)) & 15) != 0) return CIE_BAD_ARGUMENT;
    if (q_heads <= 0 || kv_heads <= 0 || head_dim <= 0 || head_dim % 32 || page_size <= 0 || table_width <= 0 ||
        N != (q_heads + 2 * kv_heads) * head_dim)
        return CIE_BAD_ARGUMENT;
    if (!positions || (rotate && (!cos_table || !sin_table)) ||
        (write_kv && (!seq_of_token || !seq_slot || !block_table || !k_pool || !v_pool)))
        return CIE_BAD_ARGUMENT;
    TileArgs p{static_cast<const bf16_t*>(a), static_cast<const bf16_t*>(w), static_cast<const bf16_t*>(bias), c, M, N, K, lda, N, 0, 0, 0,
               {cos_table, sin_table, positions, seq_of_token, seq_slot, block_table, table_width, static_cast<bf16_t*>(k_pool),
                static_cast<bf16_t*>(v_pool), q_heads, kv_heads, head_dim, page_size, rotate, write_kv}};
    p.k_per_part = (K + kSlice - 1) / kSlice * kSlice;
    return run_form<TILE_ROPE>(static_cast<hipStream_t>(stream), p, 1, columns, rows);
}

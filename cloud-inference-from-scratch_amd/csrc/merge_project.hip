// The output product of a decode step's attention, on the shares of the keys as the attention kernel left them: the merge of the
// shares rides in the product's operand.
//
//   residual[m, :] += merge(shares of row m) * W^T + bias      up to 16 rows (one token a sequence), W [N, heads * D] bf16
//
// A workgroup owns 128 of the product's k (one head of 128 dimensions, two of 64, ...) and 128 or 512 columns.  Its waves ask
// for their tiles of W first; then all threads merge the rows' shares of these 128 k (a thread four dimensions of a row and every
// GROUPS-th share; the groups meet in LDS by their maxima), round to bf16 as a merge kernel would, and pass the rows through LDS
// into the matrix operand.  Every workgroup adds its 128 k to the float32 stream with atomic adds.
//
// What bounds it: the chain W or shares -> LDS -> product -> atomics, 16 KB of W and 64 KB of shares a workgroup.  The workgroups of one slice of k
// follow one another by the number of slices, so that (16 slices, 8 XCDs) an XCD's L2 fetches the shares of two heads, not of all.
// In place of a merge kernel and a product whose waves share K, which leaves the stream's sums of squares; the SiLU-gate product
// behind it then makes its norm itself (gemm_fused.hip).  MI355X, us, attention, merge and product before and with this kernel, over
// 4,000 keys: 16 heads of 128 on 2, 2,048 columns 1 row 15.9 -> 10.4, 8 rows 21.1 -> 16.1, 16 rows 26.8 -> 21.4; 14 heads of 64 on 2, 896
// columns 8 rows 15.0 -> 11.0; 28 heads on 4, 3,584 columns 1 row 19.8 -> 17.1, 8 rows 30.1 -> 26.5 (with 128 columns a workgroup 28.9,
// every workgroup merging anew); 40 heads on 8, 5,120 columns 8 rows 45 -> 47 to 49: the sums of 40 slices that meet in the stream.
#include "common.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * kWave;
constexpr int kSlice = 128;                   // k of a workgroup
constexpr int kChunks = kSlice / 4;           // threads that cover a row of them
constexpr int kRows = 16;
constexpr int kRowBytes = kSlice * 2 + 16;    // of a row in LDS: the padding spreads the rows over the banks
constexpr int kAhead = 8;                     // shares whose loads a thread has under way at once

struct MergeProjectArgs {
    const float* part_o;   // [rows, kv_heads, splits, tile_rows, D]
    const float* part_ml;  // [rows, kv_heads, splits, tile_rows, 2]: maximum (base 2) and sum
    const bf16_t* w;       // [N, K]
    const bf16_t* bias;    // [N] or null
    float* residual;       // [M, N]
    int M, N, K;
    int q_heads, kv_heads, head_dim, n_splits, tile_rows;
};

// PADDED: M rounded up to a power of two.  TILES: tiles of 16 columns a wave.
template <int PADDED, int TILES>
__global__ void __launch_bounds__(kThreads) merge_project_kernel(MergeProjectArgs a) {
    constexpr int kItems = PADDED * kChunks;
    constexpr int kGroups = kThreads / kItems;
    __shared__ floatx4 group_sum[kGroups > 1 ? kThreads : 1];
    __shared__ float2 group_ml[kGroups > 1 ? kThreads : 1];
    __shared__ __attribute__((aligned(16))) char rows_lds[kRows * kRowBytes];
    const int lane = threadIdx.x % kWave;
    const int wave = threadIdx.x / kWave;
    const int r = lane & 15;
    const int g = lane >> 4;
    const int slices = a.K / kSlice;
    const int slice = blockIdx.x % slices;
    const int first = (blockIdx.x / slices * kWaves + wave) * TILES * 16;  // the wave's first column

    // the wave's tiles of W in the operand layout: lane (r, g) row r, k j * 32 + g * 8 .. +7 (a column past the end reads the last)
    u32x4 w[TILES][4];
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
        const bf16_t* row = a.w + static_cast<size_t>(min(first + t * 16 + r, a.N - 1)) * a.K + slice * kSlice + g * 8;
#pragma unroll
        for (int j = 0; j < 4; ++j) w[t][j] = *reinterpret_cast<const u32x4*>(row + j * 32);
    }

    const int item = threadIdx.x % kItems;
    const int mine = threadIdx.x / kItems;
    const int m = item / kChunks;
    const int column = slice * kSlice + (item % kChunks) * 4;
    const int head = column / a.head_dim;
    const int kv_head = head / (a.q_heads / a.kv_heads);
    const int row = head - kv_head * (a.q_heads / a.kv_heads);
    const size_t place0 = (static_cast<size_t>(min(m, a.M - 1)) * a.kv_heads + kv_head) * a.n_splits * a.tile_rows + row;
    const float* sums_at = a.part_o + place0 * a.head_dim + (column - head * a.head_dim);
    const float* ml_at = a.part_ml + place0 * 2;
    floatx4 num = {0.f, 0.f, 0.f, 0.f};
    float m_all = -INFINITY, den = 0.f;
#pragma unroll 1
    for (int s0 = mine; s0 < a.n_splits; s0 += kAhead * kGroups) {
        float2 ml[kAhead];
        floatx4 sums[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u)  // (a share past the last reads the last again, and is dropped below)
            ml[u] = *reinterpret_cast<const float2*>(ml_at + static_cast<size_t>(min(s0 + u * kGroups, a.n_splits - 1)) * a.tile_rows * 2);
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
            sums[u] = *reinterpret_cast<const floatx4*>(sums_at + static_cast<size_t>(min(s0 + u * kGroups, a.n_splits - 1)) * a.tile_rows * a.head_dim);
        __builtin_amdgcn_sched_barrier(0);
        float most = m_all;
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            ml[u].x = s0 + u * kGroups < a.n_splits ? ml[u].x : -INFINITY;
            most = fmaxf(most, ml[u].x);
        }
        const float keep = m_all == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_all - most);
        den *= keep;
        num = keep != 0.f ? num * keep : floatx4{0.f, 0.f, 0.f, 0.f};
        m_all = most;
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const float weight = ml[u].x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml[u].x - most);  // maxima are kept in base 2
            const float with = den + ml[u].y * weight;
            den = s0 + u * kGroups < a.n_splits ? with : den;
            const floatx4 more = num + sums[u] * weight;
#pragma unroll
            for (int i = 0; i < 4; ++i) num[i] = weight != 0.f ? more[i] : num[i];  // (a share without keys wrote no sums)
        }
    }
    if constexpr (kGroups > 1) {
        group_sum[threadIdx.x] = num;
        group_ml[threadIdx.x] = float2{m_all, den};
        __syncthreads();
        if (threadIdx.x < kItems) {
            float most = m_all;
#pragma unroll
            for (int u = 1; u < kGroups; ++u) most = fmaxf(most, group_ml[u * kItems + item].x);
            const float keep = m_all == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_all - most);
            den *= keep;
            num = keep != 0.f ? num * keep : floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int u = 1; u < kGroups; ++u) {
                const float2 ml = group_ml[u * kItems + item];
                const float weight = ml.x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml.x - most);
                den += ml.y * weight;
                const floatx4 more = num + group_sum[u * kItems + item] * weight;
                num = weight != 0.f ? more : num;
            }
        }
    }
    if (threadIdx.x < kItems) {
        const float inv = 1.0f / den;
        *reinterpret_cast<uint2*>(rows_lds + m * kRowBytes + (item % kChunks) * 8) =
            uint2{pack_bf16(num[0] * inv, num[1] * inv), pack_bf16(num[2] * inv, num[3] * inv)};
    }
    __syncthreads();
    // (rows past PADDED hold whatever LDS held: a row of the product depends on its own row only, and theirs are not stored)
    u32x4 av[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) av[j] = *reinterpret_cast<const u32x4*>(rows_lds + r * kRowBytes + j * 64 + g * 16);
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
        floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; ++j)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av[j]), __builtin_bit_cast(bf16x8, w[t][j]), acc, 0, 0, 0);
        const int n = first + t * 16 + r;
        const float add = a.bias && slice == 0 ? to_float(a.bias[min(n, a.N - 1)]) : 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (n < a.N && g * 4 + i < a.M) unsafeAtomicAdd(a.residual + static_cast<size_t>(g * 4 + i) * a.N + n, acc[i] + add);
    }
}

template <int PADDED>
int launch(hipStream_t s, int tiles, const MergeProjectArgs& a) {
    const long slices = a.K / kSlice;
    const long groups = (a.N + kWaves * tiles * 16 - 1) / (kWaves * tiles * 16);
    if (slices * groups > 0x7fffffffL) return CIE_BAD_ARGUMENT;
    const dim3 grid(static_cast<unsigned>(slices * groups));
    if (tiles == 1) merge_project_kernel<PADDED, 1><<<grid, kThreads, 0, s>>>(a);
    else merge_project_kernel<PADDED, 4><<<grid, kThreads, 0, s>>>(a);
    return cie_after_launch();
}

}  // namespace

// Row m is the one token of tile m: part_o [M, kv_heads, n_splits, tile_rows, head_dim] and part_ml (the same without head_dim, two
// numbers each) as cie_paged_attention_mfma leaves them, q_heads / kv_heads rows of a tile.  residual [M, N] float32 += merged * W^T
// + bias, W [N, q_heads * head_dim] bf16 at a 16-byte address; q_heads * head_dim a multiple of 128, head_dim of 4.  tiles: 1 or 4 tiles
// of 16 columns a wave.
CIE_API int cie_merge_project(void* stream, const float* part_o, const float* part_ml, const void* w, const void* bias, float* residual,
                              int M, int N, int q_heads, int kv_heads, int head_dim, int n_splits, int tile_rows, int tiles) {
    if (M < 1 || M > kRows || N < 1 || q_heads < 1 || kv_heads < 1 || q_heads % kv_heads || head_dim < 4 || head_dim % 4 ||
        (static_cast<long>(q_heads) * head_dim) % kSlice || n_splits < 1 || tile_rows < q_heads / kv_heads || (tiles != 1 && tiles != 4) ||
        !part_o || !part_ml || !w || !residual)
        return CIE_BAD_ARGUMENT;
    MergeProjectArgs a{part_o, part_ml, static_cast<const bf16_t*>(w), static_cast<const bf16_t*>(bias), residual,
                       M, N, q_heads * head_dim, q_heads, kv_heads, head_dim, n_splits, tile_rows};
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (M == 1) return launch<1>(s, tiles, a);
    if (M == 2) return launch<2>(s, tiles, a);
    if (M <= 4) return launch<4>(s, tiles, a);
    if (M <= 8) return launch<8>(s, tiles, a);
    return launch<16>(s, tiles, a);
}

// Mixers that carry a state of fixed size from token to token instead of a growing cache.  Every state lives in
// float32 rows of a state tensor, one row per request slot; a step reads the row its earlier steps left, runs its
// tokens in order and writes the row back, so a sequence may be cut into steps anywhere.
//
// 1. retention: a memory S [dim, vdim] per head that fades by a fixed factor per token,
//        S_t = decay * S_(t-1) + k_t v_t^T,   o_t = S_t^T q_t,
//    q and k turned by the token's position (the first `rot` dimensions of a head, pair (i, i + rot/2)), k scaled
//    after the turn; o_t divided by its root mean square over the head and multiplied by silu(gate).
// 2. a causal convolution over each channel's own last `taps` inputs, the inputs of the tokens before the step taken
//    from the state.
// 3. a gated linear recurrence per channel,
//        a = exp(c * sigmoid(r)),  S_t = a * S_(t-1) + sqrt(1 - a^2) * sigmoid(i) * u_t,   out_t = S_t * gelu(y_t),
//    with c = -8 softplus(lambda) < 0 made once per model; it also moves the convolution's state on.
//
// Sequence s of the step brings tokens q_start_loc[s] .. q_start_loc[s + 1] - 1 of the flat token axis, the first at
// position seq_start[s]; its state row is seq_slot[s].
#include "common.h"

namespace {

__device__ __forceinline__ float sigmoidf(float x) { return 1.0f / (1.0f + expf(-x)); }

// what stands between a projection and the memory: 0 nothing, 1 silu
__device__ __forceinline__ float activated(float z, int act) { return act == 1 ? z * sigmoidf(z) : z; }

__device__ __forceinline__ float gelu_tanh(float z) {
    return 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
}

// ---------------------------------------------------------------------------------------------- retention
// Three kernels, or one for steps of one token a sequence (d).  (a) Every token's queries and keys, turned by its position, the keys scaled, as float32 rows padded
// with zeros to `padded` numbers per head: [tokens, heads, 2, padded] (what passes through an activation on its way in
// does so here).  (b) The walk over the tokens, below, token by token for steps of few tokens a sequence, or (b') in
// blocks on the matrix cores for prompts' portions.  (c) The norm over a head's or over several heads' read-outs, the
// norm's weight and the gate, which need all value columns of the heads that share a root mean square.
//
// (b) A column of the memory never meets another column, and o_t is a sum over the memory's rows, so one workgroup
// takes (sequence, head, slice of up to 64 value columns, part of the rows) and the parts' shares of o_t are added
// up by (c): as many parts as give every compute unit a workgroup (a prompt of one sequence with 8 heads of 128 x 256
// would otherwise keep 32 of 256 units busy, each walking its 2,048 tokens at 64 multiply-adds per thread and token).
// Thread (column v, group g) keeps rows r0 + g * DS .. + DS - 1 of column v in registers.  Tokens go in chunks:
// the chunk's queries, keys and values are staged in LDS, every thread walks the chunk's tokens in order (no
// barrier between tokens; a thread reads its DS numbers of a query as 16-byte pieces), and the groups' shares are
// summed into the part's float32 plane [tokens, heads * vdim].  The next chunk's numbers are fetched into
// registers before the walk over the current one starts, so that their way from memory is hidden behind it.
template <typename T>
__global__ void __launch_bounds__(256)
retention_turn_kernel(const T* __restrict__ proj, long ldp, int q_off, int k_off, const float* __restrict__ cos_table,
                      const float* __restrict__ sin_table, int rot, const int* __restrict__ positions,
                      float* __restrict__ turned, int heads, int dim, int padded, float key_scale, int act) {
    const int token = blockIdx.x;
    const int half = rot / 2;
    const T* row = proj + static_cast<size_t>(token) * ldp;
    const size_t at = static_cast<size_t>(positions[token]) * half;
    // (few tokens: the workgroups of a token, blockIdx.y, share its heads' numbers)
    for (int idx = blockIdx.y * blockDim.x + threadIdx.x; idx < heads * padded; idx += blockDim.x * gridDim.y) {
        const int head = idx / padded;
        const int d = idx - head * padded;
        float qv = 0.f, kv = 0.f;
        if (d < dim) {
            const T* qh = row + q_off + head * dim;
            const T* kh = row + k_off + head * dim;
            qv = activated(to_float(qh[d]), act);
            kv = activated(to_float(kh[d]), act);
            if (d < rot) {
                const int i = d < half ? d : d - half;
                const float c = cos_table[at + i], s = sin_table[at + i];
                if (d < half) {
                    qv = qv * c - activated(to_float(qh[d + half]), act) * s;
                    kv = kv * c - activated(to_float(kh[d + half]), act) * s;
                } else {
                    qv = qv * c + activated(to_float(qh[i]), act) * s;
                    kv = kv * c + activated(to_float(kh[i]), act) * s;
                }
            }
        }
        float* dst = turned + ((static_cast<size_t>(token) * heads + head) * 2) * padded + d;
        dst[0] = qv;
        dst[padded] = kv * key_scale;
    }
}

typedef float piece_t __attribute__((ext_vector_type(4)));  // 16 bytes that stay in registers (as a struct of four
                                                            // floats, the pieces fetched ahead went through scratch memory)

constexpr int kFetchPieces = 6;  // 16-byte pieces of a chunk's queries and keys that a thread fetches ahead
constexpr int kFetchValues = 12; // ... and values

// the chunk that starts at token `from`: this thread's pieces into its registers.  Every load stands in straight-line
// code without a condition (a piece or value past the chunk's end reads the chunk's last one again, a column past the
// head's last its last): behind a load under a condition the compiler waits for it before it issues the next, and
// the eighteen loads of a thread became eighteen round trips to memory per chunk.
#define CIE_RETENTION_FETCH(from)                                                                                     \
    {                                                                                                                 \
        const int fetch_n = min(chunk, count - (from));                                                               \
        _Pragma("unroll") for (int i = 0; i < kFetchPieces; ++i) {                                                    \
            const int idx = min(static_cast<int>(threadIdx.x + i * blockDim.x), fetch_n * pieces - 1);                \
            const int t = idx / pieces;                                                                               \
            const int piece = idx - t * pieces;                                                                       \
            const int side = piece / (rows / 4); /* 0: the query, 1: the key */                                       \
            ahead[i] = *reinterpret_cast<const piece_t*>(                                                             \
                turned + ((static_cast<size_t>(first + (from) + t) * heads + head) * 2 + side) * padded + r0 +        \
                (piece - side * (rows / 4)) * 4);                                                                     \
        }                                                                                                             \
        _Pragma("unroll") for (int i = 0; i < kFetchValues; ++i) {                                                    \
            const int idx = min(static_cast<int>(threadIdx.x + i * blockDim.x), fetch_n * slice - 1);                 \
            const int t = idx / slice;                                                                                \
            const int c = min(v0 + idx - t * slice, vdim - 1);                                                        \
            ahead_v[i] = proj[static_cast<size_t>(first + (from) + t) * ldp + v_off + head * vdim + c];               \
        }                                                                                                             \
    }

template <typename T, int DS>
__global__ void __launch_bounds__(512)
retention_kernel(const T* __restrict__ proj, long ldp, int v_off, const float* __restrict__ turned,
                 const float* __restrict__ decay, float* __restrict__ state, const int* __restrict__ seq_slot,
                 const int* __restrict__ q_start_loc, float* __restrict__ raw, long plane,
                 int heads, int dim, int vdim, int slice, int slices, int groups, int padded, int chunk, int act) {
    extern __shared__ float4 lds4[];
    float* lds = reinterpret_cast<float*>(lds4);
    const int rows = groups * DS;              // rows of the memory that this workgroup keeps
    float* qk_s = lds;                         // [chunk][2][rows]: a token's query, then its key
    float* v_s = qk_s + chunk * 2 * rows;      // [chunk][slice]
    float* o_s = v_s + chunk * slice;          // [groups][chunk][slice]
    const int seq = blockIdx.x;
    const int head = blockIdx.y;
    const int part = blockIdx.z / slices;
    const int v0 = (blockIdx.z - part * slices) * slice;
    const int r0 = part * rows;
    const int first = q_start_loc[seq];
    const int count = q_start_loc[seq + 1] - first;
    const int slot = seq_slot[seq];
    const int col = threadIdx.x % slice;
    const int grp = threadIdx.x / slice;
    const bool owner = grp < groups && v0 + col < vdim;
    const int d0 = r0 + grp * DS;
    const float fade = decay[head];
    const int pieces = 2 * rows / 4;           // 16-byte pieces of one token's query and key rows
    float* mem = state + ((static_cast<size_t>(slot) * heads + head) * dim) * vdim + v0 + col;
    float* mine = raw + static_cast<size_t>(part) * plane;
    float S[DS];
#pragma unroll
    for (int r = 0; r < DS; ++r) S[r] = (owner && d0 + r < dim) ? mem[static_cast<size_t>(d0 + r) * vdim] : 0.f;
    piece_t ahead[kFetchPieces];
    T ahead_v[kFetchValues];  // (as stored: a conversion right behind the load would wait for it, and for all loads before it)
    if (count > 0) CIE_RETENTION_FETCH(0)
    for (int c0 = 0; c0 < count; c0 += chunk) {
        const int cn = min(chunk, count - c0);
#pragma unroll
        for (int i = 0; i < kFetchPieces; ++i) {
            const int idx = threadIdx.x + i * blockDim.x;
            if (idx < cn * pieces) reinterpret_cast<piece_t*>(qk_s)[idx] = ahead[i];
        }
#pragma unroll
        for (int i = 0; i < kFetchValues; ++i) {
            const int idx = threadIdx.x + i * blockDim.x;
            if (idx < cn * slice) v_s[idx] = activated(to_float(ahead_v[i]), act);
        }
        __syncthreads();
        if (c0 + chunk < count) CIE_RETENTION_FETCH(c0 + chunk)
        if (owner) {
            // (a token's numbers are read from LDS while the token before it is worked on: with one wave per SIMD
            // nothing else would hide the way from LDS, and it is as long as the arithmetic of a token)
            const float* q_base = qk_s + grp * DS;
            float4 q_next[DS / 4], k_next[DS / 4];
            float v_next = v_s[col];
#pragma unroll
            for (int r = 0; r < DS / 4; ++r) {
                q_next[r] = reinterpret_cast<const float4*>(q_base)[r];
                k_next[r] = reinterpret_cast<const float4*>(q_base + rows)[r];
            }
            for (int t = 0; t < cn; ++t) {
                float4 q_now[DS / 4], k_now[DS / 4];
                const float vt = v_next;
#pragma unroll
                for (int r = 0; r < DS / 4; ++r) {
                    q_now[r] = q_next[r];
                    k_now[r] = k_next[r];
                }
                const int ahead_t = min(t + 1, cn - 1);  // (the last token is read twice: no condition around the reads)
                v_next = v_s[ahead_t * slice + col];
#pragma unroll
                for (int r = 0; r < DS / 4; ++r) {
                    q_next[r] = reinterpret_cast<const float4*>(q_base + ahead_t * 2 * rows)[r];
                    k_next[r] = reinterpret_cast<const float4*>(q_base + ahead_t * 2 * rows + rows)[r];
                }
                float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
#pragma unroll
                for (int r = 0; r < DS / 4; ++r) {
                    const float4 k4 = k_now[r], q4 = q_now[r];
                    S[4 * r + 0] = fmaf(fade, S[4 * r + 0], k4.x * vt);
                    S[4 * r + 1] = fmaf(fade, S[4 * r + 1], k4.y * vt);
                    S[4 * r + 2] = fmaf(fade, S[4 * r + 2], k4.z * vt);
                    S[4 * r + 3] = fmaf(fade, S[4 * r + 3], k4.w * vt);
                    a0 = fmaf(S[4 * r + 0], q4.x, a0);
                    a1 = fmaf(S[4 * r + 1], q4.y, a1);
                    a2 = fmaf(S[4 * r + 2], q4.z, a2);
                    a3 = fmaf(S[4 * r + 3], q4.w, a3);
                }
                o_s[(grp * chunk + t) * slice + col] = (a0 + a1) + (a2 + a3);
            }
        }
        __syncthreads();
        for (int idx = threadIdx.x; idx < cn * slice; idx += blockDim.x) {
            const int t = idx / slice;
            const int c = idx - t * slice;
            if (v0 + c >= vdim) continue;
            float o = 0.f;
            for (int g = 0; g < groups; ++g) o += o_s[(g * chunk + t) * slice + c];
            mine[static_cast<size_t>(first + c0 + t) * heads * vdim + head * vdim + v0 + c] = o;
        }
        __syncthreads();
    }
    if (owner)
#pragma unroll
        for (int r = 0; r < DS; ++r)
            if (d0 + r < dim) mem[static_cast<size_t>(d0 + r) * vdim] = S[r];
}
#undef CIE_RETENTION_FETCH

// (b') The same walk for sequences that bring many tokens (a prompt's portion): blocks of 32 tokens on the matrix
// cores, float32 throughout (`v_mfma_f32_16x16x4_f32`: operands and sums are plain float32), and only what has to
// wait for the block before it waits.  With S the memory in front of a block of n tokens, i and j tokens of the
// block and f the head's decay:
//     o_i   = f^(i+1) * (S^T q_i)  +  sum_{j <= i} f^(i-j) (q_i . k_j) v_j
//     S_new = f^n * S  +  sum_j f^(n-1-j) k_j v_j^T
// Three kernels.  `retention_block_sums_kernel`, every block at once: the second term of o (into the first plane of
// `raw`) and the second term of S_new (into the block's place of `sums`).  `retention_scan_kernel`, one thread per
// number of the memory, over a sequence's blocks in order: the block's place gets the S in front of it, and S moves on.
// `retention_block_reads_kernel`, every block at once: the first term of o (into the second plane).  The norm kernel
// adds the planes.  Block b of sequence s has place first_token(s) / 32 + s + b: no two blocks share one, and there
// are at most tokens / 32 + sequences + 1 places.  Queries and keys are the turn kernel's float32 rows, padded to whole
// tiles of 16; a workgroup takes up to 128 value columns (a panel), rounded up to tiles of 16 (`vdim16` columns a row
// of `sums`).  Operand layouts of the 16 x 16 x 4 product: lane (l16 = lane % 16, g = lane / 16) gives A[l16][g] and
// B[g][l16] and gets rows 4 g .. 4 g + 3 of column l16; which four numbers of a sum a product takes does not matter
// as long as both operands agree, so a lane reads four neighbouring numbers at once and spends them on four products.
typedef float acc4_t __attribute__((ext_vector_type(4)));
constexpr int kBlockTokens = 32;
constexpr int kPanelCols = 128;
constexpr int kScoreStride = kBlockTokens + 4;

// rows of a panel of values in LDS start 16 banks apart: the four tokens that a product reads then touch every bank
__host__ __device__ inline int panel_stride(int cols) { return cols % 32 == 0 ? cols + 16 : cols; }

// powers of the decay by repeated multiplication, as the walk token by token makes them
__device__ __forceinline__ void decay_table(float* pw, float fade) {
    if (threadIdx.x == 0) {
        float f = 1.0f;
        for (int n = 0; n <= kBlockTokens; ++n) {
            pw[n] = f;
            f *= fade;
        }
    }
}

// What the block kernels read from memory they ask for several loads at a time, in straight-line code that ends in a
// barrier to the compiler's scheduler: in loops of one load and its use a workgroup of four waves, two to a compute unit,
// waited for some thirty loads one after another (1,999 tokens of 8 heads of 128 x 256, us: block sums 51 -> 39, reads
// 28 -> 19).
constexpr int kStageAhead = 4;
constexpr int kStageValues = 8;

// a block's queries (side 0) or keys (side 1) into LDS rows of `stride` floats; rows past the block's last token are zero
__device__ __forceinline__ void stage_rows(float* dst, int stride, const float* __restrict__ turned, int first_token,
                                           int cn, int heads, int head, int padded, int side) {
    const int row_pieces = padded / 4, pieces = kBlockTokens * row_pieces;
    for (int base = 0; base < pieces; base += kStageAhead * 256) {
        piece_t value[kStageAhead];
#pragma unroll
        for (int i = 0; i < kStageAhead; ++i) {  // (what lies past the end reads the last piece again)
            const int idx = min(base + i * 256 + static_cast<int>(threadIdx.x), pieces - 1);
            const int t = idx / row_pieces;
            value[i] = *reinterpret_cast<const piece_t*>(
                turned + ((static_cast<size_t>(first_token + min(t, cn - 1)) * heads + head) * 2 + side) * padded +
                4 * (idx - t * row_pieces));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < kStageAhead; ++i) {  // (... and writes it again: a store under a condition takes its load along)
            const int idx = min(base + i * 256 + static_cast<int>(threadIdx.x), pieces - 1);
            const int t = idx / row_pieces;
            *reinterpret_cast<piece_t*>(dst + t * stride + 4 * (idx - t * row_pieces)) =
                t < cn ? value[i] : piece_t{0.f, 0.f, 0.f, 0.f};
        }
    }
}

template <typename T>
__global__ void __launch_bounds__(256)
retention_block_sums_kernel(const T* __restrict__ proj, long ldp, int v_off, const float* __restrict__ turned,
                            const float* __restrict__ decay, const int* __restrict__ q_start_loc,
                            float* __restrict__ raw, float* __restrict__ sums, int heads, int vdim, int padded,
                            int vdim16, int act) {
    const int seq = blockIdx.x / heads;
    const int head = blockIdx.x - seq * heads;
    const int first = q_start_loc[seq];
    const int count = q_start_loc[seq + 1] - first;
    const int c0 = blockIdx.y * kBlockTokens;
    if (c0 >= count) return;                             // (the whole workgroup: the grid is sized for the longest sequence)
    const int cn = min(kBlockTokens, count - c0);
    const int panel0 = blockIdx.z * kPanelCols;
    const int cols = min(kPanelCols, vdim16 - panel0);
    const int col_tiles = cols / 16;
    const int stride = padded + 4;
    const int vstride = panel_stride(cols);
    extern __shared__ float4 lds4[];
    float* q_s = reinterpret_cast<float*>(lds4);          // [32][stride]
    float* k_s = q_s + kBlockTokens * stride;            // [32][stride]
    float* v_s = k_s + kBlockTokens * stride;            // [32][vstride]
    float* p_s = v_s + kBlockTokens * vstride;           // [32][36]: f^(i-j) (q_i . k_j), zero above the diagonal
    float* pw = p_s + kBlockTokens * kScoreStride;       // [33]
    const int lane = threadIdx.x % kWave;
    const int wave = threadIdx.x / kWave;
    const int l16 = lane % 16;
    const int g = lane / 16;
    const int tiles = padded / 16;
    decay_table(pw, decay[head]);
    stage_rows(q_s, stride, turned, first + c0, cn, heads, head, padded, 0);
    stage_rows(k_s, stride, turned, first + c0, cn, heads, head, padded, 1);
    for (int base = 0; base < kBlockTokens * cols; base += kStageValues * 256) {
        T value[kStageValues];
#pragma unroll
        for (int i = 0; i < kStageValues; ++i) {
            const int idx = min(base + i * 256 + static_cast<int>(threadIdx.x), kBlockTokens * cols - 1);
            const int t = idx / cols;
            value[i] = proj[static_cast<size_t>(first + c0 + min(t, cn - 1)) * ldp + v_off + head * vdim +
                            min(panel0 + idx - t * cols, vdim - 1)];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < kStageValues; ++i) {
            const int idx = min(base + i * 256 + static_cast<int>(threadIdx.x), kBlockTokens * cols - 1);
            const int t = idx / cols, c = idx - t * cols;
            const float number = activated(to_float(value[i]), act);
            v_s[t * vstride + c] = (t < cn && panel0 + c < vdim) ? number : 0.f;
        }
    }
    __syncthreads();
    {   // this wave's tile of the scores (the tile above the diagonal is zero)
        const int ti = wave >> 1, tj = wave & 1;
        acc4_t p = {0.f, 0.f, 0.f, 0.f};
        if (tj <= ti) {
            const float* qa = q_s + (16 * ti + l16) * stride + 4 * g;
            const float* kb = k_s + (16 * tj + l16) * stride + 4 * g;
            acc4_t p1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
            for (int m = 0; m < tiles; ++m) {
                const float4 a = *reinterpret_cast<const float4*>(qa + 16 * m);
                const float4 b = *reinterpret_cast<const float4*>(kb + 16 * m);
                p = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, p, 0, 0, 0);
                p1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, p1, 0, 0, 0);
                p = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, p, 0, 0, 0);
                p1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, p1, 0, 0, 0);
            }
            p += p1;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int apart = 16 * (ti - tj) + 4 * g + r - l16;  // i - j
            p_s[(16 * ti + 4 * g + r) * kScoreStride + 16 * tj + l16] = apart >= 0 ? p[r] * pw[min(apart, kBlockTokens)] : 0.f;
        }
    }
    __syncthreads();
    float k_fade[kBlockTokens / 4];
#pragma unroll
    for (int kk = 0; kk < kBlockTokens / 4; ++kk) k_fade[kk] = pw[max(cn - 1 - (4 * kk + g), 0)];
    const int place = first / kBlockTokens + seq + blockIdx.y;
    float* sum_rows = sums + (static_cast<size_t>(place) * heads + head) * padded * vdim16 + panel0;
    for (int ct = wave; ct < col_tiles; ct += 4) {       // this wave's tiles of value columns
        float vb[kBlockTokens / 4];
#pragma unroll
        for (int kk = 0; kk < kBlockTokens / 4; ++kk) vb[kk] = v_s[(4 * kk + g) * vstride + 16 * ct + l16];
        // the block's own sum
        acc4_t o0 = {0.f, 0.f, 0.f, 0.f}, o1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < kBlockTokens / 4; ++kk) {
            o0 = __builtin_amdgcn_mfma_f32_16x16x4f32(p_s[l16 * kScoreStride + 4 * kk + g], vb[kk], o0, 0, 0, 0);
            o1 = __builtin_amdgcn_mfma_f32_16x16x4f32(p_s[(16 + l16) * kScoreStride + 4 * kk + g], vb[kk], o1, 0, 0, 0);
        }
        const int col = panel0 + 16 * ct + l16;
        if (col < vdim) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = 4 * g + r;
                float* dst = raw + static_cast<size_t>(first + c0) * heads * vdim + head * vdim + col;
                if (i < cn) dst[static_cast<size_t>(i) * heads * vdim] = o0[r];
                if (16 + i < cn) dst[static_cast<size_t>(16 + i) * heads * vdim] = o1[r];
            }
        }
        // what the block adds to the memory
        for (int rt = 0; rt < tiles; ++rt) {
            acc4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kk = 0; kk < kBlockTokens / 4; ++kk)
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(k_s[(4 * kk + g) * stride + 16 * rt + l16] * k_fade[kk], vb[kk],
                                                          acc, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) sum_rows[static_cast<size_t>(16 * rt + 4 * g + r) * vdim16 + 16 * ct + l16] = acc[r];
        }
    }
}

// One thread per number of a head's memory (rows and columns padded as `sums` has them): over the sequence's blocks in
// order, the block's place gets the memory in front of the block, and the memory moves on by the block's sum.
__global__ void __launch_bounds__(256)
retention_scan_kernel(const float* __restrict__ decay, float* __restrict__ state, const int* __restrict__ seq_slot,
                      const int* __restrict__ q_start_loc, float* __restrict__ sums, int heads, int dim, int vdim,
                      int padded, int vdim16) {
    const int seq = blockIdx.x / heads;
    const int head = blockIdx.x - seq * heads;
    const int e = blockIdx.y * blockDim.x + threadIdx.x;
    if (e >= padded * vdim16) return;
    const int first = q_start_loc[seq];
    const int count = q_start_loc[seq + 1] - first;
    if (count <= 0) return;
    const int row = e / vdim16;
    const int col = e - row * vdim16;
    const bool real = row < dim && col < vdim;
    float* mem = state + ((static_cast<size_t>(seq_slot[seq]) * heads + head) * dim + row) * vdim + col;
    float S = real ? *mem : 0.f;
    const int blocks = (count + kBlockTokens - 1) / kBlockTokens;
    const float fade = decay[head];
    float whole = 1.0f, rest = 1.0f;
    for (int n = 0; n < kBlockTokens; ++n) whole *= fade;
    for (int n = 0; n < count - (blocks - 1) * kBlockTokens; ++n) rest *= fade;
    const size_t step = static_cast<size_t>(heads) * padded * vdim16;
    float* at = sums + (static_cast<size_t>(first / kBlockTokens + seq) * heads + head) * padded * vdim16 + e;
    float add = at[0];
    for (int b = 0; b < blocks; ++b) {
        const float next = at[static_cast<size_t>(min(b + 1, blocks - 1)) * step];  // (asked for before this block's place is written)
        at[static_cast<size_t>(b) * step] = S;
        S = (b == blocks - 1 ? rest : whole) * S + add;
        add = next;
    }
    if (real) *mem = S;
}

__global__ void __launch_bounds__(256)
retention_block_reads_kernel(const float* __restrict__ turned, const float* __restrict__ decay,
                             const int* __restrict__ q_start_loc, const float* __restrict__ sums, float* __restrict__ raw,
                             int heads, int vdim, int padded, int vdim16) {
    const int seq = blockIdx.x / heads;
    const int head = blockIdx.x - seq * heads;
    const int first = q_start_loc[seq];
    const int count = q_start_loc[seq + 1] - first;
    const int c0 = blockIdx.y * kBlockTokens;
    if (c0 >= count) return;
    const int cn = min(kBlockTokens, count - c0);
    const int panel0 = blockIdx.z * kPanelCols;
    const int col_tiles = min(kPanelCols, vdim16 - panel0) / 16;
    const int stride = padded + 4;
    extern __shared__ float4 lds4[];
    float* q_s = reinterpret_cast<float*>(lds4);          // [32][stride]
    float* pw = q_s + kBlockTokens * stride;             // [33]
    const int lane = threadIdx.x % kWave;
    const int wave = threadIdx.x / kWave;
    const int l16 = lane % 16;
    const int g = lane / 16;
    const int tiles = padded / 16;
    decay_table(pw, decay[head]);
    stage_rows(q_s, stride, turned, first + c0, cn, heads, head, padded, 0);
    __syncthreads();
    const int place = first / kBlockTokens + seq + blockIdx.y;
    const float* before = sums + (static_cast<size_t>(place) * heads + head) * padded * vdim16 + panel0;
    for (int ct = wave; ct < col_tiles; ct += 4) {
        acc4_t o0 = {0.f, 0.f, 0.f, 0.f}, o1 = {0.f, 0.f, 0.f, 0.f};
        const float* rows = before + static_cast<size_t>(4 * g) * vdim16 + 16 * ct + l16;
        for (int m0 = 0; m0 < tiles; m0 += kStageAhead) {
            float mem[kStageAhead][4];
#pragma unroll
            for (int i = 0; i < kStageAhead; ++i)  // (a tile past the last reads the last again and is left out)
#pragma unroll
                for (int j = 0; j < 4; ++j) mem[i][j] = rows[static_cast<size_t>(16 * min(m0 + i, tiles - 1) + j) * vdim16];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < kStageAhead; ++i) {
                const bool there = m0 + i < tiles;
                const int m = min(m0 + i, tiles - 1);
                const piece_t a0 = *reinterpret_cast<const piece_t*>(q_s + l16 * stride + 16 * m + 4 * g);
                const piece_t a1 = *reinterpret_cast<const piece_t*>(q_s + (16 + l16) * stride + 16 * m + 4 * g);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float b = there ? mem[i][j] : 0.f;
                    o0 = __builtin_amdgcn_mfma_f32_16x16x4f32(there ? a0[j] : 0.f, b, o0, 0, 0, 0);
                    o1 = __builtin_amdgcn_mfma_f32_16x16x4f32(there ? a1[j] : 0.f, b, o1, 0, 0, 0);
                }
            }
        }
        const int col = panel0 + 16 * ct + l16;
        if (col < vdim) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = 4 * g + r;
                float* dst = raw + static_cast<size_t>(first + c0) * heads * vdim + head * vdim + col;
                if (i < cn) dst[static_cast<size_t>(i) * heads * vdim] = o0[r] * pw[i + 1];
                if (16 + i < cn) dst[static_cast<size_t>(16 + i) * heads * vdim] = o1[r] * pw[16 + i + 1];
            }
        }
    }
}

// o / sqrt(mean(o^2) + eps) [* weight] * gate: one wave per (token, run of `span` heads).  The mean runs over the
// `span` heads of a run together (1: every head by itself; `heads`: all of a token's heads as one vector); `weight`
// [heads * vdim] float32 or null; the gate is silu(g) (gate_act 0) or sigmoid(g) (1) of the projection's gate columns.
template <typename T>
__global__ void __launch_bounds__(256)
retention_norm_kernel(float* __restrict__ raw, long plane, int parts, const T* __restrict__ proj, long ldp, int g_off,
                      T* __restrict__ out, int tokens, int heads, int vdim, float eps, int span,
                      const float* __restrict__ weight, int gate_act) {
    const int runs = heads / span;
    const int item = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
    if (item >= tokens * runs) return;  // (whole waves leave together)
    const int lane = threadIdx.x % kWave;
    const int token = item / runs;
    const int first = (item - token * runs) * span * vdim;  // the run's first column
    const int width = span * vdim;
    float* o = raw + static_cast<size_t>(token) * heads * vdim + first;
    float sum_sq = 0.f;
    for (int c = lane; c < width; c += kWave) {
        float v = o[c];
        for (int p = 1; p < parts; ++p) v += o[static_cast<size_t>(p) * plane + c];  // (the parts in their order)
        o[c] = v;  // (this lane's own column: it reads it again below)
        sum_sq += v * v;
    }
    const float inv = 1.0f / sqrtf(wave_sum(sum_sq) / static_cast<float>(width) + eps);
    const T* gate = proj + static_cast<size_t>(token) * ldp + g_off + first;
    T* dst = out + static_cast<size_t>(token) * heads * vdim + first;
    for (int c = lane; c < width; c += kWave) {
        const float g = to_float(gate[c]);
        const float open = gate_act == 1 ? sigmoidf(g) : g * sigmoidf(g);
        float y = o[c] * inv;
        if (weight) y *= weight[first + c];
        dst[c] = from_float<T>(y * open);
    }
}

// The same for runs of up to four columns a lane: the parts' columns and the gate's are asked for together and stay in
// registers (1,999 tokens of 8 heads of 256, two parts: 12.1 us, 15.8 in the kernel above, which stores the sums and reads
// them again).
constexpr int kNormColumns = 4;

template <typename T>
__global__ void __launch_bounds__(256)
retention_norm_narrow_kernel(const float* __restrict__ raw, long plane, int parts, const T* __restrict__ proj, long ldp,
                             int g_off, T* __restrict__ out, int tokens, int heads, int vdim, float eps, int span,
                             const float* __restrict__ weight, int gate_act) {
    const int runs = heads / span;
    const int item = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
    if (item >= tokens * runs) return;  // (whole waves leave together)
    const int lane = threadIdx.x % kWave;
    const int token = item / runs;
    const int first = (item - token * runs) * span * vdim;  // the run's first column
    const int width = span * vdim;
    const float* o = raw + static_cast<size_t>(token) * heads * vdim + first;
    const T* gate = proj + static_cast<size_t>(token) * ldp + g_off + first;
    T g_in[kNormColumns];
    float v[kNormColumns] = {}, gain[kNormColumns];
#pragma unroll
    for (int i = 0; i < kNormColumns; ++i) {  // (a column past the run reads its last and counts as zero)
        const int c = min(lane + i * kWave, width - 1);
        g_in[i] = gate[c];
        gain[i] = weight ? weight[first + c] : 1.f;
    }
    for (int p0 = 0; p0 < parts; p0 += 4) {
        float piece[4][kNormColumns];
#pragma unroll
        for (int p = 0; p < 4; ++p)
#pragma unroll
            for (int i = 0; i < kNormColumns; ++i)
                piece[p][i] = o[static_cast<size_t>(min(p0 + p, parts - 1)) * plane + min(lane + i * kWave, width - 1)];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int p = 0; p < 4; ++p)
#pragma unroll
            for (int i = 0; i < kNormColumns; ++i) {  // (the parts in their order)
                const float with = p0 + p == 0 ? piece[p][i] : v[i] + piece[p][i];
                v[i] = p0 + p < parts && lane + i * kWave < width ? with : v[i];
            }
    }
    float sum_sq = 0.f;
#pragma unroll
    for (int i = 0; i < kNormColumns; ++i) sum_sq += v[i] * v[i];
    const float inv = 1.0f / sqrtf(wave_sum(sum_sq) / static_cast<float>(width) + eps);
    T* dst = out + static_cast<size_t>(token) * heads * vdim + first;
#pragma unroll
    for (int i = 0; i < kNormColumns; ++i) {
        const float g = to_float(g_in[i]);
        const float open = gate_act == 1 ? sigmoidf(g) : g * sigmoidf(g);
        float y = v[i] * inv;
        if (weight) y *= gain[i];
        if (lane + i * kWave < width) dst[lane + i * kWave] = from_float<T>(y * open);
    }
}

// The same for runs wider than a wave takes well (a norm over all heads of a token): one workgroup per (token, run),
// the summed columns wait in LDS, the waves' sums of squares meet there in the waves' order.
template <typename T>
__global__ void __launch_bounds__(1024)
retention_norm_wide_kernel(const float* __restrict__ raw, long plane, int parts, const T* __restrict__ proj, long ldp,
                           int g_off, T* __restrict__ out, int heads, int vdim, float eps, int span,
                           const float* __restrict__ weight, int gate_act) {
    extern __shared__ float wide[];  // [span * vdim] the run's columns, then one sum of squares per wave
    const int runs = heads / span;
    const int token = blockIdx.x / runs;
    const int first = (blockIdx.x - token * runs) * span * vdim;
    const int width = span * vdim;
    float* partial = wide + width;
    const float* o = raw + static_cast<size_t>(token) * heads * vdim + first;
    float sum_sq = 0.f;
    for (int c = threadIdx.x; c < width; c += blockDim.x) {
        float v = o[c];
        for (int p = 1; p < parts; ++p) v += o[static_cast<size_t>(p) * plane + c];  // (the parts in their order)
        wide[c] = v;  // (this thread's own column: it reads it again below)
        sum_sq += v * v;
    }
    sum_sq = wave_sum(sum_sq);
    if (threadIdx.x % kWave == 0) partial[threadIdx.x / kWave] = sum_sq;
    __syncthreads();
    float total = 0.f;
    for (int w = 0; w < static_cast<int>(blockDim.x) / kWave; ++w) total += partial[w];
    const float inv = 1.0f / sqrtf(total / static_cast<float>(width) + eps);
    const T* gate = proj + static_cast<size_t>(token) * ldp + g_off + first;
    T* dst = out + static_cast<size_t>(token) * heads * vdim + first;
    for (int c = threadIdx.x; c < width; c += blockDim.x) {
        const float g = to_float(gate[c]);
        const float open = gate_act == 1 ? sigmoidf(g) : g * sigmoidf(g);
        float y = wide[c] * inv;
        if (weight) y *= weight[first + c];
        dst[c] = from_float<T>(y * open);
    }
}

template <typename T, int DS>
int launch_retention(hipStream_t s, dim3 grid, int threads, size_t lds, const void* proj, long ldp, int v_off,
                     const float* turned, const float* decay, float* state, const int* seq_slot, const int* q_start_loc,
                     float* raw, long plane, int heads, int dim, int vdim, int slice, int slices, int groups, int padded,
                     int chunk, int act) {
    retention_kernel<T, DS><<<grid, threads, lds, s>>>(static_cast<const T*>(proj), ldp, v_off, turned, decay, state,
                                                      seq_slot, q_start_loc, raw, plane, heads, dim, vdim, slice, slices,
                                                      groups, padded, chunk, act);
    return cie_after_launch();
}

// (d) A step of one token a sequence: one workgroup per (sequence, head) does all of (a) to (c) at once.  Such a step reads
// and writes the memory once and has next to no arithmetic, and three launches that hand float32 rows on through memory cost
// more than that.  A thread takes four adjacent columns, 16 bytes, of kStepRows rows (a wave reads whole lines; the 4-byte
// columns of (b) cost as much as the launches from some sixteen sequences on), the row groups' shares of o meet in LDS,
// and because the workgroup has all columns of its head, the norm and the gate follow there.  What the token brings is asked
// for in front of the memory's rows: behind them it waits for them, and the gate's columns asked for at the end were another
// way to memory (7.1 us for one sequence, 10.2 for eight).  In place of the three kernels, 8 heads of 128 x 256: one
// sequence 10.8 -> 6.2 us, eight 16.2 -> 9.1 (64 workgroups; the bytes take 3.2), 64 70.1 -> 33.8 (25.8); 32 heads of
// 64 x 64: 10.3 -> 3.9, 13.4 -> 5.1, 55.2 -> 16.8.  2 or 4 rows a thread and more groups are up to 6 % faster for heads
// of 64 numbers and fewer and up to 14 % slower for larger ones of many sequences.
constexpr int kStepThreads = 1024;  // (most columns and rows of a head, too: a thread prepares one of each)
constexpr int kStepRows = 8;

template <typename T>
__global__ void __launch_bounds__(kStepThreads)
retention_step_kernel(const T* __restrict__ proj, long ldp, int q_off, int k_off, int v_off, int g_off,
                      const float* __restrict__ cos_table, const float* __restrict__ sin_table, int rot,
                      const float* __restrict__ decay, float* __restrict__ state, const int* __restrict__ seq_slot,
                      const int* __restrict__ positions, const int* __restrict__ q_start_loc, T* __restrict__ out, int heads,
                      int dim, int vdim, int quads, int groups, float eps, float key_scale, int act,
                      const float* __restrict__ weight, int gate_act) {
    extern __shared__ float4 lds4[];
    float* o_s = reinterpret_cast<float*>(lds4);  // [groups][vdim]
    float* v_s = o_s + groups * vdim;             // [vdim]
    float* q_s = v_s + vdim;                      // [dim], then the keys
    float* k_s = q_s + dim;
    float* sums = k_s + dim;                      // [waves]
    const int seq = blockIdx.x / heads;
    const int head = blockIdx.x - seq * heads;
    const int first = q_start_loc[seq];
    const int end = q_start_loc[seq + 1];
    if (end <= first) return;  // (a place without a token: the whole workgroup leaves)
    const int quad = threadIdx.x % quads;
    const int grp = threadIdx.x / quads;
    const bool owner = grp < groups;
    float* mem = state + (static_cast<size_t>(seq_slot[seq]) * heads + head) * dim * vdim + quad * 4;
    const float fade = decay[head];
    // what this thread prepares: a column's value and gate, and (from the last thread on down: where the columns leave waves
    // over, those take them) a number of the query and the key with its partner in the rotation
    const int back = blockDim.x - 1 - threadIdx.x;
    const int c = min(static_cast<int>(threadIdx.x), vdim - 1);
    const int d = min(back, dim - 1);
    const int half = rot / 2;
    const bool turns = d < rot;
    const int pair = !turns ? 0 : d < half ? d : d - half;
    const int other = !turns ? d : d < half ? d + half : pair;
    const float gain = *(weight ? weight + head * vdim + c : decay);
    const float* cos_at = turns ? cos_table : decay;  // (an address that can be read either way: loads under a condition
    const float* sin_at = turns ? sin_table : decay;  // are waited for one by one)
    T v_in, g_in, q_in, k_in, q_other, k_other;
    float c_in, s_in;
    auto fetch = [&](int t) {
        const T* row = proj + static_cast<size_t>(t) * ldp;
        const T* qh = row + q_off + head * dim;
        const T* kh = row + k_off + head * dim;
        const size_t at = turns ? static_cast<size_t>(positions[t]) * half + pair : 0;
        q_in = qh[d];
        k_in = kh[d];
        q_other = qh[other];
        k_other = kh[other];
        v_in = row[v_off + head * vdim + c];
        g_in = row[g_off + head * vdim + c];
        c_in = cos_at[at];
        s_in = sin_at[at];
    };
    fetch(first);
    // (behind the token's numbers, which are needed first and would wait for whatever was asked for before them; a row past
    // the last reads the last again)
    piece_t S[kStepRows];
#pragma unroll
    for (int r = 0; r < kStepRows; ++r)
        S[r] = *reinterpret_cast<const piece_t*>(mem + static_cast<size_t>(min(grp + r * groups, dim - 1)) * vdim);
    __builtin_amdgcn_sched_barrier(0);
    for (int t = first; t < end; ++t) {
        float qv = activated(to_float(q_in), act), kv = activated(to_float(k_in), act);
        if (turns) {
            const float q2 = activated(to_float(q_other), act), k2 = activated(to_float(k_other), act);
            qv = d < half ? qv * c_in - q2 * s_in : qv * c_in + q2 * s_in;
            kv = d < half ? kv * c_in - k2 * s_in : kv * c_in + k2 * s_in;
        }
        if (back < dim) {
            q_s[d] = qv;
            k_s[d] = kv * key_scale;
        }
        if (threadIdx.x < vdim) v_s[c] = activated(to_float(v_in), act);
        const float g = to_float(g_in);
        __syncthreads();
        if (t + 1 < end) fetch(t + 1);
        if (owner) {
            const piece_t v = *reinterpret_cast<const piece_t*>(v_s + quad * 4);
            piece_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int r = 0; r < kStepRows; ++r) {
                const int at = grp + r * groups;
                const bool live = at < dim;
                const float k = k_s[min(at, dim - 1)];
                const float q = q_s[min(at, dim - 1)];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    S[r][j] = fmaf(fade, S[r][j], k * v[j]);
                    o[j] = live ? fmaf(S[r][j], q, o[j]) : o[j];  // (a row that is not there adds nothing)
                }
            }
            *reinterpret_cast<piece_t*>(o_s + grp * vdim + quad * 4) = o;
        }
        __syncthreads();
        float o = 0.f;
        if (threadIdx.x < vdim)
#pragma unroll 8
            for (int i = 0; i < groups; ++i) o += o_s[i * vdim + c];  // (the groups in their order)
        const float wave_sq = wave_sum(o * o);
        if (threadIdx.x % kWave == 0) sums[threadIdx.x / kWave] = wave_sq;
        __syncthreads();
        if (threadIdx.x < vdim) {
            float sum_sq = 0.f;
            for (int w = 0; w * kWave < vdim; ++w) sum_sq += sums[w];
            const float inv = 1.0f / sqrtf(sum_sq / static_cast<float>(vdim) + eps);
            const float open = gate_act == 1 ? sigmoidf(g) : g * sigmoidf(g);
            float y = o * inv;
            if (weight) y *= gain;
            out[(static_cast<size_t>(t) * heads + head) * vdim + c] = from_float<T>(y * open);
        }
        // (the next token's numbers go where none but the threads before the second barrier read; `sums` is written behind
        // two more)
    }
    if (owner)
#pragma unroll
        for (int r = 0; r < kStepRows; ++r)
            if (grp + r * groups < dim) *reinterpret_cast<piece_t*>(mem + static_cast<size_t>(grp + r * groups) * vdim) = S[r];
}

// ---------------------------------------------------------------------------------------------- convolution
// (`act`: what the sum passes through, 0 nothing, 1 silu; O: the type it is stored in)
template <typename T, typename O>
__global__ void __launch_bounds__(256)
causal_conv_kernel(const T* __restrict__ x, long ldx, const T* __restrict__ taps_w, const T* __restrict__ bias,
                   const float* __restrict__ past, const int* __restrict__ seq_of_token, const int* __restrict__ seq_slot,
                   const int* __restrict__ q_start_loc, O* __restrict__ out, int channels, int taps, int act) {
    const int token = blockIdx.y;
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= channels) return;
    const int seq = seq_of_token[token];
    const int first = q_start_loc[seq];
    const int t = token - first;
    const float* before = past + static_cast<size_t>(seq_slot[seq]) * max(taps - 1, 1) * channels;
    float acc = 0.f;
    for (int j = 0; j < taps; ++j) {
        const int src = t - (taps - 1) + j;  // the last tap is this token's input
        const float in = src >= 0 ? to_float(x[static_cast<size_t>(first + src) * ldx + c])
                                  : before[static_cast<size_t>(taps - 1 + src) * channels + c];
        acc = fmaf(to_float(taps_w[static_cast<size_t>(c) * taps + j]), in, acc);
    }
    if (bias) acc += to_float(bias[c]);
    out[static_cast<size_t>(token) * channels + c] = from_float<O>(activated(acc, act));
}

// Four taps over 16-bit inputs, eight channels and kTokens neighbouring tokens a thread: the inputs, the weights (eight
// channels' four stand side by side: four pieces of 16 bytes) and the outputs move in 16-byte pieces, a thread's tokens
// share weights and inputs, and the sums are the ones above, in their order.  The kernel above reads two bytes at a time
// and a channel's weights eight bytes apart.  What bounds it is the chain of a thread's loads: the inputs do not wait for
// the token's sequence, only what the state holds for a sequence's first three tokens does.  1,999 tokens of 2,048 channels:
// 22.6 -> 8.5 us, 8 tokens 4.8 as before.
typedef uint32_t words_t __attribute__((ext_vector_type(4)));  // eight 16-bit numbers

__device__ __forceinline__ words_t load_words(const bf16_t* p) { return *reinterpret_cast<const words_t*>(p); }
__device__ __forceinline__ float number(words_t w, int i) {
    return __uint_as_float(i % 2 ? w[i / 2] & 0xffff0000u : w[i / 2] << 16);
}

template <typename O, int kTokens>
__global__ void __launch_bounds__(256)
causal_conv4_vec8_kernel(const bf16_t* __restrict__ x, long ldx, const bf16_t* __restrict__ taps_w,
                         const bf16_t* __restrict__ bias, const float* __restrict__ past,
                         const int* __restrict__ seq_of_token, const int* __restrict__ seq_slot,
                         const int* __restrict__ q_start_loc, O* __restrict__ out, int tokens, int channels, int act) {
    constexpr int kTaps = 4;
    const int per_token = channels / 8;
    const long item = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
    const int token0 = static_cast<int>(item / per_token) * kTokens;
    if (token0 >= tokens) return;
    const int c = static_cast<int>(item % per_token) * 8;
    words_t in[kTokens + kTaps - 1], w[kTaps], b = {};
    int seq[kTokens];
#pragma unroll
    for (int i = 0; i < kTokens; ++i) seq[i] = seq_of_token[min(token0 + i, tokens - 1)];
#pragma unroll
    for (int j = 0; j < kTokens + kTaps - 1; ++j)  // (rows outside the step are clamped, and used for no token)
        in[j] = load_words(x + static_cast<size_t>(max(0, min(token0 - (kTaps - 1) + j, tokens - 1))) * ldx + c);
#pragma unroll
    for (int i = 0; i < kTaps; ++i) w[i] = load_words(taps_w + static_cast<size_t>(c) * kTaps + 8 * i);
    if (bias) b = load_words(bias + c);
#pragma unroll
    for (int i = 0; i < kTokens; ++i) {
        const int token = token0 + i;
        if (token >= tokens) break;
        const int t = token - q_start_loc[seq[i]];
        float acc[8] = {};
        if (t >= kTaps - 1) {
#pragma unroll
            for (int j = 0; j < kTaps; ++j)
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    acc[e] = fmaf(number(w[(kTaps * e + j) / 8], (kTaps * e + j) % 8), number(in[i + j], e), acc[e]);
        } else {
            const float* before = past + static_cast<size_t>(seq_slot[seq[i]]) * (kTaps - 1) * channels + c;
            piece_t held[kTaps - 1][2];  // (all of them, at once; the rows that the step itself brings are not used)
#pragma unroll
            for (int j = 0; j < kTaps - 1; ++j) {
                const float* src = before + static_cast<size_t>(min(max(j + t, 0), kTaps - 2)) * channels;
                held[j][0] = reinterpret_cast<const piece_t*>(src)[0];
                held[j][1] = reinterpret_cast<const piece_t*>(src)[1];
            }
#pragma unroll
            for (int j = 0; j < kTaps; ++j)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    float v = number(in[i + j], e);
                    if (j < kTaps - 1) v = t - (kTaps - 1) + j < 0 ? held[j < kTaps - 1 ? j : 0][e / 4][e % 4] : v;
                    acc[e] = fmaf(number(w[(kTaps * e + j) / 8], (kTaps * e + j) % 8), v, acc[e]);
                }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = activated(bias ? acc[e] + number(b, e) : acc[e], act);
        O* dst = out + static_cast<size_t>(token) * channels + c;
        if constexpr (sizeof(O) == 2) {
            *reinterpret_cast<words_t*>(dst) = words_t{pack_bf16(acc[0], acc[1]), pack_bf16(acc[2], acc[3]),
                                                       pack_bf16(acc[4], acc[5]), pack_bf16(acc[6], acc[7])};
        } else {
            *reinterpret_cast<piece_t*>(dst) = piece_t{acc[0], acc[1], acc[2], acc[3]};
            *reinterpret_cast<piece_t*>(dst + 4) = piece_t{acc[4], acc[5], acc[6], acc[7]};
        }
    }
}

// The convolution's state moved on by a step's inputs: of [what the state held, the step's inputs] the last
// taps - 1 rows.  One thread per (sequence, channel); runs behind the convolution that still read the old rows.
template <typename T>
__global__ void __launch_bounds__(256)
conv_keep_kernel(const T* __restrict__ x, long ldx, float* __restrict__ past, const int* __restrict__ seq_slot,
                 const int* __restrict__ q_start_loc, int channels, int taps) {
    const int seq = blockIdx.y;
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    const int keep_n = taps - 1;
    if (c >= channels || keep_n <= 0) return;
    const int first = q_start_loc[seq];
    const int count = q_start_loc[seq + 1] - first;
    float* before = past + static_cast<size_t>(seq_slot[seq]) * keep_n * channels;
    float old[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) old[j] = j < keep_n ? before[static_cast<size_t>(j) * channels + c] : 0.f;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        if (j >= keep_n) break;
        const int src = count + j;  // index into [old (keep_n), new (count)]
        before[static_cast<size_t>(j) * channels + c] =
            src < keep_n ? old[src < 16 ? src : 0] : to_float(x[static_cast<size_t>(first + src - keep_n) * ldx + c]);
    }
}

// ---------------------------------------------------------------------------------------------- gated recurrence
// a_t and x_t of one token and channel, from what stands in memory for them
struct GateStep {
    float a, x;
};

__device__ __forceinline__ GateStep gate_step(float r_pre, float i_pre, float u, float coef) {
    const float log_a = coef * sigmoidf(r_pre);
    return {expf(log_a), sqrtf(-expm1f(2.0f * log_a)) * (sigmoidf(i_pre) * u)};  // sqrt(1 - a^2), no cancellation
}

constexpr int kMaxTaps = 16;

// the convolution's last taps - 1 inputs: those of this step, and behind them what the state held
template <typename T>
__device__ __forceinline__ void keep_inputs(float* before, const T* __restrict__ x_in, long ldx, int first, int count,
                                            int c, int channels, int keep_n) {
    float old[kMaxTaps];
#pragma unroll
    for (int j = 0; j < kMaxTaps; ++j) old[j] = j < keep_n ? before[static_cast<size_t>(j) * channels + c] : 0.f;
#pragma unroll
    for (int j = 0; j < kMaxTaps; ++j) {
        if (j >= keep_n) break;
        const int src = count + j;  // index into [old (keep_n), new (count)]
        before[static_cast<size_t>(j) * channels + c] =
            src < keep_n ? old[src < kMaxTaps ? src : 0] : to_float(x_in[static_cast<size_t>(first + src - keep_n) * ldx + c]);
    }
}

// The walk in order (decode steps, short portions): one thread per (sequence, channel), 64 channels a workgroup.
template <typename T>
__global__ void __launch_bounds__(64)
gated_recurrence_kernel(const T* __restrict__ y_pre, long ldy, const T* __restrict__ x_in, long ldx,
                        const T* __restrict__ u, const float* __restrict__ gates, int block_width,
                        const float* __restrict__ rate, float* __restrict__ state, float* __restrict__ past,
                        const int* __restrict__ seq_slot, const int* __restrict__ q_start_loc, T* __restrict__ out,
                        int channels, int taps) {
    const int seq = blockIdx.y;
    const int c = blockIdx.x * 64 + threadIdx.x;
    if (c >= channels) return;
    const int first = q_start_loc[seq];
    const int count = q_start_loc[seq + 1] - first;
    const int slot = seq_slot[seq];
    const int block = c / block_width;
    const size_t r_at = static_cast<size_t>(block) * 2 * block_width + (c - block * block_width);
    const size_t i_at = r_at + block_width;
    const float coef = rate[c];
    float S = state[static_cast<size_t>(slot) * channels + c];
#pragma unroll 4
    for (int t = 0; t < count; ++t) {  // (four tokens per turn: their loads travel together)
        const size_t token = static_cast<size_t>(first + t);
        const GateStep now = gate_step(gates[token * 2 * channels + r_at], gates[token * 2 * channels + i_at],
                                       to_float(u[token * channels + c]), coef);
        S = fmaf(now.a, S, now.x);
        out[token * channels + c] = from_float<T>(S * gelu_tanh(to_float(y_pre[token * ldy + c])));
    }
    state[static_cast<size_t>(slot) * channels + c] = S;
    if (taps > 1)
        keep_inputs(past + static_cast<size_t>(slot) * (taps - 1) * channels, x_in, ldx, first, count, c, channels, taps - 1);
}

// A step in which no sequence brings more than one token, in bfloat16: the gates' block-diagonal product and the walk's one
// step at once.  A workgroup owns 16 channels of 16 sequences.  Its four waves take every fourth slice of 32 k of both gates
// (v_mfma_f32_16x16x32_bf16), the sums meet in LDS in the waves' order, and every thread then moves the state of one channel
// and sequence: the float32 gates never go through memory and a launch falls away.  What bounds it are chains, not bytes (a
// layer's gates are 2 MB): a wave's slices and what the step itself needs are all asked for before the first product,
// and a lane of one wave that moved the four states whose gates it held spent 0.65 us on each, one after the other.
// In place of the product and the walk, 8 blocks of 256: one sequence 6.6 -> 4.2 us, eight 7.2 -> 4.3, 64 11.4 -> 6.5.  From
// four to six workgroups a unit on, by the blocks' width, every 16 sequences' new reading of the weights costs more than the launch
// (16 blocks of 256, 128 sequences 15.9 -> 16.9; at five a unit 14.0 -> 13.2; 20 blocks of 128 11.7 -> 13.5): kernels/ops.py
// draws the line.
typedef __bf16 gate_piece_t __attribute__((ext_vector_type(8)));
constexpr int kGateSlices = 4;  // of 32 k under way at once, a wave
constexpr int kStepTaps = 4;    // inputs kept beside the token's own, at most (longer convolutions take the general path)

__global__ void __launch_bounds__(256)
gated_recurrence_step_kernel(const bf16_t* __restrict__ y_pre, long ldy, const bf16_t* __restrict__ x_in, long ldx,
                             const bf16_t* __restrict__ u, const bf16_t* __restrict__ weight, const bf16_t* __restrict__ bias,
                             int block_width, int tiles, const float* __restrict__ rate, float* __restrict__ state,
                             float* __restrict__ past, const int* __restrict__ seq_slot, const int* __restrict__ q_start_loc,
                             bf16_t* __restrict__ out, int sequences, int tokens, int channels, int keep_n) {
    __shared__ float sums[4][2][16][17];  // [wave][gate][sequence][channel]
    const int lane = threadIdx.x % kWave;
    const int wave = threadIdx.x / kWave;
    const int r = lane & 15;
    const int g = lane >> 4;
    const int groups = gridDim.x;  // (neighbouring channels on one XCD, whose L2 then holds a line's both halves and a block's rows)
    const int group = groups % 8 == 0 ? (blockIdx.x % 8) * (groups / 8) + blockIdx.x / 8 : blockIdx.x;
    const int block = group / tiles;
    const int n0 = (group - block * tiles) * 16;
    const int seq0 = blockIdx.y * 16;
    // (a channel past the block's last reads the last, a sequence past the last too; a place without a token reads some token
    // and stores nothing)
    const int n = min(n0 + r, block_width - 1);
    const bf16_t* a_row = u + static_cast<size_t>(min(q_start_loc[min(seq0 + r, sequences - 1)], tokens - 1)) * channels +
                          static_cast<size_t>(block) * block_width;
    const bf16_t* r_row = weight + (static_cast<size_t>(block) * 2 * block_width + n) * block_width;
    const bf16_t* i_row = r_row + static_cast<size_t>(block_width) * block_width;
    words_t av[kGateSlices], rv[kGateSlices], iv[kGateSlices];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int s = 0; s < kGateSlices; ++s) {
            const int at = min(k0 + 32 * (4 * s + wave) + g * 8, block_width - 8);
            rv[s] = *reinterpret_cast<const words_t*>(r_row + at);
            iv[s] = *reinterpret_cast<const words_t*>(i_row + at);
            av[s] = *reinterpret_cast<const words_t*>(a_row + at);
        }
    };
    fetch(0);
    // the step's own: one channel of one sequence a thread
    const int mine = threadIdx.x / 16;
    const int col = threadIdx.x % 16;
    const int seq = min(seq0 + mine, sequences - 1);
    const int inside = min(n0 + col, block_width - 1);
    const int c = block * block_width + inside;
    const int start = q_start_loc[seq];
    const bool steps = n0 + col < block_width && seq0 + mine < sequences && q_start_loc[seq + 1] > start;
    const size_t token = static_cast<size_t>(min(start, tokens - 1));
    const size_t slot = static_cast<size_t>(seq_slot[seq]);
    const bf16_t* b_row = bias + static_cast<size_t>(block) * 2 * block_width + inside;
    const bf16_t r_bias = b_row[0], i_bias = b_row[block_width];
    const float coef = rate[c];
    const float S = state[slot * channels + c];
    const bf16_t y_in = y_pre[token * ldy + c], u_in = u[token * channels + c], x_new = x_in[token * ldx + c];
    float* before = past + slot * max(keep_n, 1) * channels + c;
    float old[kStepTaps];
#pragma unroll
    for (int j = 0; j < kStepTaps; ++j) old[j] = before[static_cast<size_t>(min(j, max(keep_n - 1, 0))) * channels];
    __builtin_amdgcn_sched_barrier(0);
    acc4_t r_sum = {0.f, 0.f, 0.f, 0.f}, i_sum = {0.f, 0.f, 0.f, 0.f};
    const words_t nothing = {0u, 0u, 0u, 0u};
    for (int k0 = 0; k0 < block_width; k0 += 4 * 32 * kGateSlices) {
        if (k0 > 0) fetch(k0);
#pragma unroll
        for (int s = 0; s < kGateSlices; ++s) {
            // (a group of 8 past the end read the last group again and counts as zeros, on both sides)
            const bool there = k0 + 32 * (4 * s + wave) + g * 8 < block_width;
            const gate_piece_t a = __builtin_bit_cast(gate_piece_t, there ? av[s] : nothing);
            r_sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(gate_piece_t, there ? rv[s] : nothing), r_sum, 0, 0, 0);
            i_sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(gate_piece_t, there ? iv[s] : nothing), i_sum, 0, 0, 0);
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        sums[wave][0][g * 4 + i][r] = r_sum[i];
        sums[wave][1][g * 4 + i][r] = i_sum[i];
    }
    __syncthreads();
    if (!steps) return;
    float r_pre = sums[0][0][mine][col], i_pre = sums[0][1][mine][col];
#pragma unroll
    for (int w = 1; w < 4; ++w) {
        r_pre += sums[w][0][mine][col];
        i_pre += sums[w][1][mine][col];
    }
    const GateStep now = gate_step(r_pre + to_float(r_bias), i_pre + to_float(i_bias), to_float(u_in), coef);
    const float next = fmaf(now.a, S, now.x);
    out[token * channels + c] = from_float<bf16_t>(next * gelu_tanh(to_float(y_in)));
    state[slot * channels + c] = next;
#pragma unroll
    for (int j = 0; j < kStepTaps; ++j)
        if (j < keep_n) before[static_cast<size_t>(j) * channels] = j + 1 < keep_n ? old[j + 1 < kStepTaps ? j + 1 : j] : to_float(x_new);
}

// Prompts' portions in bfloat16, whatever their number: the gates' block-diagonal product and the walk over the step's flat tokens
// at once, in chunks of 64 tokens whose first token may be a sequence's or not.  (a) A workgroup owns 64 channels of a chunk: the
// chunk's rows of the block's channels lie in LDS, a wave has its 16 channels' rows of both gates' weights in registers, and the
// product comes out with a token a lane and four channels each, so that everything behind it moves in 16-byte pieces.  The walk
// is linear in S, S_t = a_t S_(t-1) + x_t, and composed in the registers: 16 lanes' tokens by doubling, four such runs one after the
// other.  (A, B) of every token, its state as A * (the state in front of the chunk) + B, go to memory, and the chunk's last pair
// beside them.  A sequence's first token takes its slot's state in: A = 0 from there on.  (b) Every workgroup joins the chunks in front
// of its own and makes the outputs; the token that ends a sequence writes the states.
//
// What bounds it: the way to memory, 16 bytes a token and channel between the two where the gates took as many, and the gates' five
// transcendental functions (some 3,000 of a wave's instructions: 21 of (a)'s 30 us at 1,999 tokens of 2,048 channels; (b) 15.6).  In
// place of the product, whose waves each fetched the same rows, and of a walk of 32 tokens a thread, 16 neighbouring channels a row: 87
// -> 45 us there, 579 tokens of eight sequences 32.6 -> 25.5.  (b) also moves the convolutions' states, a workgroup a sequence behind its
// tokens': done by the threads of a sequence's last token this took 8 us.
constexpr int kChunkTokens = 64;
constexpr int kChunkChannels = 64;
constexpr int kOutputTokens = 32;  // of a workgroup of (b)

// The value of the lane APART in front, of a row of 16 (the first ones have `first`, or keep theirs), and that of a row's last lane.
template <int APART>
__device__ __forceinline__ float lane_before(float v, float first) {
    return __uint_as_float(static_cast<uint32_t>(__builtin_amdgcn_update_dpp(
        static_cast<int>(__float_as_uint(first)), static_cast<int>(__float_as_uint(v)), 0x110 + APART, 0xf, 0xf, false)));
}
template <int APART>
__device__ __forceinline__ float lane_before(float v) {
    return lane_before<APART>(v, v);
}
__device__ __forceinline__ float row_last(float v) {
    const int own = static_cast<int>(__float_as_uint(v));
    return __uint_as_float(static_cast<uint32_t>(__builtin_amdgcn_update_dpp(own, own, 0x15f, 0xf, 0xf, false)));
}

// One doubling of the walk over a row's 16 tokens: what the tokens APART in front made joins, unless a sequence begins between.
template <int APART>
__device__ __forceinline__ void join_before(float (&a)[4], float (&b)[4], int r, int from, int place) {
    const bool joins = r >= APART && from <= place - APART;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float pa = lane_before<APART>(a[i]), pb = lane_before<APART>(b[i]);
        b[i] = joins ? fmaf(a[i], pb, b[i]) : b[i];
        a[i] = joins ? a[i] * pa : a[i];
    }
}

template <int BW>
__global__ void __launch_bounds__(256, 4)
gated_chunks_kernel(const bf16_t* __restrict__ u, const bf16_t* __restrict__ weight, const bf16_t* __restrict__ bias,
                    const float* __restrict__ rate, const float* __restrict__ state, const int* __restrict__ seq_of_token,
                    const int* __restrict__ seq_slot, const int* __restrict__ q_start_loc, float* __restrict__ plane_a,
                    float* __restrict__ plane_b, float* __restrict__ carry, int tokens, int channels, int chunks) {
    constexpr int kSlices = BW / 32;
    constexpr int kRowBytes = BW * 2 + 16;  // the padding spreads the rows over the banks
    constexpr int kTiles = kChunkTokens / 16;
    __shared__ __attribute__((aligned(16))) char rows[kChunkTokens * kRowBytes];
    // where a token's sequence begins, counted from the chunk's first token: what lies in front of it is never multiplied with what
    // lies behind (its state may be infinite); the sequence's slot, if the token is its first, -1 for any other, -2 past the last
    __shared__ int begins[kChunkTokens], first_slot[kChunkTokens];
    const int lane = threadIdx.x % kWave;
    const int wave = threadIdx.x / kWave;
    const int r = lane & 15;
    const int g = lane >> 4;
    constexpr int kGroups = BW / kChunkChannels;
    const int blocks = channels / BW, per = chunks * kGroups;
    // (a block's rows and weights stay on one XCD where the blocks can be dealt out so)
    const int own = blocks % 8 == 0 ? blockIdx.x / 8 : blockIdx.x;
    const int block = blocks % 8 == 0 ? blockIdx.x % 8 + 8 * (own / per) : own / per;
    const int chunk = own % per / kGroups;
    const int n0 = own % kGroups * kChunkChannels + wave * 16;  // the wave's channels in the block
    const int t0 = chunk * kChunkTokens;

    words_t wr[kSlices], wi[kSlices], piece[kSlices];
    const bf16_t* w_row = weight + (static_cast<size_t>(block) * 2 * BW + n0 + r) * BW + g * 8;
    constexpr int kPieces = BW / 8;  // of 16 bytes, of a token's row
#pragma unroll
    for (int s = 0; s < kSlices; ++s) {
        const int at = threadIdx.x + s * 256;
        piece[s] = load_words(u + static_cast<size_t>(min(t0 + at / kPieces, tokens - 1)) * channels + block * BW + at % kPieces * 8);
    }
#pragma unroll
    for (int s = 0; s < kSlices; ++s) {
        wr[s] = load_words(w_row + s * 32);
        wi[s] = load_words(w_row + static_cast<size_t>(BW) * BW + s * 32);
    }
    const int c = block * BW + n0 + g * 4;  // the lane's first channel
    const piece_t coef = *reinterpret_cast<const piece_t*>(rate + c);
    float r_bias[4], i_bias[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        r_bias[i] = to_float(bias[static_cast<size_t>(block) * 2 * BW + n0 + g * 4 + i]);
        i_bias[i] = to_float(bias[static_cast<size_t>(block) * 2 * BW + BW + n0 + g * 4 + i]);
    }
    if (threadIdx.x < kChunkTokens) {
        const int t = t0 + threadIdx.x;
        const int seq = seq_of_token[min(t, tokens - 1)];
        const int first = q_start_loc[seq];
        begins[threadIdx.x] = first - t0;
        first_slot[threadIdx.x] = t >= tokens ? -2 : first == t ? seq_slot[seq] : -1;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < kSlices; ++s) {
        const int at = threadIdx.x + s * 256;
        *reinterpret_cast<words_t*>(rows + at / kPieces * kRowBytes + at % kPieces * 16) = piece[s];
    }
    __syncthreads();
    acc4_t r_sum[kTiles], i_sum[kTiles];
#pragma unroll
    for (int t = 0; t < kTiles; ++t) r_sum[t] = i_sum[t] = acc4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < kSlices; ++s)
#pragma unroll
        for (int t = 0; t < kTiles; ++t) {
            const gate_piece_t row = __builtin_bit_cast(gate_piece_t, *reinterpret_cast<const words_t*>(rows + (t * 16 + r) * kRowBytes + s * 64 + g * 16));
            r_sum[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gate_piece_t, wr[s]), row, r_sum[t], 0, 0, 0);
            i_sum[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gate_piece_t, wi[s]), row, i_sum[t], 0, 0, 0);
        }
    float before_a[4], before_b[4];  // all tokens of the chunk in front of the tile
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        before_a[i] = 1.f;
        before_b[i] = 0.f;
    }
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
        const int place = t * 16 + r;
        const int slot = first_slot[place], from = begins[place];
        const uint2 own_u = *reinterpret_cast<const uint2*>(rows + place * kRowBytes + (n0 + g * 4) * 2);
        const float u_in[4] = {__uint_as_float(own_u.x << 16), __uint_as_float(own_u.x & 0xffff0000u),
                               __uint_as_float(own_u.y << 16), __uint_as_float(own_u.y & 0xffff0000u)};
        float a[4], b[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const GateStep now = gate_step(r_sum[t][i] + r_bias[i], i_sum[t][i] + i_bias[i], u_in[i], coef[i]);
            a[i] = slot == -2 ? 1.f : now.a;
            b[i] = slot == -2 ? 0.f : now.x;
        }
        if (slot >= 0) {
            const piece_t S = *reinterpret_cast<const piece_t*>(state + static_cast<size_t>(slot) * channels + c);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                b[i] = fmaf(a[i], S[i], b[i]);
                a[i] = 0.f;
            }
        }
        const float own_a[4] = {a[0], a[1], a[2], a[3]}, own_b[4] = {b[0], b[1], b[2], b[3]};
        join_before<1>(a, b, r, from, place);
        join_before<2>(a, b, r, from, place);
        join_before<4>(a, b, r, from, place);
        join_before<8>(a, b, r, from, place);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const bool joins = from < t * 16;
            b[i] = joins ? fmaf(a[i], before_b[i], b[i]) : b[i];
            a[i] = joins ? a[i] * before_a[i] : a[i];
            // Up to six roundings by now: the step over again from the token in front has the walk's one, and fades what the tokens
            // in front have of them, twice (states off 64 bits by 7.9e-8 without, 7.2e-8 so, 7.1e-8 in order; 1,999 tokens of 2,048
            // channels 43.9 -> 44.7 us).
            const bool steps = from < place && place > 0;
#pragma unroll
            for (int again = 0; again < 2; ++again) {
                const float in_front = lane_before<1>(b[i], before_b[i]);
                b[i] = steps ? fmaf(own_a[i], in_front, own_b[i]) : b[i];
            }
            before_a[i] = row_last(a[i]);
            before_b[i] = row_last(b[i]);
        }
        if (t0 + place < tokens) {
            const size_t at = static_cast<size_t>(t0 + place) * channels + c;
            *reinterpret_cast<piece_t*>(plane_a + at) = piece_t{a[0], a[1], a[2], a[3]};
            *reinterpret_cast<piece_t*>(plane_b + at) = piece_t{b[0], b[1], b[2], b[3]};
        }
    }
    if (r == 15) {
        float* to = carry + static_cast<size_t>(chunk) * 2 * channels + c;
        *reinterpret_cast<piece_t*>(to) = piece_t{before_a[0], before_a[1], before_a[2], before_a[3]};
        *reinterpret_cast<piece_t*>(to + channels) = piece_t{before_b[0], before_b[1], before_b[2], before_b[3]};
    }
}

__global__ void __launch_bounds__(256)
gated_outputs_kernel(const bf16_t* __restrict__ y_pre, long ldy, const bf16_t* __restrict__ x_in, long ldx,
                     const float* __restrict__ plane_a, const float* __restrict__ plane_b, const float* __restrict__ carry,
                     float* __restrict__ state, float* __restrict__ past, const int* __restrict__ seq_of_token,
                     const int* __restrict__ seq_slot, const int* __restrict__ q_start_loc, bf16_t* __restrict__ out, int tokens,
                     int channels, int keep_n, int token_groups) {
    __shared__ float start[256];  // the channels' states in front of the chunk
    // (one grid dimension: portions and sequences together may be more than the others hold)
    const int channel_groups = (channels + 255) / 256;
    const int c0 = blockIdx.x % channel_groups * 256, place = blockIdx.x / channel_groups;
    if (place >= token_groups) {  // behind the tokens: a sequence's inputs, a channel a thread
        const int keeps = place - token_groups, own = c0 + threadIdx.x;
        if (own < channels)
            keep_inputs(past + static_cast<size_t>(seq_slot[keeps]) * keep_n * channels, x_in, ldx, q_start_loc[keeps],
                        q_start_loc[keeps + 1] - q_start_loc[keeps], own, channels, keep_n);
        return;
    }
    const int t0 = place * kOutputTokens;
    const int chunk = t0 / kChunkTokens;
    const int c = c0 + threadIdx.x % 32 * 8;
    const int cc = min(c, channels - 8);  // (a thread past the last channel reads and stores nothing of its own)
    constexpr int kTurns = kOutputTokens / 8;
    piece_t a[kTurns][2], b[kTurns][2];
    words_t y[kTurns];
    int seq[kTurns];
#pragma unroll
    for (int i = 0; i < kTurns; ++i) {
        const int t = min(t0 + i * 8 + static_cast<int>(threadIdx.x) / 32, tokens - 1);
        const size_t at = static_cast<size_t>(t) * channels + cc;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            a[i][h] = *reinterpret_cast<const piece_t*>(plane_a + at + 4 * h);
            b[i][h] = *reinterpret_cast<const piece_t*>(plane_b + at + 4 * h);
        }
        y[i] = load_words(y_pre + static_cast<size_t>(t) * ldy + cc);
        seq[i] = seq_of_token[t];
    }
    {
        const int own = min(c0 + static_cast<int>(threadIdx.x), channels - 1);
        const int from = q_start_loc[seq_of_token[chunk * kChunkTokens]] / kChunkTokens;
        float S = 0.f;  // (the first of these chunks holds its sequence's first token: its A is 0)
        for (int k0 = from; k0 < chunk; k0 += 8) {
            float ka[8], kb[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const float* pair = carry + static_cast<size_t>(min(k0 + k, chunk - 1)) * 2 * channels + own;
                ka[k] = pair[0];
                kb[k] = pair[channels];
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) S = k0 + k < chunk ? fmaf(ka[k], S, kb[k]) : S;
        }
        start[threadIdx.x] = S;
    }
    __syncthreads();
    if (c >= channels) return;
    float S0[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) S0[e] = start[c - c0 + e];
#pragma unroll
    for (int i = 0; i < kTurns; ++i) {
        const int t = t0 + i * 8 + static_cast<int>(threadIdx.x) / 32;
        if (t >= tokens) break;
        const int first = q_start_loc[seq[i]];
        const bool joins = first < chunk * kChunkTokens;  // (its sequence does not begin in this chunk)
        float S[8], o[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float with = fmaf(a[i][e / 4][e % 4], S0[e], b[i][e / 4][e % 4]);
            S[e] = joins ? with : b[i][e / 4][e % 4];
            o[e] = S[e] * gelu_tanh(number(y[i], e));
        }
        *reinterpret_cast<words_t*>(out + static_cast<size_t>(t) * channels + c) =
            words_t{pack_bf16(o[0], o[1]), pack_bf16(o[2], o[3]), pack_bf16(o[4], o[5]), pack_bf16(o[6], o[7])};
        if (q_start_loc[seq[i] + 1] != t + 1) continue;
        const int slot = seq_slot[seq[i]];  // the sequence ends here: its states
        float* to = state + static_cast<size_t>(slot) * channels + c;
        *reinterpret_cast<piece_t*>(to) = piece_t{S[0], S[1], S[2], S[3]};
        *reinterpret_cast<piece_t*>(to + 4) = piece_t{S[4], S[5], S[6], S[7]};
    }
}

// Long portions.  S_t = a_t S_(t-1) + x_t is linear in S, so `segments` stretches of up to 32 tokens run side by side:
// thread (channel, stretch) folds its stretch into (A, B) with S_out = A S_in + B, the stretches before it give its
// S_in (a chain of at most `segments` multiply-adds), and a second walk makes the outputs.  A portion of more than
// segments * 32 tokens goes in rounds of that many.
//
// What bounds it is the way to memory: 14 bytes a token and channel, and a thread that waits for one token's loads at a
// time waits some hundred times.  So a stretch is short, its a_t and x_t stay in registers between the walks (no second
// read, no second exponential and root), and four tokens' loads travel together.  16 channels a workgroup, and
// neighbouring workgroups' channels on one XCD, whose L2 then serves both halves of a 128-byte line.  1,999 tokens of 2,048
// channels: 107 us in 16 stretches that were read twice, 44 in 64 stretches (16 us is the memory's part).
constexpr int kMaxSegments = 64;
constexpr int kScanChannels = 16;
constexpr int kScanTokens = 32;  // of a stretch: 64 registers of the 128 that 1,024 threads leave a thread
constexpr int kScanAhead = 4;

template <typename T>
__global__ void __launch_bounds__(kScanChannels * kMaxSegments)
gated_recurrence_stretches_kernel(const T* __restrict__ y_pre, long ldy, const T* __restrict__ x_in, long ldx,
                                  const T* __restrict__ u, const float* __restrict__ gates, int block_width,
                                  const float* __restrict__ rate, float* __restrict__ state, float* __restrict__ past,
                                  const int* __restrict__ seq_slot, const int* __restrict__ q_start_loc,
                                  T* __restrict__ out, int channels, int taps, int segments) {
    __shared__ float a_s[kMaxSegments][kScanChannels];
    __shared__ float b_s[kMaxSegments][kScanChannels];
    const int seq = blockIdx.y;
    const int lane = threadIdx.x % kScanChannels;
    const int seg = threadIdx.x / kScanChannels;
    const int groups = gridDim.x;
    const int group = groups % 8 == 0 ? (blockIdx.x % 8) * (groups / 8) + blockIdx.x / 8 : blockIdx.x;
    const int c = group * kScanChannels + lane;
    const bool live = c < channels;
    const int ch = min(c, channels - 1);  // (a thread past the last channel walks along and stores nothing)
    const int first = q_start_loc[seq];
    const int count = q_start_loc[seq + 1] - first;
    const int slot = seq_slot[seq];
    const int block = ch / block_width;
    const size_t r_at = static_cast<size_t>(block) * 2 * block_width + (ch - block * block_width);
    const size_t i_at = r_at + block_width;
    const float coef = rate[ch];
    float S = state[static_cast<size_t>(slot) * channels + ch];  // in front of the round's first token
    for (int base = 0; base < count; base += segments * kScanTokens) {
        const int round = min(count - base, segments * kScanTokens);
        const int per = (round + segments - 1) / segments;
        const int t0 = base + min(seg * per, round), t1 = min(t0 + per, base + round);
        float a[kScanTokens], x[kScanTokens];
        float A = 1.f, B = 0.f;
#pragma unroll
        for (int k0 = 0; k0 < kScanTokens; k0 += kScanAhead) {
            if (k0 >= per) break;  // (the same for the whole workgroup)
            float r_pre[kScanAhead], i_pre[kScanAhead];
            T u_in[kScanAhead];
#pragma unroll
            for (int k = 0; k < kScanAhead; ++k) {  // (a token past the stretch reads the portion's last and is dropped below)
                const size_t token = static_cast<size_t>(first + min(t0 + k0 + k, count - 1));
                r_pre[k] = gates[token * 2 * channels + r_at];
                i_pre[k] = gates[token * 2 * channels + i_at];
                u_in[k] = u[token * channels + ch];
            }
#pragma unroll
            for (int k = 0; k < kScanAhead; ++k) {
                const GateStep now = gate_step(r_pre[k], i_pre[k], to_float(u_in[k]), coef);
                const bool mine = t0 + k0 + k < t1;
                a[k0 + k] = mine ? now.a : 1.f;
                x[k0 + k] = mine ? now.x : 0.f;
                B = fmaf(a[k0 + k], B, x[k0 + k]);
                A *= a[k0 + k];
            }
        }
        a_s[seg][lane] = A;
        b_s[seg][lane] = B;
        __syncthreads();
        for (int before = 0; before < seg; ++before) S = fmaf(a_s[before][lane], S, b_s[before][lane]);
#pragma unroll
        for (int k0 = 0; k0 < kScanTokens; k0 += kScanAhead) {
            if (k0 >= per) break;
            T y_in[kScanAhead];
#pragma unroll
            for (int k = 0; k < kScanAhead; ++k)
                y_in[k] = y_pre[static_cast<size_t>(first + min(t0 + k0 + k, count - 1)) * ldy + ch];
#pragma unroll
            for (int k = 0; k < kScanAhead; ++k) {
                S = fmaf(a[k0 + k], S, x[k0 + k]);
                if (live && t0 + k0 + k < t1)
                    out[static_cast<size_t>(first + t0 + k0 + k) * channels + c] =
                        from_float<T>(S * gelu_tanh(to_float(y_in[k])));
            }
        }
        __syncthreads();
        if (seg == segments - 1) a_s[0][lane] = S;  // (the last stretch ends where the round ends)
        __syncthreads();
        S = a_s[0][lane];
        __syncthreads();
    }
    if (!live || seg != segments - 1) return;
    state[static_cast<size_t>(slot) * channels + c] = S;
    if (taps > 1)
        keep_inputs(past + static_cast<size_t>(slot) * (taps - 1) * channels, x_in, ldx, first, count, c, channels, taps - 1);
}

}  // namespace

CIE_API int cie_retention(void* stream, int dtype, const void* proj, long ldp, int q_off, int k_off, int v_off, int g_off,
                          const float* cos_table, const float* sin_table, int rot, const float* decay, float* state,
                          const int* seq_slot, const int* positions, const int* q_start_loc, float* turned, float* raw,
                          void* out, int tokens, int sequences, int heads, int dim, int vdim, int rows_per_thread,
                          int groups, int parts, int slice, int chunk, float eps, float key_scale, int act,
                          int norm_span, const float* norm_weight, int gate_act, int blocks, float* sums) {
    if (act < 0 || act > 1 || norm_span < 1 || heads % norm_span || gate_act < 0 || gate_act > 1) return CIE_BAD_ARGUMENT;
    if (blocks) {
        // the walk in blocks on the matrix cores: two planes of o, queries and keys padded to whole tiles of 16
        if (!sums) return CIE_BAD_ARGUMENT;
        groups = 1;
        rows_per_thread = 16;
        parts = (dim + 15) / 16;
        slice = vdim < 16 ? vdim : 16;
        chunk = 1;
    }
    if (sequences < 0 || tokens < 0 || heads <= 0 || heads > 65535 || dim <= 0 || vdim <= 0 || groups <= 0 || chunk <= 0 ||
        parts <= 0 || slice <= 0 || slice > vdim || rot < 0 || rot % 2 || rot > dim ||
        (rot > 0 && (!cos_table || !sin_table)) || !(eps > 0.f) ||
        static_cast<long>(rows_per_thread) * groups * parts < dim || !raw || !turned)
        return CIE_BAD_ARGUMENT;
    const int slices = (vdim + slice - 1) / slice;
    const int threads = ((slice * groups + kWave - 1) / kWave) * kWave;
    const int rows = groups * rows_per_thread;
    const int padded = rows * parts;
    const size_t lds = sizeof(float) * static_cast<size_t>(chunk) *
                       (2 * static_cast<size_t>(rows) + slice + static_cast<size_t>(groups) * slice);
    if (!blocks && (threads > 512 || lds > 64 * 1024 || static_cast<long>(slices) * parts > 65535 ||
                    static_cast<long>(chunk) * 2 * rows / 4 > static_cast<long>(kFetchPieces) * threads ||
                    static_cast<long>(chunk) * slice > static_cast<long>(kFetchValues) * threads))
        return CIE_BAD_ARGUMENT;
    const int vdim16 = (vdim + 15) / 16 * 16;
    const int panels = (vdim16 + kPanelCols - 1) / kPanelCols;
    const int most_blocks = (tokens + kBlockTokens - 1) / kBlockTokens;  // (of one sequence: the grid's second size)
    const size_t sums_lds = sizeof(float) * (2 * static_cast<size_t>(kBlockTokens) * (padded + 4) +
                                             kBlockTokens * panel_stride(vdim16 < kPanelCols ? vdim16 : kPanelCols) +
                                             kBlockTokens * kScoreStride + 36);
    const size_t reads_lds = sizeof(float) * (static_cast<size_t>(kBlockTokens) * (padded + 4) + 36);
    if (blocks && (sums_lds > 64 * 1024 || most_blocks > 65535 || panels > 65535 ||
                   static_cast<long>(sequences) * heads > 0x7fffffffL))
        return CIE_BAD_ARGUMENT;
    if (sequences == 0 || tokens == 0) return CIE_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
    // a step of few tokens: up to sixteen workgroups a token, so that a single token's heads do not wait for one
    const int turn_blocks = (heads * padded + 255) / 256;
    const int per_token = tokens >= 256 ? 1 : (turn_blocks < 16 ? turn_blocks : 16);
    const dim3 turn_grid(tokens, per_token);
    if (dtype == CIE_F32)
        retention_turn_kernel<float><<<turn_grid, 256, 0, s>>>(static_cast<const float*>(proj), ldp, q_off, k_off, cos_table,
                                                           sin_table, rot, positions, turned, heads, dim, padded, key_scale, act);
    else if (dtype == CIE_BF16)
        retention_turn_kernel<bf16_t><<<turn_grid, 256, 0, s>>>(static_cast<const bf16_t*>(proj), ldp, q_off, k_off, cos_table,
                                                            sin_table, rot, positions, turned, heads, dim, padded, key_scale, act);
    else
        return CIE_BAD_ARGUMENT;
    const long plane = static_cast<long>(tokens) * heads * vdim;
    int code = CIE_BAD_ARGUMENT;
    if (blocks) {
        const dim3 block_grid(sequences * heads, most_blocks, panels);
        if (dtype == CIE_F32)
            retention_block_sums_kernel<float><<<block_grid, 256, sums_lds, s>>>(
                static_cast<const float*>(proj), ldp, v_off, turned, decay, q_start_loc, raw, sums, heads, vdim, padded,
                vdim16, act);
        else
            retention_block_sums_kernel<bf16_t><<<block_grid, 256, sums_lds, s>>>(
                static_cast<const bf16_t*>(proj), ldp, v_off, turned, decay, q_start_loc, raw, sums, heads, vdim, padded,
                vdim16, act);
        code = cie_after_launch();
        if (code != CIE_OK) return code;
        const dim3 scan_grid(sequences * heads, (padded * vdim16 + 255) / 256);
        retention_scan_kernel<<<scan_grid, 256, 0, s>>>(decay, state, seq_slot, q_start_loc, sums, heads, dim, vdim, padded,
                                                       vdim16);
        code = cie_after_launch();
        if (code != CIE_OK) return code;
        retention_block_reads_kernel<<<block_grid, 256, reads_lds, s>>>(turned, decay, q_start_loc, sums, raw + plane, heads,
                                                                         vdim, padded, vdim16);
        code = cie_after_launch();
        parts = 2;
    } else {
        dim3 grid(sequences, heads, slices * parts);
#define CIE_RETENTION(T, DS)                                                                                         \
        code = launch_retention<T, DS>(s, grid, threads, lds, proj, ldp, v_off, turned, decay, state, seq_slot,          \
                                       q_start_loc, raw, plane, heads, dim, vdim, slice, slices, groups, padded, chunk, act)
        if (dtype == CIE_F32) {
            if (rows_per_thread == 4) CIE_RETENTION(float, 4);
            else if (rows_per_thread == 8) CIE_RETENTION(float, 8);
            else if (rows_per_thread == 16) CIE_RETENTION(float, 16);
            else if (rows_per_thread == 32) CIE_RETENTION(float, 32);
        } else {
            if (rows_per_thread == 4) CIE_RETENTION(bf16_t, 4);
            else if (rows_per_thread == 8) CIE_RETENTION(bf16_t, 8);
            else if (rows_per_thread == 16) CIE_RETENTION(bf16_t, 16);
            else if (rows_per_thread == 32) CIE_RETENTION(bf16_t, 32);
        }
#undef CIE_RETENTION
    }
    if (code != CIE_OK) return code;
    const int items = tokens * (heads / norm_span);
    const int width = norm_span * vdim;
    if (width > 256 && (static_cast<size_t>(width) + 16) * sizeof(float) <= 60 * 1024) {
        // (which kernel norms depends on the run's width alone, never on what else the step holds)
        const int threads = width >= 2048 ? 1024 : width >= 1024 ? 512 : 256;
        const size_t norm_lds = (static_cast<size_t>(width) + 16) * sizeof(float);
        if (dtype == CIE_F32)
            retention_norm_wide_kernel<float><<<items, threads, norm_lds, s>>>(
                raw, plane, parts, static_cast<const float*>(proj), ldp, g_off, static_cast<float*>(out), heads, vdim, eps,
                norm_span, norm_weight, gate_act);
        else
            retention_norm_wide_kernel<bf16_t><<<items, threads, norm_lds, s>>>(
                raw, plane, parts, static_cast<const bf16_t*>(proj), ldp, g_off, static_cast<bf16_t*>(out), heads, vdim,
                eps, norm_span, norm_weight, gate_act);
        return cie_after_launch();
    }
    const int norm_blocks = (items + 3) / 4;
#define CIE_NORM(KERNEL, T)                                                                                           \
    KERNEL<T><<<norm_blocks, 256, 0, s>>>(raw, plane, parts, static_cast<const T*>(proj), ldp, g_off, static_cast<T*>(out), \
                                          tokens, heads, vdim, eps, norm_span, norm_weight, gate_act)
    if (width <= kNormColumns * kWave) {
        if (dtype == CIE_F32) CIE_NORM(retention_norm_narrow_kernel, float);
        else CIE_NORM(retention_norm_narrow_kernel, bf16_t);
    } else {  // (a run that not even the wide kernel's LDS holds)
        if (dtype == CIE_F32) CIE_NORM(retention_norm_kernel, float);
        else CIE_NORM(retention_norm_kernel, bf16_t);
    }
#undef CIE_NORM
    return cie_after_launch();
}

CIE_API int cie_retention_step(void* stream, int dtype, const void* proj, long ldp, int q_off, int k_off, int v_off, int g_off,
                               const float* cos_table, const float* sin_table, int rot, const float* decay, float* state,
                               const int* seq_slot, const int* positions, const int* q_start_loc, void* out, int sequences,
                               int heads, int dim, int vdim, float eps, float key_scale, int act,
                               const float* norm_weight, int gate_act) {
    if (act < 0 || act > 1 || gate_act < 0 || gate_act > 1 || sequences < 0 || heads <= 0 || dim <= 0 || dim > kStepThreads ||
        vdim <= 0 || vdim % 4 || vdim > kStepThreads || rot < 0 || rot % 2 || rot > dim ||
        (rot > 0 && (!cos_table || !sin_table)) || !(eps > 0.f) || reinterpret_cast<size_t>(state) % 16 ||
        static_cast<long>(sequences) * heads > 0x7fffffffL || (dtype != CIE_F32 && dtype != CIE_BF16))
        return CIE_BAD_ARGUMENT;
    const int quads = vdim / 4;
    const int groups = (dim + kStepRows - 1) / kStepRows;
    if (quads * groups > kStepThreads) return CIE_BAD_ARGUMENT;
    if (sequences == 0) return CIE_OK;
    int threads = quads * groups;
    threads = threads < vdim ? vdim : threads;
    threads = threads < dim ? dim : threads;
    threads = (threads + kWave - 1) / kWave * kWave;
    const size_t lds = sizeof(float) * (static_cast<size_t>(groups + 1) * vdim + 2 * static_cast<size_t>(dim) + threads / kWave);
    hipStream_t s = static_cast<hipStream_t>(stream);
#define CIE_STEP(T)                                                                                                        \
    retention_step_kernel<T><<<sequences * heads, threads, lds, s>>>(                                                      \
        static_cast<const T*>(proj), ldp, q_off, k_off, v_off, g_off, cos_table, sin_table, rot, decay, state, seq_slot,   \
        positions, q_start_loc, static_cast<T*>(out), heads, dim, vdim, quads, groups, eps, key_scale, act, norm_weight,   \
        gate_act)
    if (dtype == CIE_F32) CIE_STEP(float);
    else CIE_STEP(bf16_t);
#undef CIE_STEP
    return cie_after_launch();
}

CIE_API int cie_causal_conv(void* stream, int dtype, const void* x, long ldx, const void* taps_w, const void* bias,
                            const float* past, const int* seq_of_token, const int* seq_slot, const int* q_start_loc,
                            void* out, int tokens, int channels, int taps, int act, int out_f32) {
    if (tokens < 0 || tokens > 65535 * 1 || channels <= 0 || taps < 1 || taps > kMaxTaps || ldx < channels || act < 0 ||
        act > 1)
        return CIE_BAD_ARGUMENT;
    if (tokens == 0) return CIE_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    if (dtype == CIE_BF16 && taps == 4 && channels % 8 == 0 && ldx % 8 == 0 && aligned(x) && aligned(taps_w) &&
        aligned(bias) && aligned(past) && aligned(out)) {
        // (tokens that share a thread save loads; with few of them more threads shorten the way)
        const int each = tokens > 128 ? 4 : 1;
        const long items = static_cast<long>((tokens + each - 1) / each) * (channels / 8);
        const unsigned blocks = static_cast<unsigned>((items + 255) / 256);
#define CIE_CONV4(O, EACH)                                                                                           \
    causal_conv4_vec8_kernel<O, EACH><<<blocks, 256, 0, s>>>(                                                          \
        static_cast<const bf16_t*>(x), ldx, static_cast<const bf16_t*>(taps_w), static_cast<const bf16_t*>(bias), past,  \
        seq_of_token, seq_slot, q_start_loc, static_cast<O*>(out), tokens, channels, act)
        if (out_f32 && each == 4) CIE_CONV4(float, 4);
        else if (out_f32) CIE_CONV4(float, 1);
        else if (each == 4) CIE_CONV4(bf16_t, 4);
        else CIE_CONV4(bf16_t, 1);
#undef CIE_CONV4
        return cie_after_launch();
    }
    dim3 grid((channels + 255) / 256, tokens);
#define CIE_CONV(T, O)                                                                                              \
    causal_conv_kernel<T, O><<<grid, 256, 0, s>>>(static_cast<const T*>(x), ldx, static_cast<const T*>(taps_w),          \
                                                  static_cast<const T*>(bias), past, seq_of_token, seq_slot,            \
                                                  q_start_loc, static_cast<O*>(out), channels, taps, act)
    if (dtype == CIE_F32) CIE_CONV(float, float);
    else if (dtype == CIE_BF16 && out_f32) CIE_CONV(bf16_t, float);
    else if (dtype == CIE_BF16) CIE_CONV(bf16_t, bf16_t);
#undef CIE_CONV
    else
        return CIE_BAD_ARGUMENT;
    return cie_after_launch();
}

// Moves the convolution's state on by the step's inputs (see conv_keep_kernel); call it behind cie_causal_conv.
CIE_API int cie_conv_keep(void* stream, int dtype, const void* x, long ldx, float* past, const int* seq_slot,
                          const int* q_start_loc, int sequences, int channels, int taps) {
    if (sequences < 0 || sequences > 65535 || channels <= 0 || taps < 1 || taps > kMaxTaps || ldx < channels)
        return CIE_BAD_ARGUMENT;
    if (sequences == 0 || taps == 1) return CIE_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
    dim3 grid((channels + 255) / 256, sequences);
    if (dtype == CIE_F32)
        conv_keep_kernel<float><<<grid, 256, 0, s>>>(static_cast<const float*>(x), ldx, past, seq_slot, q_start_loc,
                                                     channels, taps);
    else if (dtype == CIE_BF16)
        conv_keep_kernel<bf16_t><<<grid, 256, 0, s>>>(static_cast<const bf16_t*>(x), ldx, past, seq_slot, q_start_loc,
                                                      channels, taps);
    else
        return CIE_BAD_ARGUMENT;
    return cie_after_launch();
}

CIE_API int cie_gated_recurrence(void* stream, int dtype, const void* y_pre, long ldy, const void* x_in, long ldx,
                                 const void* u, const float* gates, int block_width, const float* rate, float* state,
                                 float* past, const int* seq_slot, const int* q_start_loc, void* out, int sequences,
                                 int channels, int taps, int segments) {
    if (sequences < 0 || sequences > 65535 || channels <= 0 || block_width <= 0 || channels % block_width || taps < 1 ||
        taps > kMaxTaps || ldy < channels || ldx < channels || segments < 1 || segments > kMaxSegments)
        return CIE_BAD_ARGUMENT;
    if (sequences == 0) return CIE_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
#define CIE_SCAN(T)                                                                                                 \
    if (segments == 1)                                                                                              \
        gated_recurrence_kernel<T><<<dim3((channels + 63) / 64, sequences), 64, 0, s>>>(                             \
            static_cast<const T*>(y_pre), ldy, static_cast<const T*>(x_in), ldx, static_cast<const T*>(u), gates,     \
            block_width, rate, state, past, seq_slot, q_start_loc, static_cast<T*>(out), channels, taps);             \
    else                                                                                                            \
        gated_recurrence_stretches_kernel<T>                                                                         \
            <<<dim3((channels + kScanChannels - 1) / kScanChannels, sequences), kScanChannels * segments, 0, s>>>(    \
                static_cast<const T*>(y_pre), ldy, static_cast<const T*>(x_in), ldx, static_cast<const T*>(u), gates, \
                block_width, rate, state, past, seq_slot, q_start_loc, static_cast<T*>(out), channels, taps, segments)
    if (dtype == CIE_F32) {
        CIE_SCAN(float);
    } else if (dtype == CIE_BF16) {
        CIE_SCAN(bf16_t);
    }
#undef CIE_SCAN
    else
        return CIE_BAD_ARGUMENT;
    return cie_after_launch();
}

CIE_API int cie_gated_recurrence_step(void* stream, const void* y_pre, long ldy, const void* x_in, long ldx, const void* u,
                                      const void* weight, const void* bias, int block_width, const float* rate, float* state,
                                      float* past, const int* seq_slot, const int* q_start_loc, void* out, int sequences,
                                      int tokens, int channels, int taps) {
    if (sequences < 0 || tokens < 0 || channels <= 0 || block_width <= 0 || block_width % 8 || channels % block_width ||
        taps < 1 || taps > kStepTaps + 1 || ldy < channels || ldx < channels || sequences > 16 * 65535 ||
        reinterpret_cast<size_t>(u) % 16 || reinterpret_cast<size_t>(weight) % 16)
        return CIE_BAD_ARGUMENT;
    if (sequences == 0 || tokens == 0) return CIE_OK;
    const int tiles = (block_width + 15) / 16;
    gated_recurrence_step_kernel<<<dim3(channels / block_width * tiles, (sequences + 15) / 16), 256, 0,
                                   static_cast<hipStream_t>(stream)>>>(
        static_cast<const bf16_t*>(y_pre), ldy, static_cast<const bf16_t*>(x_in), ldx, static_cast<const bf16_t*>(u),
        static_cast<const bf16_t*>(weight), static_cast<const bf16_t*>(bias), block_width, tiles, rate, state, past, seq_slot,
        q_start_loc, static_cast<bf16_t*>(out), sequences, tokens, channels, taps - 1);
    return cie_after_launch();
}

// The same for any portions of tokens, in chunks (see gated_chunks_kernel).  block_width 64, 128 or 256; u, weight, y_pre, planes, carry
// and state at 16-byte addresses, ldy a multiple of 8.  planes: 2 * tokens * channels floats, carry: 2 * channels for every 64 tokens.
CIE_API int cie_gated_recurrence_chunks(void* stream, const void* y_pre, long ldy, const void* x_in, long ldx, const void* u,
                                        const void* weight, const void* bias, int block_width, const float* rate, float* state,
                                        float* past, const int* seq_of_token, const int* seq_slot, const int* q_start_loc, void* out,
                                        float* planes, float* carry, int sequences, int tokens, int channels, int taps) {
    const auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    if (sequences < 0 || tokens < 0 || channels <= 0 || (block_width != 64 && block_width != 128 && block_width != 256) || channels % block_width ||
        taps < 1 || taps > kMaxTaps || ldy < channels || ldy % 8 || ldx < channels || !aligned(y_pre) || !aligned(u) || !aligned(weight) ||
        !aligned(rate) || !aligned(state) || !aligned(out) || !aligned(planes) || !aligned(carry))
        return CIE_BAD_ARGUMENT;
    if (tokens == 0) return CIE_OK;
    const int chunks = (tokens + kChunkTokens - 1) / kChunkTokens;
    const long groups = static_cast<long>(chunks) * (channels / kChunkChannels);
    const int token_groups = (tokens + kOutputTokens - 1) / kOutputTokens;
    const long outputs = (channels + 255L) / 256 * (token_groups + (taps > 1 ? static_cast<long>(sequences) : 0L));
    if (groups > 0x7fffffffL || outputs > 0x7fffffffL) return CIE_BAD_ARGUMENT;
    hipStream_t s = static_cast<hipStream_t>(stream);
    float* plane_b = planes + static_cast<size_t>(tokens) * channels;
#define CIE_CHUNKS(BW)                                                                                                     \
    gated_chunks_kernel<BW><<<static_cast<unsigned>(groups), 256, 0, s>>>(                                                  \
        static_cast<const bf16_t*>(u), static_cast<const bf16_t*>(weight), static_cast<const bf16_t*>(bias), rate, state,   \
        seq_of_token, seq_slot, q_start_loc, planes, plane_b, carry, tokens, channels, chunks)
    if (block_width == 64) CIE_CHUNKS(64);
    else if (block_width == 128) CIE_CHUNKS(128);
    else CIE_CHUNKS(256);
#undef CIE_CHUNKS
    const int code = cie_after_launch();
    if (code != CIE_OK) return code;
    gated_outputs_kernel<<<static_cast<unsigned>(outputs), 256, 0, s>>>(
        static_cast<const bf16_t*>(y_pre), ldy, static_cast<const bf16_t*>(x_in), ldx, planes, plane_b, carry, state, past, seq_of_token,
        seq_slot, q_start_loc, static_cast<bf16_t*>(out), tokens, channels, taps - 1, token_groups);
    return cie_after_launch();
}

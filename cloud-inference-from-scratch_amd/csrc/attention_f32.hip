// Paged grouped-query attention in true float32 on the matrix cores (v_mfma_f32_16x16x4_f32: float32 products and
// sums), heads of 32, 64, 96 or 128 dimensions, pages of a power of two >= 4 tokens, up to 64 query heads a key head.
//
//   q      [tokens, q_heads, D] with row stride q_row_stride (elements)
//   keys   [pages, kv_heads, page_size, D],  values [pages, kv_heads, D, page_size] (transposed)
//   out    [tokens, q_heads * D]
//
// Tiles hold consecutive tokens of one sequence; a tile's rows are (token, head of the group): row = token * G + head,
// up to 64 of them, 16 to a wave.  Both forms do the same arithmetic for a row, in the same order, so a token's result
// does not depend on how its prompt was cut, on what else is in the batch, or on the form:
//
//   keys in blocks of 64 (counted from the sequence's start);  in a block  s = (q . k) * scale,  m = max of the keys
//   that the row sees,  p = exp(s - m),  l = sum p,  o = sum p v;  the blocks joined one after the other:
//   M' = max(M, m),  L = L exp(M - M') + l exp(m - M'),  O alike (a block without a key of the row changes nothing);
//   out = O / L.
//
// Operands: S^T = K . Q^T leaves lane (r = lane % 16, g = lane / 16) the scores of row r and keys 4g .. 4g + 3 of each 16,
// which is the operand of P . V as it stands (an instruction takes one key of each quarter of 16); a lane's
// operands of K and Q are one number of each four dimensions (16-byte loads change places over the wave's quarters), so
// that a score is the sum over ascending dimensions.
//
// * attention_f32_prompt_kernel: four waves share a tile's 64 keys and values through LDS, the next 64 on their way in
//   registers; bound by the matrix cores (16 rows x 64 keys x 128 dimensions: 8,192 cycles a wave).
// * attention_f32_block_kernel: a wave, or four, per 16 rows and block, straight from memory, the blocks' (m, l, o) to a workspace,
//   and attention_f32_join_kernel joins them: single tokens, and tiles too few to fill the units.
//
// Measured (MI355X, us a layer; the generic kernel, one thread a key and an output number, in brackets): a prompt of 517
// tokens with 16 query heads on 2 key heads of 128 66 in blocks, 79 in whole tiles (634), 4 tokens over 1,000 keys 11.4 for
// both kernels (117).
#include "common.h"

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kKeys = 64;      // keys of a block
constexpr int kRowsTile = 64;  // rows of a tile
constexpr int kTileWaves = 4;

struct Args {
    const float* q;
    int q_row_stride;
    const float *k_pool, *v_pool;
    const int* block_table;
    int table_width;
    const int *tile_seq, *tile_q0;  // both or neither: tile i is the first of sequence i
    const int *seq_slot, *seq_start, *seq_q_len, *q_start_loc;
    float* out;
    float *part_o, *part_ml;  // [tiles, kv_heads, blocks, rows, D] and [.., rows, 2]; packed: a tile has the blocks it needs
    int rows;                 // of a tile in the workspace
    int blocks;               // ... and the most blocks of a tile
    int capacity;             // 0: every tile has `blocks` places in the workspace; else places that a round of tiles shares
    int round;                // packed: the round that runs (prompt form: the first that it runs)
    int q_heads, kv_heads, page_shift, window;
    float scale;
    int tokens_per_tile;
};

struct Tile {
    int start, q0, tokens, first_row_token, lo, hi;
    const int* table;
};

__device__ __forceinline__ Tile tile_of(const Args& a, int index) {
    Tile t;
    const int seq = a.tile_seq ? a.tile_seq[index] : index;
    t.q0 = a.tile_seq ? a.tile_q0[index] : 0;
    t.start = a.seq_start[seq];
    t.tokens = min(a.tokens_per_tile, a.seq_q_len[seq] - t.q0);
    t.first_row_token = a.q_start_loc[seq] + t.q0;
    t.hi = t.start + t.q0 + t.tokens;  // keys that some row of the tile sees: [lo, hi)
    t.lo = a.window > 0 ? max(0, t.start + t.q0 + 1 - a.window) : 0;
    t.table = a.block_table + static_cast<size_t>(a.seq_slot[seq]) * a.table_width;
    return t;
}

__device__ __forceinline__ int blocks_of(const Tile& t) { return (t.hi - 1) / kKeys - t.lo / kKeys + 1; }

// Packed, the tiles' blocks lie one behind the other in the workspace, in rounds of `capacity` places (a round's last tile may
// reach beyond it, by less than `blocks`): what a captured step launches, and the memory it takes, then follow the lengths
// that the device knows, not the longest contexts that it may ever see.  The blocks of the tiles before this one; every lane
// of a wave calls it.
__device__ __forceinline__ int blocks_before(const Args& a, int index) {
    int before = 0;
    for (int j = threadIdx.x % kWave; j < index; j += kWave) before += blocks_of(tile_of(a, j));
#pragma unroll
    for (int offset = kWave / 2; offset > 0; offset >>= 1) before += __shfl_xor(before, offset, kWave);
    return before;
}

// Where the parts of (tile, kv head) begin in the workspace, in rows; false: the tile is another round's.
__device__ __forceinline__ bool tile_place(const Args& a, int index, int count, int kv_head, size_t& at) {
    if (a.capacity == 0) {
        at = (static_cast<size_t>(index) * a.kv_heads + kv_head) * a.blocks * a.rows;
        return true;
    }
    const int before = blocks_before(a, index);
    at = (static_cast<size_t>(before % a.capacity) * a.kv_heads + static_cast<size_t>(kv_head) * count) * a.rows;
    return before / a.capacity == a.round;
}

__device__ __forceinline__ bool is_finite_bits(float v) { return (__float_as_uint(v) & 0x7f800000u) != 0x7f800000u; }

// q . k of 16 keys and 16 rows, the dimensions in ascending order (what an instruction takes of 16 dimensions are four
// neighbours, one of each quarter of the wave)
template <int kG, typename Keys>
__device__ __forceinline__ floatx4 scores(const Keys& keys, const floatx4 (&q)[kG]) {
    floatx4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < kG; ++i) {
        const floatx4 k = keys(i);
#pragma unroll
        for (int j = 0; j < 4; ++j) sum = __builtin_amdgcn_mfma_f32_16x16x4f32(k[j], q[i][j], sum, 0, 0, 0);
    }
    return sum;
}

// A row's block: masked scores to probabilities; m and l in every lane of the row's column of four.
__device__ __forceinline__ void block_softmax(floatx4 (&s)[kKeys / 16], int kb, int pos, int row_lo, float scale, int g,
                                              float& m, float& l) {
    m = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < kKeys / 16; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int key = kb + 16 * kt + 4 * g + i;
            s[kt][i] = key <= pos && key >= row_lo ? s[kt][i] * scale : -INFINITY;
            m = fmaxf(m, s[kt][i]);
        }
    m = rows_max(m);
    const float from = m == -INFINITY ? 0.f : m;
    l = 0.f;
#pragma unroll
    for (int kt = 0; kt < kKeys / 16; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            s[kt][i] = expf(s[kt][i] - from);
            l += s[kt][i];
        }
    l = rows_sum(l);
}

// The join of a block's m with the running M: the factors of what stands and of what comes, and the new M.
__device__ __forceinline__ void join_factors(float& M, float m, float& stands, float& comes) {
    const float to = fmaxf(M, m);
    const float from = to == -INFINITY ? 0.f : to;
    stands = expf(M - from);
    comes = expf(m - from);
    M = to;
}

// A block some of whose values are infinite or NaN, and which some row does not see whole: the product took such values
// as 0 (0 times them is a NaN, in the rows that do not see them too), and here the rows that see them get them.  A lane
// holds dimension 16 dt + r of rows 4 g + i, its n-th dt = first + n * apart; the probability of (row, key 16 kt + 4 gg + j) lies in
// lane 16 gg + row.
template <int D, int kOwn>
__device__ __forceinline__ void add_odd_values(const Args& a, const Tile& t, int kb, int kv_head, int pos, int r, int g,
                                               const floatx4 (&p)[kKeys / 16], const float (&factor)[4], floatx4 (&o)[kOwn],
                                               int first = 0, int apart = 1) {
#pragma unroll 1
    for (int c = 0; c < kKeys; ++c) {
        const int key = kb + c;
        if (key < t.lo || key >= t.hi) continue;
        const float* v = a.v_pool + ((static_cast<size_t>(t.table[key >> a.page_shift]) * a.kv_heads + kv_head) * D << a.page_shift) +
                         (key & ((1 << a.page_shift) - 1));
        float here = 0.f;
#pragma unroll
        for (int kt = 0; kt < kKeys / 16; ++kt)
#pragma unroll
            for (int j = 0; j < 4; ++j) here = kt == c / 16 && j == c % 4 ? p[kt][j] : here;
        float of_row[4];
        bool sees[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            of_row[i] = __shfl(here, 16 * (c % 16 / 4) + 4 * g + i, kWave) * factor[i];
            const int at = __shfl(pos, 4 * g + i, kWave);
            sees[i] = key <= at && !(a.window > 0 && key < at + 1 - a.window);
        }
#pragma unroll
        for (int dt = 0; dt < kOwn; ++dt) {
            const float x = v[static_cast<size_t>(16 * min(first + dt * apart, D / 16 - 1) + r) << a.page_shift];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (sees[i] && !is_finite_bits(x)) o[dt][i] = fmaf(of_row[i], x, o[dt][i]);
        }
    }
}

template <int D>
__device__ __forceinline__ int k_chunk(int row, int c) {  // 16-byte chunk c of key `row` in LDS
    constexpr int kChunks = D / 4;
    return row * D + 4 * (kChunks % 16 == 0 ? c ^ (row & 15) : c ^ ((row >> 1) & 7));
}
__device__ __forceinline__ int v_chunk(int d, int c) { return d * kKeys + 4 * (c ^ (d & 15)); }  // keys 4c.. of dimension d

template <int D>
__global__ void __launch_bounds__(kTileWaves * kWave, 2) attention_f32_prompt_kernel(Args a) {
    constexpr int kG = D / 16;                                           // 16-wide pieces of a head
    constexpr int kLoads = kKeys * D / 4 / (kTileWaves * kWave);         // 16-byte loads of a thread for 64 keys
    __shared__ float k_s[kKeys * D];
    __shared__ float v_s[kKeys * D];
    __shared__ int odd[2];  // whether a block's values hold an infinity or a NaN (two take turns)
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int r = lane % 16, g = lane / 16;
    const int kv_head = blockIdx.y;
    const int group = a.q_heads / a.kv_heads;
    // (the longest tiles first)
    const int index = gridDim.x - 1 - blockIdx.x;
    const Tile t = tile_of(a, index);
    if (a.capacity && blocks_before(a, index) / a.capacity < a.round) return;  // (a tile of the block form's rounds)
    const int page_mask = (1 << a.page_shift) - 1;

    // this lane's row
    const int row = 16 * wave + r;
    const bool valid = row < t.tokens * group;
    const int tok = valid ? row / group : 0;
    const int head = valid ? row - tok * group : 0;
    const int pos = valid ? t.start + t.q0 + tok : -1;
    const int row_lo = a.window > 0 ? pos + 1 - a.window : 0;
    floatx4 q[kG];
    const float* q_row = a.q + static_cast<size_t>(t.first_row_token + tok) * a.q_row_stride +
                         static_cast<size_t>(kv_head * group + head) * D + 4 * g;
#pragma unroll
    for (int i = 0; i < kG; ++i) q[i] = across_quarters(*reinterpret_cast<const floatx4*>(q_row + 16 * i));
    // positions of the tile's first row and of this wave's last one: where masks matter, where the wave is done
    const int first_pos = t.start + t.q0;
    const int wave_rows = min(16 * wave + 16, t.tokens * group);
    const int wave_last = 16 * wave < t.tokens * group ? first_pos + (wave_rows - 1) / group : -1;

    const int v_shift = min(a.page_shift, 6) - 2;  // 16-byte chunks of a dimension's values in a block's page, as a shift
    floatx4 k_next[kLoads], v_next[kLoads];
    auto fetch = [&](int kb) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int e = threadIdx.x + i * kTileWaves * kWave;
            const int key = max(min(kb + e / (D / 4), t.hi - 1), t.lo);  // (keys outside [lo, hi) may have no page)
            const int page = t.table[key >> a.page_shift];
            k_next[i] = *reinterpret_cast<const floatx4*>(
                a.k_pool + (((static_cast<size_t>(page) * a.kv_heads + kv_head) << a.page_shift) + (key & page_mask)) * D + 4 * (e % (D / 4)));
            // values: consecutive threads take a dimension's chunks of a page, then the next dimension's
            const int in_page = e & ((1 << v_shift) - 1), d = (e >> v_shift) % D, p = (e >> v_shift) / D;
            const int chunk = (p << v_shift) + in_page;
            const int v_key = max(min(kb + 4 * chunk, (t.hi - 1) & ~3), t.lo & ~3);
            const int v_page = t.table[v_key >> a.page_shift];
            v_next[i] = *reinterpret_cast<const floatx4*>(
                a.v_pool + (((static_cast<size_t>(v_page) * a.kv_heads + kv_head) * D + d) << a.page_shift) + (v_key & page_mask));
        }
    };

    float M = -INFINITY, L = 0.f;
    floatx4 o[kG];
#pragma unroll
    for (int i = 0; i < kG; ++i) o[i] = floatx4{0.f, 0.f, 0.f, 0.f};
    int kb = t.lo & ~(kKeys - 1);
    int turn = 0;
    if (threadIdx.x < 2) odd[threadIdx.x] = 0;
    fetch(kb);
    for (; kb < t.hi; kb += kKeys, turn ^= 1) {
        __syncthreads();  // the block before has been read by all waves
        // a block of which some row does not see some key
        const bool edge = kb + kKeys - 1 > first_pos || (a.window > 0 && kb < t.hi - a.window);
        bool any_odd = false;
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int e = threadIdx.x + i * kTileWaves * kWave;
            *reinterpret_cast<floatx4*>(k_s + k_chunk<D>(e / (D / 4), e % (D / 4))) = k_next[i];
            const int in_page = e & ((1 << v_shift) - 1), d = (e >> v_shift) % D, p = (e >> v_shift) / D;
            const int chunk = (p << v_shift) + in_page;
            floatx4 v = v_next[i];
            if (edge) {
                // what no row sees is no value; an infinity or NaN times a masked row's 0 would be a NaN: such values
                // count as 0 in the product, and the rows that do see them get them below
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int key = kb + 4 * chunk + j;
                    const bool there = key >= t.lo && key < t.hi;
                    any_odd |= there && !is_finite_bits(v[j]);
                    v[j] = there && is_finite_bits(v[j]) ? v[j] : 0.f;
                }
            }
            *reinterpret_cast<floatx4*>(v_s + v_chunk(d, chunk)) = v;
        }
        if (any_odd) odd[turn] = 1;
        if (threadIdx.x == 0) odd[turn ^ 1] = 0;
        if (kb + kKeys < t.hi) fetch(kb + kKeys);
        __syncthreads();
        if (kb > wave_last) continue;  // (the wave's barriers are those at the loop's head)

        floatx4 s[kKeys / 16];
#pragma unroll
        for (int kt = 0; kt < kKeys / 16; ++kt) {
            s[kt] = scores<kG>([&](int i) {
                return across_quarters(*reinterpret_cast<const floatx4*>(k_s + k_chunk<D>(16 * kt + r, 4 * i + g)));
            }, q);
        }
        float m, l;
        block_softmax(s, kb, pos, row_lo, a.scale, g, m, l);
        float stands, comes;
        join_factors(M, m, stands, comes);
        L = fmaf(l, comes, L * stands);
        float row_stands[4], row_comes[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            row_stands[i] = __shfl(stands, 4 * g + i, kWave);
            row_comes[i] = __shfl(comes, 4 * g + i, kWave);
        }
        const bool some_odd = edge && odd[turn];  // (the same for the whole workgroup)
#pragma unroll
        for (int dt = 0; dt < kG; ++dt) {
            floatx4 part = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kt = 0; kt < kKeys / 16; ++kt) {
                const floatx4 v = *reinterpret_cast<const floatx4*>(v_s + v_chunk(16 * dt + r, 4 * kt + g));
#pragma unroll
                for (int j = 0; j < 4; ++j) part = __builtin_amdgcn_mfma_f32_16x16x4f32(s[kt][j], v[j], part, 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) o[dt][i] = fmaf(part[i], row_comes[i], o[dt][i] * row_stands[i]);
        }
        if (some_odd) add_odd_values<D, kG>(a, t, kb, kv_head, pos, r, g, s, row_comes, o);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int out_row = 16 * wave + 4 * g + i;
        const float den = __shfl(L, 4 * g + i, kWave);
        if (out_row >= t.tokens * group) continue;
        const int out_tok = out_row / group, out_head = out_row - out_tok * group;
        float* to = a.out + (static_cast<size_t>(t.first_row_token + out_tok) * a.q_heads + kv_head * group + out_head) * D + r;
#pragma unroll
        for (int dt = 0; dt < kG; ++dt) to[16 * dt] = o[dt][i] / den;
    }
}

// blockIdx: (tile, kv head and 16 rows of the tile, first of the workgroup's blocks: it takes every gridDim.z-th).
// kWaves: 1, or 4 that share a block where there are few: each takes 16 of its keys and a quarter of the dimensions, so that a wave has
// 16 KB to ask for and a fourth of the products, which a wave alone on its unit made one after the other; the scores meet in LDS, and every
// sum stays in its order.  (A wave of the four makes the whole softmax, so where many blocks fill the units one wave is the better.)
// Both kernels, 16 heads of 128 on 2, one sequence of 1,000 keys 15.5 -> 10.7 us, four 15.9 -> 11.4, eight 16.2 -> 12.2; 14 heads of 64 11.6
// -> 9.6 of four.
template <int D, int kWaves>
__global__ void __launch_bounds__(kWaves * kWave, 1) attention_f32_block_kernel(Args a) {
    constexpr int kG = D / 16;
    constexpr int kOwnKeys = kKeys / 16 / kWaves;               // tiles of 16 keys of a wave ...
    constexpr int kOwnDims = (kG + kWaves - 1) / kWaves;        // ... and pieces of 16 dimensions: wave, wave + kWaves, ...
    const int lane = threadIdx.x % kWave, r = lane % 16, g = lane / 16;
    const int wave = kWaves > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) : 0;
    __shared__ floatx4 met[kWaves > 1 ? 2 : 1][kWaves > 1 ? kKeys / 16 : 1][kWaves > 1 ? kWave : 1];  // (two take turns)
    const int group = a.q_heads / a.kv_heads;
    const int row_tiles = gridDim.y / a.kv_heads;
    const int kv_head = blockIdx.y / row_tiles, row_tile = blockIdx.y % row_tiles;
    const Tile t = tile_of(a, blockIdx.x);
    const int rows = t.tokens * group;
    if (16 * row_tile >= rows) return;
    const int first_block = t.lo / kKeys, last_block = (t.hi - 1) / kKeys;
    size_t place;
    if (!tile_place(a, blockIdx.x, last_block - first_block + 1, kv_head, place)) return;
    const int page_mask = (1 << a.page_shift) - 1;
    const int row = 16 * row_tile + r;
    const bool valid = row < rows;
    const int tok = valid ? row / group : 0;
    const int head = valid ? row - tok * group : 0;
    const int pos = valid ? t.start + t.q0 + tok : -1;
    const int row_lo = a.window > 0 ? pos + 1 - a.window : 0;
    const int first_pos = t.start + t.q0;
    floatx4 q[kG];
    const float* q_row = a.q + static_cast<size_t>(t.first_row_token + tok) * a.q_row_stride +
                         static_cast<size_t>(kv_head * group + head) * D + 4 * g;
#pragma unroll
    for (int i = 0; i < kG; ++i) q[i] = *reinterpret_cast<const floatx4*>(q_row + 16 * i);
#pragma unroll
    for (int i = 0; i < kG; ++i) q[i] = across_quarters(q[i]);

    int turn = 0;
    for (int block = first_block + blockIdx.z; block <= last_block; block += gridDim.z, turn ^= 1) {
        const int kb = block * kKeys;
        const bool edge = kb + kKeys - 1 > first_pos || (a.window > 0 && kb < t.hi - a.window);
        // every load of the block is on its way before the first is used: the barriers keep the compiler from placing
        // each beside its use, where a wave that is alone on its SIMD waits for them one after another (four sequences of
        // 1,012 keys: 18.2 -> 12.6 us)
        floatx4 s[kKeys / 16], k[kOwnKeys][kG], v[kOwnDims][kKeys / 16];
        int key_page[kOwnKeys], value_page[kKeys / 16];
#pragma unroll
        for (int n = 0; n < kOwnKeys; ++n)
            key_page[n] = t.table[max(min(kb + 16 * (wave + n) + r, t.hi - 1), t.lo) >> a.page_shift];
#pragma unroll
        for (int kt = 0; kt < kKeys / 16; ++kt)
            value_page[kt] = t.table[max(min(kb + 16 * kt + 4 * g, (t.hi - 1) & ~3), t.lo & ~3) >> a.page_shift];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int n = 0; n < kOwnKeys; ++n) {
            const int key = max(min(kb + 16 * (wave + n) + r, t.hi - 1), t.lo);
            const float* k_row = a.k_pool + (((static_cast<size_t>(key_page[n]) * a.kv_heads + kv_head) << a.page_shift) +
                                             (key & page_mask)) * D + 4 * g;
#pragma unroll
            for (int i = 0; i < kG; ++i) k[n][i] = *reinterpret_cast<const floatx4*>(k_row + 16 * i);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kt = 0; kt < kKeys / 16; ++kt) {
            const int key = max(min(kb + 16 * kt + 4 * g, (t.hi - 1) & ~3), t.lo & ~3);
            const float* v_base = a.v_pool + ((static_cast<size_t>(value_page[kt]) * a.kv_heads + kv_head) * D << a.page_shift) +
                                  (key & page_mask);
#pragma unroll
            for (int n = 0; n < kOwnDims; ++n)  // (a piece past the last reads that one, and is not stored)
                v[n][kt] = *reinterpret_cast<const floatx4*>(
                    v_base + (static_cast<size_t>(16 * min(wave + n * kWaves, kG - 1) + r) << a.page_shift));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int n = 0; n < kOwnKeys; ++n) {
            const floatx4 own = scores<kG>([&](int i) { return across_quarters(k[n][i]); }, q);
            if constexpr (kWaves > 1) met[turn][wave][lane] = own;
            else s[n] = own;
        }
        bool any_odd = false;
        if (edge) {
#pragma unroll
            for (int n = 0; n < kOwnDims; ++n)
#pragma unroll
                for (int kt = 0; kt < kKeys / 16; ++kt)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int key = kb + 16 * kt + 4 * g + j;
                        const bool there = key >= t.lo && key < t.hi;
                        any_odd |= there && !is_finite_bits(v[n][kt][j]);
                        v[n][kt][j] = there && is_finite_bits(v[n][kt][j]) ? v[n][kt][j] : 0.f;
                    }
        }
        if constexpr (kWaves > 1) {
            __syncthreads();
#pragma unroll
            for (int kt = 0; kt < kKeys / 16; ++kt) s[kt] = met[turn][kt][lane];
        }
        float m, l;
        block_softmax(s, kb, pos, row_lo, a.scale, g, m, l);
        const size_t at = place + static_cast<size_t>(block - first_block) * a.rows;
        if (wave == 0 && g == 0 && row < a.rows) {
            a.part_ml[(at + row) * 2] = m;
            a.part_ml[(at + row) * 2 + 1] = l;
        }
        const bool some_odd = __any(any_odd);
        floatx4 o[kOwnDims];
#pragma unroll
        for (int n = 0; n < kOwnDims; ++n) {
            floatx4 part = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kt = 0; kt < kKeys / 16; ++kt)
#pragma unroll
                for (int j = 0; j < 4; ++j) part = __builtin_amdgcn_mfma_f32_16x16x4f32(s[kt][j], v[n][kt][j], part, 0, 0, 0);
            o[n] = part;
        }
        if (some_odd) {
            const float whole[4] = {1.f, 1.f, 1.f, 1.f};
            add_odd_values<D, kOwnDims>(a, t, kb, kv_head, pos, r, g, s, whole, o, wave, kWaves);
        }
#pragma unroll
        for (int n = 0; n < kOwnDims; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int out_row = 16 * row_tile + 4 * g + i;
                if (out_row < a.rows && wave + n * kWaves < kG) a.part_o[(at + out_row) * D + 16 * (wave + n * kWaves) + r] = o[n][i];
            }
    }
}

// Places of 16 rows and a block up to which four waves share one: heads of 64 dimensions and more, and of 32, whose wave has a fourth
// to do (us, one wave and four: 16 heads of 128 on 2, 1,280 places 23.3, 18.6, 1,024 26.6, 25.9, 1,008 of 63 a tile level; of 64, 1,280
// 14.8, 13.1; 4 heads of 32 on 2, 128 9.7, 9.0, 512 10.4, 10.5, 1,024 11.5, 11.9).
constexpr long kShareUpTo = 2048, kShareUpToNarrow = 256;
constexpr int kJoin = 16;  // blocks that a thread asks for at once (16 blocks a row: 8.0 -> 4.6 us)

// One workgroup per (tile, token of the tile, query head), a thread a dimension: the row's blocks joined in order.
template <int D>
__global__ void __launch_bounds__((D + kWave - 1) / kWave * kWave) attention_f32_join_kernel(Args a) {
    const int group = a.q_heads / a.kv_heads;
    const int tok = blockIdx.y / a.q_heads, q_head = blockIdx.y % a.q_heads;
    const Tile t = tile_of(a, blockIdx.x);
    const int d = threadIdx.x;
    if (tok >= t.tokens) return;
    const int kv_head = q_head / group, row = tok * group + q_head % group;
    const int count = blocks_of(t);
    size_t base;
    if (!tile_place(a, blockIdx.x, count, kv_head, base) || d >= D) return;
    base += row;
    float M = -INFINITY, L = 0.f, o = 0.f;
    for (int first = 0; first < count; first += kJoin) {
        float m[kJoin], l[kJoin], part[kJoin];
#pragma unroll
        for (int i = 0; i < kJoin; ++i) {  // (a block past the last is read again and dropped)
            const size_t at = base + static_cast<size_t>(min(first + i, count - 1)) * a.rows;
            m[i] = a.part_ml[at * 2];
            l[i] = a.part_ml[at * 2 + 1];
            part[i] = a.part_o[at * D + d];
        }
        __builtin_amdgcn_sched_barrier(0);  // (all of them on their way before the first is used)
#pragma unroll
        for (int i = 0; i < kJoin; ++i) {  // (a select, no way out: behind one the compiler waits for load after load)
            const bool there = first + i < count;
            float stands, comes, M_next = M;
            join_factors(M_next, m[i], stands, comes);
            const float L_next = fmaf(l[i], comes, L * stands), o_next = fmaf(part[i], comes, o * stands);
            M = there ? M_next : M;
            L = there ? L_next : L;
            o = there ? o_next : o;
        }
    }
    a.out[(static_cast<size_t>(t.first_row_token + tok) * a.q_heads + q_head) * D + d] = o / L;
}

template <int D>
int run(hipStream_t s, const Args& a, int n_tiles, int row_tiles, int turns) {
    if (turns == 0) {
        attention_f32_prompt_kernel<D><<<dim3(n_tiles, a.kv_heads), kTileWaves * kWave, 0, s>>>(a);
    } else {
        const dim3 grid(n_tiles, a.kv_heads * row_tiles, turns);
        if (static_cast<long>(n_tiles) * a.kv_heads * row_tiles * turns <= (D >= 64 ? kShareUpTo : kShareUpToNarrow))
            attention_f32_block_kernel<D, kTileWaves><<<grid, kTileWaves * kWave, 0, s>>>(a);
        else
            attention_f32_block_kernel<D, 1><<<grid, kWave, 0, s>>>(a);
        attention_f32_join_kernel<D><<<dim3(n_tiles, a.tokens_per_tile * a.q_heads), (D + kWave - 1) / kWave * kWave, 0, s>>>(a);
    }
    return cie_after_launch();
}

}  // namespace

// `turns` 0: the prompt form.  Otherwise the block form with that many waves to a tile's 16 rows, and the workspaces part_o
// [n_tiles, kv_heads, blocks, rows, D] and part_ml [.., 2] with rows >= tokens_per_tile * group and blocks enough for every
// tile's keys.  `capacity` > 0: the tiles of round `round`, packed into workspaces of (capacity + blocks) * kv_heads * rows
// rows; the prompt form then runs the tiles of that round and all later ones.
CIE_API int cie_paged_attention_f32(void* stream, const float* q, int q_row_stride, const float* k_pool, const float* v_pool,
                                    const int* block_table, int table_width, const int* tile_seq, const int* tile_q0,
                                    int n_tiles, const int* seq_slot, const int* seq_start, const int* seq_q_len,
                                    const int* q_start_loc, float* out, float* part_o, float* part_ml, int rows, int blocks,
                                    int capacity, int round, int turns, int q_heads, int kv_heads, int head_dim, int page_size,
                                    int window, float scale, int tokens_per_tile) {
    if (n_tiles < 0 || q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads || page_size < 4 ||
        (page_size & (page_size - 1)) || tokens_per_tile < 1 || tokens_per_tile * (q_heads / kv_heads) > kRowsTile ||
        q_row_stride % 4 || table_width < 1 || (tile_seq == nullptr) != (tile_q0 == nullptr) || kv_heads > 16383 ||
        static_cast<long>(tokens_per_tile) * q_heads > 65535 || turns < 0 || turns > 65535 || capacity < 0 || round < 0)
        return CIE_BAD_ARGUMENT;
    if (turns && (!part_o || !part_ml || blocks < 1 || rows < tokens_per_tile * (q_heads / kv_heads))) return CIE_BAD_ARGUMENT;
    if (capacity && static_cast<long>(n_tiles) * blocks > (1L << 30)) return CIE_BAD_ARGUMENT;
    if (n_tiles == 0) return CIE_OK;
    int shift = 0;
    while ((1 << shift) < page_size) ++shift;
    const Args a{q, q_row_stride, k_pool, v_pool, block_table, table_width, tile_seq, tile_q0, seq_slot, seq_start,
                 seq_q_len, q_start_loc, out, part_o, part_ml, rows, blocks, capacity, round, q_heads, kv_heads, shift, window, scale, tokens_per_tile};
    const int row_tiles = (tokens_per_tile * (q_heads / kv_heads) + 15) / 16;
    hipStream_t s = static_cast<hipStream_t>(stream);
    switch (head_dim) {
        case 32: return run<32>(s, a, n_tiles, row_tiles, turns);
        case 64: return run<64>(s, a, n_tiles, row_tiles, turns);
        case 96: return run<96>(s, a, n_tiles, row_tiles, turns);
        case 128: return run<128>(s, a, n_tiles, row_tiles, turns);
    }
    return CIE_BAD_ARGUMENT;
}

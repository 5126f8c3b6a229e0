// Paged grouped-query attention for prompt portions: eight waves per tile of 128 (token, head) rows.
//
// A workgroup takes one tile (up to 128 rows = tokens_per_tile tokens x the heads of one kv head's group)
// and walks the tile's keys 64 at a time.  The keys and values of those 64 positions are read from the
// cache once per workgroup, by loads that write LDS themselves (1 KB each, 16 bytes a lane), in the order the matrix
// instructions take their operands; every wave then reads them from there.  Two stages of LDS take turns, so that the loads of
// the next 64 keys are under way while a block is worked on, and one barrier a stage frees the one and has the other whole.
// (Carried through registers and stored to LDS by the waves, as far ahead, the pieces held 32 registers and took 12 stores a
// wave and stage: MI355X, us, 2,048 tokens of one prompt, 3B heads 43.6 -> 36.4, behind 14,336 keys 342 -> 270; 777 tokens behind
// 4,000, 7B heads 104 -> 80; 14 heads of 64 dimensions 30.3 -> 24.6.  A third stage changes nothing.)  The products run at a
// raised priority where the head has 128 dimensions: a wave that multiplies goes before the one beside it that does its
// softmax (85 -> 80 and 284 -> 270 of these; with 64 dimensions, half the products, 41.5 -> 44.5: not there).
//
// Wave w owns rows 32 * (w % 4) .. + 31 of the tile and, of each 64 keys, the half w / 4: four waves
// cover the rows, two such sets the keys.  A wave holds 32 rows of the output (64 accumulator registers
// where the head has 128 dimensions), so that two waves fit on a SIMD and the softmax arithmetic of one
// overlaps the matrix products of the other.  The two halves of the keys meet in LDS at the end.
//
// Per block of 32 keys a wave computes, as the other forms do (csrc/attention_mfma.hip):
//   S^T[key, row] = K[key, :] . Q[row, :]     v_mfma_f32_16x16x32_bf16, A = K (from LDS), B = Q (registers)
//   P = 2^(S * scale * log2 e - m)            float32; the reference m of a row moves lazily
//   O[row, d] += P[row, key] * V[key, d]      A = P (registers), B = V^T (from LDS)
//
// Which row of a block's two 16-key products a key is, is free: row m of product kt is key 8 (m / 4) + 4 kt + m % 4 of the 32,
// so that a lane ends with the probabilities of eight neighbouring keys, and takes their values as the cache has them.
//
// LDS layout of one stage (D = head size, C = D / 8 sixteen-byte chunks of a key):
//   keys    64 rows of CS chunk slots (CS = C rounded up to a power of two); chunk c of key k lies in slot
//           c ^ swizzle(k), so that the 16 lanes that read the same chunk of 16 different keys hit 16
//           different groups of banks
//   values  four groups of 16 keys, each D rows of 32 bytes: dimension d's values of the keys, eight a chunk, the two
//           chunks exchanged where d / 8 is odd
#include "attention_args.h"
#include "common.h"

using namespace cie_attention;

namespace {

constexpr int kKeysPerStage = 2 * kKeysPerBlock;  // 64: one block for each half of the waves

// The largest of three or two numbers in one instruction each, and the largest over the four 16-lane rows of a
// wave, written as instructions: the compiler's own maxima first copy every operand onto itself (to quiet
// signalling NaNs, which the hardware's maximum does anyway), three instructions where one does.
__device__ __forceinline__ float max3(float a, float b, float c) {
    float out;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(out) : "v"(a), "v"(b), "v"(c));
    return out;
}

__device__ __forceinline__ float max2(float a, float b) {
    float out;
    asm("v_max_f32 %0, %1, %2" : "=v"(out) : "v"(a), "v"(b));
    return out;
}

__device__ __forceinline__ float rows_max_lean(float v) {
    swap_pair_t a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = max2(__uint_as_float(a[0]), __uint_as_float(a[1]));
    swap_pair_t b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return max2(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

template <int D>
struct PromptLayout {
    static constexpr int C = D / 8;
    static constexpr int CS = C <= 4 ? 4 : C <= 8 ? 8 : C <= 16 ? 16 : 32;
    static constexpr int kKeyBytes = kKeysPerStage * CS * 16;
    static constexpr int kValueBlockBytes = D * 64;
    static constexpr int kStageBytes = kKeyBytes + 2 * kValueBlockBytes;
    static constexpr int kKeyPieces = CS / 4, kValuePieces = D / 32;  // loads of 1 KB that a group of 16 keys takes
    static constexpr int kKeysPerPiece = 64 / CS;
    // the swizzle of a key's chunk slots: over the 16 keys that one product reads (bits 0, 1, 3 and 4 of their places take
    // every value), the same chunk lands in 16 different sixteen-byte columns of the 256 bytes that the banks span
    __device__ static __forceinline__ int key_swizzle(int k) {
        if (CS >= 16) return (k & 3) | (k >> 3 & 3) << 2;
        if (CS == 8) return (k >> 1 & 1) | (k >> 3 & 3) << 1;
        return k >> 3 & 3;
    }
};

typedef __attribute__((address_space(3))) void* lds_pointer;
// (16 bytes as one value.  Read from a stage as a uint4, a structure, they made the compiler wait for every load that writes LDS
// in front of each block's first read.)
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// Behind it all of this wave's loads but the youngest kYounger are in LDS, and what it read there is in registers.
template <int kYounger>
__device__ __forceinline__ void wait_for_loads() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kYounger) : "memory");
}

// WAVES = 8: tiles of 128 rows; WAVES = 4: the same with tiles of 64 rows, two such workgroups to a compute unit,
// which then walk their keys independently of each other (one's matrix products beside the other's softmax).
template <int D, int WAVES>
__global__ void __launch_bounds__(64 * WAVES, WAVES == 4 ? 2 : 1) paged_attention_prompt_kernel(AttentionArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)  // (the host's pass has no type for a buffer's description)
    using L = PromptLayout<D>;
    constexpr int NK = D / 32;
    constexpr int ND = D / 16;
    constexpr int RT = 2;  // 16-row tiles of a wave
    constexpr int QUARTERS = WAVES / 2;        // sets of 32 rows of the tile
    constexpr int kTileRows = 32 * QUARTERS;
    extern __shared__ __align__(1024) unsigned char lds[];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int quarter = wave % QUARTERS;   // which 32 rows of the tile
    const int half = wave / QUARTERS;      // which 32 of each 64 keys
    const int r = lane & 15;
    const int g = lane >> 4;

    // tiles of a kv head go to that head's XCDs where the heads divide the 8 XCDs (see attention_mfma.hip)
    int tile_index, kv_head;
    if (a.xcds_per_head > 0) {
        const int xcd = blockIdx.x % kXcds;
        kv_head = xcd % a.kv_heads;
        tile_index = (blockIdx.x / kXcds) * a.xcds_per_head + xcd / a.kv_heads;
    } else {
        kv_head = blockIdx.x % a.kv_heads;
        tile_index = blockIdx.x / a.kv_heads;
    }
    if (tile_index >= a.n_tiles) return;  // padding of the grid; the whole workgroup leaves
    // The last tiles of a prompt see the most keys: they start first.  Where two workgroups share a compute
    // unit (WAVES = 4) the first half of the launch are the longest tiles in falling order and the second half
    // the shortest in rising order: the hardware fills the units' second places in the order of the first, so
    // that a unit gets a long tile and a short one, every unit about as many keys.
    int tile = a.n_tiles - 1 - tile_index;
    if (WAVES == 4 && tile_index >= (a.n_tiles + 1) / 2) tile = tile_index - (a.n_tiles + 1) / 2;
    const int group = a.q_heads / a.kv_heads;
    const int seq = a.tile_seq ? a.tile_seq[tile] : tile;
    const int q0 = a.tile_seq ? a.tile_q0[tile] : 0;
    const int start = a.seq_start[seq];
    const int n_tok = min(a.tokens_per_tile, a.seq_q_len[seq] - q0);
    const int n_rows = n_tok * group;
    const int first_row_token = a.q_start_loc[seq] + q0;
    const int page_mask = (1 << a.page_shift) - 1;
    const int* table = a.block_table + static_cast<size_t>(a.seq_slot[seq]) * a.table_width;
    const float scale_log2 = a.scale * 1.44269504088896341f;
    const int hi = start + q0 + n_tok;
    const int lo = (a.window > 0) ? max(0, start + q0 + 1 - a.window) : 0;
    int range_begin = lo & ~(kKeysPerBlock - 1);
    int range_end = hi;
    bool whole = a.n_splits == 1;  // this workgroup sees all the tile's keys and writes its result itself
    if (a.n_splits > 1) {
        int per_split = a.keys_per_split;
        if (a.max_context_dev) {
            int most = *a.max_context_dev;
            if (a.window > 0) most = min(most, a.window + 2 * kKeysPerBlock);
            per_split = ((most + a.n_splits - 1) / a.n_splits + kKeysPerBlock - 1) & ~(kKeysPerBlock - 1);
        }
        if (a.whole_in_first_share && all_in_first_share(range_begin, hi, per_split)) {
            if (blockIdx.y > 0) return;  // (the merge leaves such a tile alone too)
            whole = true;
        } else {
            range_begin += blockIdx.y * per_split;
            range_end = min(hi, range_begin + per_split);
            if (range_begin >= range_end) {  // no keys in this share: its statistics say so, its sums are never read
                float* pml = a.part_ml + ((static_cast<size_t>(tile) * a.kv_heads + kv_head) * a.n_splits + blockIdx.y) * kTileRows * 2;
                if (threadIdx.x < kTileRows) {
                    pml[threadIdx.x * 2] = -INFINITY;
                    pml[threadIdx.x * 2 + 1] = 0.f;
                }
                return;
            }
        }
    }
    const int last_group = (hi - 1) & ~15;  // the last 16 keys that have a page

    // ---- this wave's rows
    const int wave_row0 = quarter * 32;
    const int wave_rows = min(32, n_rows - wave_row0);  // <= 0: the wave has no rows, it only helps to load
    const int wave_first_pos = start + q0 + wave_row0 / group;
    const int wave_last_pos = start + q0 + (wave_row0 + max(wave_rows, 1) - 1) / group;
    uint4 qf[RT][NK];
    int row_pos[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int row = wave_row0 + rt * 16 + r;
        const bool valid = row < n_rows;
        const int tok = row / group;
        const int head = row - tok * group;
        row_pos[rt] = valid ? start + q0 + tok : -1;
        const bf16_t* q_row = a.q + static_cast<size_t>(first_row_token + tok) * a.q_row_stride +
                              static_cast<size_t>(kv_head * group + head) * D + g * 8;
#pragma unroll
        for (int j = 0; j < NK; ++j)  // product j takes dimensions (j*4 + g)*8 .. +7 of both operands
            qf[rt][j] = valid ? *reinterpret_cast<const uint4*>(q_row + j * 32) : uint4{0, 0, 0, 0};
    }
    // The sums of a row's probabilities come from the matrix cores too: one more product of P with a column
    // of ones.  They are then the sums of the very (rounded) probabilities that weigh the values, they lie in
    // the accumulators' layout (lane group g holds rows g*4 .. +3), and the vector unit, which is the busy
    // one here, adds nothing.
    float m_run[RT];
    floatx4 o[RT][ND], l_acc[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        m_run[rt] = -INFINITY;
        l_acc[rt] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int dt = 0; dt < ND; ++dt) o[rt][dt] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
    const bf16x8 ones = __builtin_bit_cast(bf16x8, (uint4{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u}));

    // ---- this wave's share of the loads.  A stage is four groups of 16 keys (each within one page): wave w fetches group
    // w % 4, with eight waves every second of its pieces, so that which page its loads read is one number.  A lane's place in
    // LDS is given (16 bytes behind its neighbour's), so it picks the chunk that belongs there.
    constexpr int kSharers = WAVES / 4, kPieces = L::kKeyPieces + L::kValuePieces;
    const int loads_group = wave % 4, loads_first = wave / 4;
    unsigned key_from[L::kKeyPieces];  // bytes from the group's first key
#pragma unroll
    for (int i = 0; i < L::kKeyPieces; ++i) {
        const int key = i * L::kKeysPerPiece + lane / L::CS;
        const int chunk = (lane % L::CS) ^ L::key_swizzle(loads_group * 16 + key);
        key_from[i] = (key * D + (chunk < L::C ? chunk : 0) * 8) * 2;  // (a slot that holds no chunk is never read)
    }
    const unsigned value_from = ((lane / 2 << a.page_shift) + ((lane % 2) ^ (lane >> 4 & 1)) * 8) * 2;

    typedef const __attribute__((address_space(4))) int* const_int_ptr;
    const const_int_ptr table_c = (const_int_ptr)(uintptr_t)table;
    // the page of the 16 keys from `first` on (clamped to keys that have a page; what lies past the end is
    // masked where it is used)
    auto page_of = [&](int first) {
        return table_c[__builtin_amdgcn_readfirstlane(min(first, last_group) >> a.page_shift)];
    };
    auto page_at = [&](int kb) { return page_of(kb + loads_group * 16); };  // ... of this wave's group of the stage at key kb
    auto fetch = [&](int kb, int page, int stage) __attribute__((always_inline)) {
        const int first = min(kb + loads_group * 16, last_group);
        const size_t page_head = static_cast<size_t>(page) * a.kv_heads + kv_head;
        const __amdgpu_buffer_rsrc_t keys = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<bf16_t*>(a.k_pool + ((page_head << a.page_shift) + (first & page_mask)) * D), 0, 0xffffffffu, 0x00027000);
        const __amdgpu_buffer_rsrc_t values = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<bf16_t*>(a.v_pool + (page_head * D << a.page_shift) + (first & page_mask)), 0, 0xffffffffu, 0x00027000);
        unsigned char* key_to = lds + stage * L::kStageBytes + loads_group * (16 * L::CS * 16);
        unsigned char* value_to = lds + stage * L::kStageBytes + L::kKeyBytes + loads_group * (D * 32);
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            if (kSharers == 2 && i % 2 != loads_first) continue;
            if (i < L::kKeyPieces)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(keys, (lds_pointer)(key_to + i * 1024), 16, key_from[i < L::kKeyPieces ? i : 0], 0, 0, 0);
            else
                __builtin_amdgcn_raw_ptr_buffer_load_lds(values, (lds_pointer)(value_to + (i - L::kKeyPieces) * 1024), 16, value_from,
                                                         (i - L::kKeyPieces) * 64 << a.page_shift, 0, 0);
        }
    };

    // ---- a lane's constant parts of its operand addresses in a stage
    // (row r of product kt is key 8 (r / 4) + r % 4 + 4 kt of the half; bit 2 of a key's place is not in its swizzle)
    const int k_read = (half * 32 + r / 4 * 8 + r % 4) * L::CS * 16;  // + kt * 4 * CS * 16, + swizzled chunk
    const int k_sw = L::key_swizzle(half * 32 + r / 4 * 8 + r % 4);
    const int v_read = L::kKeyBytes + (half * 2 + g / 2) * (D * 32) + r * 32 + ((g % 2) ^ (r >> 3)) * 16;  // + dt * 512

    const int n_iter = (range_end - range_begin + kKeysPerStage - 1) / kKeysPerStage;
    int page = 0;
    if (n_iter > 0) {
        const int first_page = page_at(range_begin);
        page = page_at(range_begin + kKeysPerStage);
        fetch(range_begin, first_page, 0);
        if (n_iter > 1) {
            fetch(range_begin + kKeysPerStage, page, 1);
            wait_for_loads<kPieces / kSharers>();
        } else {
            wait_for_loads<0>();
        }
        asm volatile("s_barrier" ::: "memory");
    }

    for (int it = 0; it < n_iter; ++it) {
        const int kb = range_begin + it * kKeysPerStage + half * kKeysPerBlock;  // this wave's 32 keys
        const unsigned char* stage = lds + (it & 1) * L::kStageBytes;
        // the page of the stage after next, asked for early: the loads that need it come a whole block later
        if (it + 2 < n_iter) page = page_at(range_begin + (it + 2) * kKeysPerStage);
        if (wave_rows > 0 && kb < range_end && kb <= wave_last_pos) {
            // ---- S^T = K . Q^T for two 16-key tiles
            floatx4 s[RT][2];
            if constexpr (D > 64) __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
                u32x4 kf[NK];
#pragma unroll
                for (int j = 0; j < NK; ++j)
                    kf[j] = *reinterpret_cast<const u32x4*>(stage + k_read + kt * (4 * L::CS * 16) +
                                                            (((j * 4 + g) ^ k_sw) << 4));
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int j = 0; j < NK; ++j)
                        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, kf[j]),
                                                                      __builtin_bit_cast(bf16x8, qf[rt][j]), acc, 0, 0, 0);
                    s[rt][kt] = acc;
                }
            }
            if constexpr (D > 64) __builtin_amdgcn_s_setprio(0);
            // ---- the block's values: asked for now, used after the softmax arithmetic
            u32x4 vf[ND];
#pragma unroll
            for (int dt = 0; dt < ND; ++dt) vf[dt] = *reinterpret_cast<const u32x4*>(stage + v_read + dt * 512);
            // ---- running maxima; masks only in blocks that reach a row's edge
            const bool edge = kb + kKeysPerBlock - 1 > wave_first_pos || kb + kKeysPerBlock > range_end ||
                              (a.window > 0 && kb < wave_last_pos + 1 - a.window);
            // A row's reference moves only if one of its scores passes it by the margin, and each of the row's four
            // lanes can tell that of its own eight scores: the common block needs no maximum across lanes at all.
            float own_max[RT];
            bool moved = false;
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                if (edge) {
                    const int pos = min(row_pos[rt], range_end - 1);  // (a row that does not exist has -1: nothing seen)
                    const int row_lo = (a.window > 0) ? row_pos[rt] + 1 - a.window : 0;
                    const int first_key = kb + g * 8;
#pragma unroll
                    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int key = first_key + kt * 4 + i;
                            if (!(key <= pos && key >= row_lo)) s[rt][kt][i] = -INFINITY;
                        }
                }
                own_max[rt] = max3(max3(s[rt][0][0], s[rt][0][1], s[rt][0][2]),
                                   max3(s[rt][0][3], s[rt][1][0], s[rt][1][1]),
                                   max3(s[rt][1][2], s[rt][1][3], s[rt][1][3]));
                moved = moved || own_max[rt] * scale_log2 > m_run[rt] + kLazyRescale;  // (the scale is positive)
            }
            if (__any(moved)) {
                // some row's reference moves (rare once the first blocks have set every row's scale): what the
                // row has summed so far is scaled down to the new reference
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    const float block_max = rows_max_lean(own_max[rt]) * scale_log2;  // maxima are kept in scaled base-2 units
                    const float m_new = (block_max > m_run[rt] + kLazyRescale) ? block_max : m_run[rt];
                    const float m_safe = (m_new == -INFINITY) ? 0.f : m_new;
                    const float alpha = __builtin_amdgcn_exp2f(m_run[rt] - m_safe);  // m_run = -inf: 0, and the sums are 0 anyway
                    m_run[rt] = m_new;
                    float alpha_o[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) alpha_o[i] = __shfl(alpha, g * 4 + i, kWave);
#pragma unroll
                    for (int i = 0; i < 4; ++i) l_acc[rt][i] *= alpha_o[i];
#pragma unroll
                    for (int dt = 0; dt < ND; ++dt)
#pragma unroll
                        for (int i = 0; i < 4; ++i) o[rt][dt][i] *= alpha_o[i];
                }
            }
            // ---- probabilities (one fused multiply-add and one exp2 each), then O += P . V and l += P . 1
            bf16x8 p_frag[RT];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const float m_ref = (m_run[rt] == -INFINITY) ? 0.f : m_run[rt];
                uint32_t pw[4];
#pragma unroll
                for (int kt = 0; kt < 2; ++kt) {
                    const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[rt][kt][0], scale_log2, -m_ref));
                    const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[rt][kt][1], scale_log2, -m_ref));
                    const float p2 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[rt][kt][2], scale_log2, -m_ref));
                    const float p3 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[rt][kt][3], scale_log2, -m_ref));
                    pw[kt * 2] = pack_bf16(p0, p1);
                    pw[kt * 2 + 1] = pack_bf16(p2, p3);
                }
                p_frag[rt] = __builtin_bit_cast(bf16x8, (uint4{pw[0], pw[1], pw[2], pw[3]}));
            }
            if constexpr (D > 64) __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
                l_acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p_frag[rt], ones, l_acc[rt], 0, 0, 0);
#pragma unroll
            for (int dt = 0; dt < ND; ++dt)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
                    o[rt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p_frag[rt], __builtin_bit_cast(bf16x8, vf[dt]),
                                                                        o[rt][dt], 0, 0, 0);
        }
        __builtin_amdgcn_s_setprio(0);
        // ---- the next stage has arrived by now (and whoever reads this one has read it): ask for the one after
        wait_for_loads<0>();
        asm volatile("s_barrier" ::: "memory");
        if (it + 2 < n_iter) fetch(range_begin + (it + 2) * kKeysPerStage, page, it & 1);
    }

    // ---- the two halves of the keys meet: the upper waves hand their sums to the lower ones through LDS,
    // one 16-row tile at a time (the references of the rows, then ND tiles of the output and one of the
    // probabilities' sums, each as the 4 x 64 numbers the lanes hold)
    float* lds_m = reinterpret_cast<float*>(lds);                    // [quarters][16 rows]
    float* lds_o = reinterpret_cast<float*>(lds) + QUARTERS * 16;    // [quarters][(ND + 1) * 4][64 lanes]
    constexpr int kMeetTile = (ND + 1) * 4;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        if (rt > 0) __syncthreads();  // the tile before has been read
        if (half == 1) {
            if (g == 0) lds_m[quarter * 16 + r] = m_run[rt];
#pragma unroll
            for (int dt = 0; dt < ND; ++dt)
#pragma unroll
                for (int i = 0; i < 4; ++i) lds_o[(quarter * kMeetTile + dt * 4 + i) * kWave + lane] = o[rt][dt][i];
#pragma unroll
            for (int i = 0; i < 4; ++i) lds_o[(quarter * kMeetTile + ND * 4 + i) * kWave + lane] = l_acc[rt][i];
        }
        __syncthreads();
        if (half == 1 || wave_rows <= 0) continue;
        const float m_other = lds_m[quarter * 16 + r];
        const float m_all = fmaxf(m_run[rt], m_other);
        const float m_safe = (m_all == -INFINITY) ? 0.f : m_all;
        const float w_own = __builtin_amdgcn_exp2f(m_run[rt] - m_safe);
        const float w_other = __builtin_amdgcn_exp2f(m_other - m_safe);
        float w_own_o[4], w_other_o[4], l[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {  // from the lane of row r to the lanes that hold row g*4 + i
            w_own_o[i] = __shfl(w_own, g * 4 + i, kWave);
            w_other_o[i] = __shfl(w_other, g * 4 + i, kWave);
            l[i] = l_acc[rt][i] * w_own_o[i] + lds_o[(quarter * kMeetTile + ND * 4 + i) * kWave + lane] * w_other_o[i];
        }
#pragma unroll
        for (int dt = 0; dt < ND; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                o[rt][dt][i] = o[rt][dt][i] * w_own_o[i] +
                               lds_o[(quarter * kMeetTile + dt * 4 + i) * kWave + lane] * w_other_o[i];
        if (!whole) {  // this share's sums and statistics for the merge kernel
            const size_t unit = (static_cast<size_t>(tile) * a.kv_heads + kv_head) * a.n_splits + blockIdx.y;
            float* po = a.part_o + unit * kTileRows * D;
            float* pml = a.part_ml + unit * kTileRows * 2;
            if (g == 0) pml[(wave_row0 + rt * 16 + r) * 2] = m_all;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = wave_row0 + rt * 16 + g * 4 + i;
                if (r == 0) pml[row * 2 + 1] = l[i];
#pragma unroll
                for (int dt = 0; dt < ND; ++dt) po[static_cast<size_t>(row) * D + dt * 16 + r] = o[rt][dt][i];
            }
            continue;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = wave_row0 + rt * 16 + g * 4 + i;
            if (row < n_rows) {
                const int tok = row / group;
                const int head = row - tok * group;
                bf16_t* dst = a.out + static_cast<size_t>(first_row_token + tok) * a.q_heads * D +
                              static_cast<size_t>(kv_head * group + head) * D;
                const float inv = 1.0f / l[i];
#pragma unroll
                for (int dt = 0; dt < ND; ++dt) dst[dt * 16 + r] = from_float<bf16_t>(o[rt][dt][i] * inv);
            }
        }
    }
#endif
}

template <int D, int WAVES>
int launch(hipStream_t s, const AttentionArgs& a) {
    using L = PromptLayout<D>;
    // the stages, or the meeting place of the two halves at the end, whichever is larger
    constexpr int kMeetBytes = ((WAVES / 2) * 16 + (WAVES / 2) * ((D / 16 + 1) * 4) * kWave) * 4;
    constexpr int kLdsBytes = 2 * L::kStageBytes > kMeetBytes ? 2 * L::kStageBytes : kMeetBytes;
    static_assert(kLdsBytes <= 64 * 1024, "a workgroup's LDS without asking for more");
    const dim3 grid = a.xcds_per_head > 0
                          ? dim3(kXcds * ((a.n_tiles + a.xcds_per_head - 1) / a.xcds_per_head), a.n_splits)
                          : dim3(static_cast<unsigned>(a.n_tiles) * a.kv_heads, a.n_splits);
    paged_attention_prompt_kernel<D, WAVES><<<grid, 64 * WAVES, kLdsBytes, s>>>(a);
    return cie_after_launch();
}

}  // namespace

namespace cie_attention {

int launch_prompt_form(hipStream_t stream, const AttentionArgs& a, int head_dim, int waves) {
    if (waves == 4) {
        switch (head_dim) {
            case 32: return launch<32, 4>(stream, a);
            case 64: return launch<64, 4>(stream, a);
            case 96: return launch<96, 4>(stream, a);
            case 128: return launch<128, 4>(stream, a);
            default: return CIE_BAD_ARGUMENT;
        }
    }
    switch (head_dim) {
        case 32: return launch<32, 8>(stream, a);
        case 64: return launch<64, 8>(stream, a);
        case 96: return launch<96, 8>(stream, a);
        case 128: return launch<128, 8>(stream, a);
        default: return CIE_BAD_ARGUMENT;  // wider heads: a wave's 32 rows of accumulators would not fit
    }
}

}  // namespace cie_attention

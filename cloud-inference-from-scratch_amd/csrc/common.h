// Shared device helpers for the gfx950 kernels: storage types, bf16 conversion,
// wave64 and workgroup reductions, launch-error reporting.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#define CIE_API extern "C" __attribute__((visibility("default")))

// Return codes of every entry point.  0 is success; the Python side turns the
// others into exceptions that name the entry point.
enum {
    CIE_OK = 0,
    CIE_BAD_ARGUMENT = 1,   // a size or option the kernel does not take
    CIE_LAUNCH_FAILED = 2,  // hipGetLastError() after the launch
    CIE_TOO_LARGE = 3,      // more than the fixed scratch memory of an entry point that allocates nothing holds
    CIE_SETUP_FAILED = 4,   // the library's own device memory could not be found on this device
};

constexpr int kWave = 64;

// Activation / weight storage.  dtype codes used across the C ABI.
enum { CIE_F32 = 0, CIE_BF16 = 1 };

struct bf16_t {
    uint16_t bits;
};

__device__ __forceinline__ float to_float(float x) { return x; }
__device__ __forceinline__ float to_float(bf16_t x) {
    return __uint_as_float(static_cast<uint32_t>(x.bits) << 16);
}

// Round to nearest even; NaN stays NaN.
__device__ __forceinline__ uint16_t bf16_bits_from_float(float x) {
    uint32_t u = __float_as_uint(x);
    if ((u & 0x7fffffffu) > 0x7f800000u) return static_cast<uint16_t>((u >> 16) | 0x0040u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return static_cast<uint16_t>(u >> 16);
}

// Two floats to two bfloat16 in one word (low half first), round to nearest even: on gfx950 this is
// the v_cvt_pk_bf16_f32 instruction.
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    typedef float floatx2_t __attribute__((ext_vector_type(2)));
    const floatx2_t v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}

template <typename T>
__device__ __forceinline__ T from_float(float x);
template <>
__device__ __forceinline__ float from_float<float>(float x) {
    return x;
}
template <>
__device__ __forceinline__ bf16_t from_float<bf16_t>(float x) {
    bf16_t r;
    r.bits = static_cast<uint16_t>(pack_bf16(x, 0.f) & 0xffffu);
    return r;
}

// The lane's partner N (1, 2, 4 or 8) lanes further round its row of 16, in the vector ALU.
template <int N>
__device__ __forceinline__ float turned(float v) {
    return __uint_as_float(static_cast<uint32_t>(
        __builtin_amdgcn_update_dpp(0, static_cast<int>(__float_as_uint(v)), 0x120 + N, 0xf, 0xf, true)));
}

// The sum over a wave, in every lane: lanes 32, 16, 8, 4, 2 and 1 apart in turn.  Rows are swapped, and within a row turned
// (what lanes 8 apart share repeats after 8, and so on), without a round trip through LDS a step: 12 instructions where six
// exchanges through LDS, each waiting for the one before, took some 0.3 us of a norm's 4.7.
__device__ __forceinline__ float wave_sum(float v) {
    typedef unsigned pair_t __attribute__((ext_vector_type(2)));
    const pair_t halves = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(halves[0]) + __uint_as_float(halves[1]);
    const pair_t rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(rows[0]) + __uint_as_float(rows[1]);
    v += turned<8>(v);
    v += turned<4>(v);
    v += turned<2>(v);
    return v + turned<1>(v);
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int offset = kWave / 2; offset > 0; offset >>= 1) v = fmaxf(v, __shfl_xor(v, offset, kWave));
    return v;
}

// Eight neighbouring numbers as float32, in 16-byte pieces.
typedef float eight_t __attribute__((ext_vector_type(8)));
typedef float half_eight_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ eight_t load_eight(const float* p) {
    const half_eight_t lo = reinterpret_cast<const half_eight_t*>(p)[0], hi = reinterpret_cast<const half_eight_t*>(p)[1];
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}
__device__ __forceinline__ void store_eight(float* p, eight_t v) {
    reinterpret_cast<half_eight_t*>(p)[0] = __builtin_shufflevector(v, v, 0, 1, 2, 3);
    reinterpret_cast<half_eight_t*>(p)[1] = __builtin_shufflevector(v, v, 4, 5, 6, 7);
}
// ... and the sum of their squares, in the one order that whoever makes a norm uses.
__device__ __forceinline__ float sum_of_squares(eight_t x) {
    return ((x[0] * x[0] + x[1] * x[1]) + (x[2] * x[2] + x[3] * x[3])) + ((x[4] * x[4] + x[5] * x[5]) + (x[6] * x[6] + x[7] * x[7]));
}

// Reductions over the four 16-lane rows of a wave (lanes r, r+16, r+32, r+48; every lane gets the
// result) with gfx950's row-swap instructions, which stay in the vector ALU: no round trip through LDS.
// v_permlane16_swap(a, b) exchanges the odd rows of a with the even rows of b; v_permlane32_swap(a, b)
// the upper half of a with the lower half of b.  Fed the same value twice, the two results hold, in
// every lane, the lane's own value and its partner's.
typedef unsigned swap_pair_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float rows_max(float v) {
    swap_pair_t a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    swap_pair_t b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

__device__ __forceinline__ float rows_sum(float v) {
    swap_pair_t a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    swap_pair_t b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// A 4 x 4 transposition over the four 16-lane rows of a wave: row q comes with x[4 q + j] in v[j] and leaves with
// x[4 t + q] in v[t].
typedef float quarter_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ quarter_t across_quarters(quarter_t v) {
    const swap_pair_t a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[0]), __float_as_uint(v[2]), false, false);
    const swap_pair_t b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[1]), __float_as_uint(v[3]), false, false);
    const swap_pair_t c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
    const swap_pair_t d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    return quarter_t{__uint_as_float(c[0]), __uint_as_float(c[1]), __uint_as_float(d[0]), __uint_as_float(d[1])};
}

// Sum over a workgroup of up to 16 waves; every thread gets the result.
// `scratch` is at least 16 floats of LDS; the call contains barriers.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
    const int lane = threadIdx.x % kWave;
    const int wave = threadIdx.x / kWave;
    const int waves = (blockDim.x + kWave - 1) / kWave;
    v = wave_sum(v);
    __syncthreads();
    if (lane == 0) scratch[wave] = v;
    __syncthreads();
    float total = 0.f;
    for (int w = 0; w < waves; ++w) total += scratch[w];
    return total;
}

__device__ __forceinline__ float block_max(float v, float* scratch) {
    const int lane = threadIdx.x % kWave;
    const int wave = threadIdx.x / kWave;
    const int waves = (blockDim.x + kWave - 1) / kWave;
    v = wave_max(v);
    __syncthreads();
    if (lane == 0) scratch[wave] = v;
    __syncthreads();
    float total = scratch[0];
    for (int w = 1; w < waves; ++w) total = fmaxf(total, scratch[w]);
    return total;
}

static inline int cie_after_launch() {
    return hipGetLastError() == hipSuccess ? CIE_OK : CIE_LAUNCH_FAILED;
}

// The float32 stream of a decoder whose layers add their branches in parallel and whose next input is a
// weighted average over the depth: one kernel per layer boundary.
//
//   v      = x + mult * (branch_a + branch_b + sum_p parts[p])        (each optional; float32 sum, the parts in order)
//   history[newest] = v                              (what the layer left, before any averaging)
//   v      = sum_j weights[j] * history[j], j < terms (terms = 0: no averaging)
//   stream = v
//   out1   = v / sqrt(mean(v^2) + eps) * gain1       (RMS norms with one gain for all coordinates; each optional)
//   out2   = v / sqrt(mean(v^2) + eps) * gain2
//
// x [rows, hidden] float32; branches and outputs in the activation type; parts [n_parts, rows, hidden] float32 (a branch
// that comes as the parts of a product whose K was cut); history [layers + 1, rows, hidden]
// float32.  One workgroup per row; the row passes through LDS, so hidden * 4 bytes must fit in 64 KB.
#include "common.h"

template <typename T>
__global__ void depth_stream_kernel(const float* __restrict__ x, const T* __restrict__ branch_a,
                                    const T* __restrict__ branch_b, float mult, float* __restrict__ history,
                                    long layer_stride, int newest, const float* __restrict__ weights, int terms,
                                    float* __restrict__ stream, T* __restrict__ out1, float gain1,
                                    T* __restrict__ out2, float gain2, int hidden, float eps,
                                    const float* __restrict__ parts, int n_parts) {
    extern __shared__ float staged[];
    __shared__ float scratch[16];
    const size_t row = static_cast<size_t>(blockIdx.x) * hidden;
    const size_t apart = static_cast<size_t>(gridDim.x) * hidden;
    float sum_sq = 0.f;
    for (int h = threadIdx.x; h < hidden; h += blockDim.x) {
        float v = x[row + h];
        if (branch_a || n_parts) {
            float s = branch_a ? to_float(branch_a[row + h]) : 0.f;
            if (branch_b) s += to_float(branch_b[row + h]);
            for (int p = 0; p < n_parts; ++p) s += parts[p * apart + row + h];
            v = v + mult * s;
        }
        if (newest >= 0) history[static_cast<size_t>(newest) * layer_stride + row + h] = v;
        if (terms > 0) {
            // (the loads of the earlier layers' rows do not depend on one another: none stands behind a condition,
            // so that they travel together; the row just made comes from its register, last)
            float acc = 0.f;
            const float* past = history + row + h;
            const int own = (newest >= 0 && newest < terms) ? newest : terms;
#pragma unroll 4
            for (int j = 0; j < own; ++j) acc = fmaf(weights[j], past[static_cast<size_t>(j) * layer_stride], acc);
#pragma unroll 4
            for (int j = own + 1; j < terms; ++j) acc = fmaf(weights[j], past[static_cast<size_t>(j) * layer_stride], acc);
            if (own < terms) acc = fmaf(weights[own], v, acc);
            v = acc;
        }
        if (stream) stream[row + h] = v;
        staged[h] = v;
        sum_sq += v * v;
    }
    if (!out1 && !out2) return;
    const float total = block_sum(sum_sq, scratch);
    const float inv = 1.0f / sqrtf(total / static_cast<float>(hidden) + eps);
    for (int h = threadIdx.x; h < hidden; h += blockDim.x) {
        const float unit = staged[h] * inv;
        if (out1) out1[row + h] = from_float<T>(unit * gain1);
        if (out2) out2[row + h] = from_float<T>(unit * gain2);
    }
}

// The same with four neighbouring numbers a thread, for rows whose pieces of 16 bytes lie on 16-byte lines.  What bounds it
// is the memory's rate over the earlier layers' rows (a boundary in the middle of 13 reads some 7 of them), and a thread
// has to keep enough of them on their way: up to eight rows' pieces are asked for before the first is used.  Measured (a
// boundary in the middle of 12 layers of 2,048, us, single numbers -> this): 1,999 rows 64 -> 34 (5.8 TB/s),
// 8 rows 6.8 -> 5.1, and 5.3 where the feed-forward comes in eight parts.
typedef float four_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ four_t load_four(const float* p) { return *reinterpret_cast<const four_t*>(p); }
__device__ __forceinline__ four_t load_four(const bf16_t* p) {
    const uint2 raw = *reinterpret_cast<const uint2*>(p);
    return four_t{__uint_as_float(raw.x << 16), __uint_as_float(raw.x & 0xffff0000u), __uint_as_float(raw.y << 16),
                  __uint_as_float(raw.y & 0xffff0000u)};
}
__device__ __forceinline__ void store_four(float* p, four_t v) { *reinterpret_cast<four_t*>(p) = v; }
__device__ __forceinline__ void store_four(bf16_t* p, four_t v) {
    *reinterpret_cast<uint2*>(p) = uint2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
}

// (kAhead earlier rows' pieces at once: eight for few rows, where the chain of loads is the time; four for many, whose
// other workgroups fill the wait: 1,999 rows take 34 us with four and 35 with eight)
template <typename T, int kBranches, bool kParts, int kAhead>
__global__ void __launch_bounds__(1024)
depth_stream_vec4_kernel(const float* __restrict__ x, const T* __restrict__ branch_a, const T* __restrict__ branch_b,
                         float mult, float* __restrict__ history, long layer_stride, int newest,
                         const float* __restrict__ weights, int terms, float* __restrict__ stream, T* __restrict__ out1,
                         float gain1, T* __restrict__ out2, float gain2, int hidden, float eps,
                         const float* __restrict__ parts, int n_parts) {
    extern __shared__ four_t staged4[];
    __shared__ float scratch[16];
    const size_t row = static_cast<size_t>(blockIdx.x) * hidden;
    const int own = (newest >= 0 && newest < terms) ? newest : terms;  // the term that this boundary makes itself
    const int earlier = own < terms ? terms - 1 : terms;
    float sum_sq = 0.f;
    for (int h = threadIdx.x * 4; h < hidden; h += blockDim.x * 4) {
        // (no load stands behind a condition, and none may move to its use: each would be waited for alone)
        const float* past = history + row + h;
        four_t v = load_four(x + row + h), branch[kBranches + 1], ahead[kAhead];
        if constexpr (kBranches > 0) branch[0] = load_four(branch_a + row + h);
        if constexpr (kBranches > 1) branch[1] = load_four(branch_b + row + h);
        const auto ask = [&](four_t (&piece)[kAhead], const float* from, size_t apart, int first, int count, int leave_out) {
#pragma unroll
            for (int k = 0; k < kAhead; ++k) {  // (a piece past the last reads the last again and is dropped)
                const int j = min(first + k, count - 1);
                piece[k] = load_four(from + static_cast<size_t>(j + (j >= leave_out)) * apart);
            }
        };
        if (earlier > 0) ask(ahead, past, layer_stride, 0, earlier, own);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (kBranches > 0 || kParts) {
            four_t s = {0.f, 0.f, 0.f, 0.f};
            if constexpr (kBranches > 0) s = branch[0];
            if constexpr (kBranches > 1) s += branch[1];
            if constexpr (kParts) {
                for (int p0 = 0; p0 < n_parts; p0 += kAhead) {
                    four_t piece[kAhead];
                    ask(piece, parts + row + h, static_cast<size_t>(gridDim.x) * hidden, p0, n_parts, n_parts);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int k = 0; k < kAhead; ++k) {
                        const four_t with = s + piece[k];
                        s = p0 + k < n_parts ? with : s;
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = v[i] + mult * s[i];
        }
        if (newest >= 0) store_four(history + static_cast<size_t>(newest) * layer_stride + row + h, v);
        if (terms > 0) {
            // (the terms in the layers' order, the row just made last, from its register)
            four_t acc = {0.f, 0.f, 0.f, 0.f};
            for (int j0 = 0; j0 < earlier; j0 += kAhead) {
                if (j0 > 0) ask(ahead, past, layer_stride, j0, earlier, own);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int k = 0; k < kAhead; ++k) {
                    const int j = min(j0 + k, earlier - 1);
                    const float weight = weights[j + (j >= own)];
                    four_t with;
#pragma unroll
                    for (int i = 0; i < 4; ++i) with[i] = fmaf(weight, ahead[k][i], acc[i]);
                    acc = j0 + k < earlier ? with : acc;
                }
            }
            if (own < terms) {
                const float weight = weights[own];
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[i] = fmaf(weight, v[i], acc[i]);
            }
            v = acc;
        }
        if (stream) store_four(stream + row + h, v);
        staged4[h / 4] = v;
        sum_sq += (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]);
    }
    if (!out1 && !out2) return;
    const float total = block_sum(sum_sq, scratch);
    const float inv = 1.0f / sqrtf(total / static_cast<float>(hidden) + eps);
    for (int h = threadIdx.x * 4; h < hidden; h += blockDim.x * 4) {
        const four_t unit = staged4[h / 4] * inv;
        if (out1) store_four(out1 + row + h, unit * gain1);
        if (out2) store_four(out2 + row + h, unit * gain2);
    }
}

CIE_API int cie_depth_stream(void* stream_handle, int dtype, const float* x, const void* branch_a, const void* branch_b,
                             float mult, float* history, long layer_stride, int newest, const float* weights,
                             int terms, float* stream, void* out1, float gain1, void* out2, float gain2, int rows,
                             int hidden, float eps, const float* parts, int n_parts) {
    if (rows < 0 || hidden <= 0 || hidden * sizeof(float) > 64 * 1024 || !(eps > 0.f) || terms < 0) return CIE_BAD_ARGUMENT;
    if ((newest >= 0 || terms > 0) && (!history || layer_stride < static_cast<long>(rows) * hidden)) return CIE_BAD_ARGUMENT;
    if (terms > 0 && !weights) return CIE_BAD_ARGUMENT;
    if (branch_b && !branch_a) return CIE_BAD_ARGUMENT;
    if (n_parts < 0 || (n_parts && !parts)) return CIE_BAD_ARGUMENT;
    if (rows == 0) return CIE_OK;
    hipStream_t s = static_cast<hipStream_t>(stream_handle);
    const auto aligned = [](const void* p, size_t bytes) { return reinterpret_cast<uintptr_t>(p) % bytes == 0; };
    const auto wide = [&](size_t piece) {  // (a piece of the activation type: four numbers)
        return hidden % 4 == 0 && (!history || layer_stride % 4 == 0) && aligned(x, 16) && aligned(history, 16) &&
               aligned(stream, 16) && aligned(branch_a, piece) && aligned(branch_b, piece) && aligned(out1, piece) &&
               aligned(out2, piece) && aligned(parts, 16);
    };
#define CIE_DEPTH(KERNEL, T, ...)                                                                                     \
    KERNEL<T __VA_OPT__(,) __VA_ARGS__><<<rows, threads, hidden * sizeof(float), s>>>(                                                           \
        x, static_cast<const T*>(branch_a), static_cast<const T*>(branch_b), mult, history, layer_stride, newest,      \
        weights, terms, stream, static_cast<T*>(out1), gain1, static_cast<T*>(out2), gain2, hidden, eps, parts, n_parts)
    // (two branches and parts beside them: the form of single numbers; no layer brings them)
    if (!(n_parts && branch_b) && ((dtype == CIE_F32 && wide(16)) || (dtype == CIE_BF16 && wide(8)))) {
        const int threads = min(1024, (hidden / 4 + kWave - 1) / kWave * kWave);
#define CIE_DEPTH4(T, AHEAD)                                                                                          \
    if (n_parts && branch_a) CIE_DEPTH(depth_stream_vec4_kernel, T, 1, true, AHEAD);                              \
    else if (n_parts) CIE_DEPTH(depth_stream_vec4_kernel, T, 0, true, AHEAD);                                          \
    else if (branch_b) CIE_DEPTH(depth_stream_vec4_kernel, T, 2, false, AHEAD);                                        \
    else if (branch_a) CIE_DEPTH(depth_stream_vec4_kernel, T, 1, false, AHEAD);                                        \
    else CIE_DEPTH(depth_stream_vec4_kernel, T, 0, false, AHEAD)
        if (dtype == CIE_F32 && rows <= 128) {
            CIE_DEPTH4(float, 8);
        } else if (dtype == CIE_F32) {
            CIE_DEPTH4(float, 4);
        } else if (rows <= 128) {
            CIE_DEPTH4(bf16_t, 8);
        } else {
            CIE_DEPTH4(bf16_t, 4);
        }
#undef CIE_DEPTH4
        return cie_after_launch();
    }
    // few rows (a decode step): a row is one workgroup's, so its width is spread over as many threads as it has
    // numbers, up to 1,024; many rows fill the GPU with smaller workgroups
    int threads = hidden >= 1024 ? 256 : 128;
    if (rows <= 128) threads = hidden >= 1024 ? 1024 : hidden >= 512 ? 512 : threads;
    if (dtype == CIE_F32) CIE_DEPTH(depth_stream_kernel, float);
    else if (dtype == CIE_BF16) CIE_DEPTH(depth_stream_kernel, bf16_t);
    else
        return CIE_BAD_ARGUMENT;
#undef CIE_DEPTH
    return cie_after_launch();
}

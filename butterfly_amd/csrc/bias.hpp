// Bias of a butterfly layer: output = multiply(...) + bias, and d_bias = sum of grad over the batch.
//
// The forward kernels that write the final output add the bias themselves (one register per
// element a thread owns, loaded once); bias_add_kernel is the fallback for schedules whose
// last pass runs in a kernel without that hook.  The bias gradient is a column sum of the
// output gradient: row partitions first (each thread adds its rows in ascending order); the
// partitions are then added by reduce_partials_kernel, next to the sums of the factors' gradient,
// in its fixed order -- no atomics, so it is bitwise reproducible.
#pragma once

#include "common.hpp"

namespace bf {

constexpr int kBiasThreads = 256;

struct BiasArgs {
    const void *bias;      // (S, width) dense
    void *out;             // forward fallback: output, updated in place
    const void *grad;      // gradient: (B, S, width) through `view`
    void *partial;         // (nparts, S, stride)
    int64_t stride;        // width rounded up: every slice starts at a multiple of 16 bytes
    StackView view;
    int64_t batch;
    int64_t width;         // columns that exist (output_size)
    int64_t rows_per_part;
    int64_t nparts;
};

// grid: (ceil(width / kBiasThreads), S, row partitions)
template <typename T>
__global__ __launch_bounds__(kBiasThreads) void bias_add_kernel(BiasArgs a)
{
    const int64_t col = (int64_t)blockIdx.x * kBiasThreads + threadIdx.x;
    const int stack = blockIdx.y;
    if (col >= a.width) return;
    const int64_t vc = view_col(stack_view(a.view, stack), col);
    if (vc < 0) return;
    const T b = reinterpret_cast<const T *>(a.bias)[stack * a.width + col];
    T *out = reinterpret_cast<T *>(a.out) + stack * a.view.ss + vc * a.view.se;
    const int64_t r0 = (int64_t)blockIdx.z * a.rows_per_part;
    const int64_t r1 = r0 + a.rows_per_part < a.batch ? r0 + a.rows_per_part : a.batch;
    for (int64_t r = r0; r < r1; ++r) out[r * a.view.sb] = add(out[r * a.view.sb], b);
}

template <typename T>
__global__ __launch_bounds__(kBiasThreads) void bias_grad_partial_kernel(BiasArgs a)
{
    const int64_t col = (int64_t)blockIdx.x * kBiasThreads + threadIdx.x;
    const int stack = blockIdx.y;
    if (col >= a.width) return;
    const int64_t vc = view_col(stack_view(a.view, stack), col);
    const T *g = reinterpret_cast<const T *>(a.grad) + stack * a.view.ss + (vc < 0 ? 0 : vc) * a.view.se;
    const int64_t r0 = (int64_t)blockIdx.z * a.rows_per_part;
    const int64_t r1 = vc < 0 ? r0 : (r0 + a.rows_per_part < a.batch ? r0 + a.rows_per_part : a.batch);
    // four running sums keep four loads in flight; they are combined in a fixed order
    T s0 = zero_of(T()), s1 = s0, s2 = s0, s3 = s0;
    int64_t r = r0;
    for (; r + 4 <= r1; r += 4) {
        s0 = add(s0, g[r * a.view.sb]);
        s1 = add(s1, g[(r + 1) * a.view.sb]);
        s2 = add(s2, g[(r + 2) * a.view.sb]);
        s3 = add(s3, g[(r + 3) * a.view.sb]);
    }
    for (; r < r1; ++r) s0 = add(s0, g[r * a.view.sb]);
    reinterpret_cast<T *>(a.partial)[((int64_t)blockIdx.z * gridDim.y + stack) * a.stride + col] =
        add(add(s0, s1), add(s2, s3));
}

// ---- input gradient of stacks that share their input ------------------------------------------------

constexpr int kSumStacksPerThread = 4;

struct SumStacksArgs {
    const void *in;      // (B, S, width) dense floats
    void *out;           // (B, width) dense
    int64_t width, nstacks, total;   // total = B * width
};

// out[b][c] = sum over the stacks of in[b][s][c], ascending.  Bound by the memory it reads; float4
// accesses where the rows allow them (their width a multiple of four, and every row starts 16-byte
// aligned then).
__global__ __launch_bounds__(256) void sum_stacks_kernel(SumStacksArgs a)
{
    const float *in = reinterpret_cast<const float *>(a.in);
    float *out = reinterpret_cast<float *>(a.out);
    const int64_t step = (int64_t)gridDim.x * 256;
    const bool wide = (a.width & 3) == 0 && (reinterpret_cast<unsigned long long>(a.out) & 15) == 0;
    if (wide) {
        for (int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4; i < a.total; i += step * 4) {
            const int64_t b = i / a.width;
            const float *src = in + b * a.nstacks * a.width + (i - b * a.width);
            float4 t = *reinterpret_cast<const float4 *>(src);
            for (int64_t s = 1; s < a.nstacks; ++s) {
                const float4 v = *reinterpret_cast<const float4 *>(src + s * a.width);
                t.x += v.x; t.y += v.y; t.z += v.z; t.w += v.w;
            }
            *reinterpret_cast<float4 *>(out + i) = t;
        }
        return;
    }
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < a.total; i += step) {
        const int64_t b = i / a.width;
        const float *src = in + b * a.nstacks * a.width + (i - b * a.width);
        float t = src[0];
        for (int64_t s = 1; s < a.nstacks; ++s) t += src[s * a.width];
        out[i] = t;
    }
}

}  // namespace bf

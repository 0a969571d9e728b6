// Definitions of the launchers of launch.hpp.
#pragma once

#include "launch.hpp"

namespace bf {

// paired: the grid holds two workgroups per compute unit (fw_wg_per_cu)
template <int L, int NB, bool INC>
void launch_fast_fw_t(bool cplx, bool paired, const FastFwArgs &a, dim3 grid, hipStream_t stream)
{
    if constexpr (NB == 1) {
        if (cplx && (a.in_real || a.out_real)) {
            hipLaunchKernelGGL((fast_fw_kernel<float2, FastPlan<L, NB, INC>, kFastFwRowsComplex, 4, true>), grid,
                               dim3(kFastThreads), 0, stream, a);
            return;
        }
        if (cplx) {
            hipLaunchKernelGGL((fast_fw_kernel<float2, FastPlan<L, NB, INC>, kFastFwRowsComplex>), grid, dim3(kFastThreads), 0,
                               stream, a);
            return;
        }
    } else if constexpr (fw_pairable(L, INC)) {
        if (paired) {
            hipLaunchKernelGGL((fast_fw_kernel<float, FastPlan<L, NB, INC>, kFastFwRows, 8>), grid, dim3(kFastThreads), 0,
                               stream, a);
            return;
        }
    }
    hipLaunchKernelGGL((fast_fw_kernel<float, FastPlan<L, NB, INC>, kFastFwRows>), grid, dim3(kFastThreads), 0, stream, a);
}

template <int L, int NB, bool INC>
void launch_fast_bw_t(bool cplx, bool two_rows, const FastBwArgs &a, dim3 grid, hipStream_t stream)
{
    if constexpr (NB == 1) {
        if (cplx && (a.x_real || a.g_real)) {
            hipLaunchKernelGGL((fast_bw_kernel<float2, FastPlan<L, NB, INC>, 1, true>), grid, dim3(kFastThreads), 0, stream, a);
            return;
        }
        if (cplx) {
            hipLaunchKernelGGL((fast_bw_kernel<float2, FastPlan<L, NB, INC>>), grid, dim3(kFastThreads), 0, stream, a);
            return;
        }
        if constexpr (L >= 7) {
            if (two_rows) {
                hipLaunchKernelGGL((fast_bw_kernel<float, FastPlan<L, NB, INC>, 2>), grid, dim3(kFastThreads), 0, stream, a);
                return;
            }
        }
    }
    hipLaunchKernelGGL((fast_bw_kernel<float, FastPlan<L, NB, INC>>), grid, dim3(kFastThreads), 0, stream, a);
}

// SpanPlan passes: the LOW kernels on the tiles of a span of q.H high bits.
template <int H, int MODE>
bool launch_span_t(bool cplx, bool backward, bool two_rows, const FastFwArgs *fw, const FastBwArgs *bw, dim3 grid,
                   hipStream_t stream)
{
    using P = SpanPlan<H, MODE>;
    const dim3 block(kFastThreads);
    // which combinations the host plans: float spans of up to kSpanMaxBits bits, complex64 ones of
    // up to kSpanMaxBitsComplex bits and kSpanMaxStagesComplex stages
    constexpr bool for_float = H <= kSpanMaxBits;
    constexpr bool for_complex = H * (MODE == 2 ? 2 : 1) <= kSpanMaxStagesComplex;
    if (cplx) {
        if constexpr (for_complex) {
            // (a span of both sweeps stands in the middle of a schedule: its rows are the workspace's)
            if constexpr (MODE != 2) {
                if (!backward && (fw->in_real || fw->out_real)) {
                    hipLaunchKernelGGL((fast_fw_kernel<float2, P, kFastFwRowsComplex, 4, true>), grid, block, 0, stream, *fw);
                    return true;
                }
                if (backward && (bw->x_real || bw->g_real)) {
                    hipLaunchKernelGGL((fast_bw_kernel<float2, P, 1, true>), grid, block, 0, stream, *bw);
                    return true;
                }
            }
            if (!backward) hipLaunchKernelGGL((fast_fw_kernel<float2, P, kFastFwRowsComplex>), grid, block, 0, stream, *fw);
            else hipLaunchKernelGGL((fast_bw_kernel<float2, P>), grid, block, 0, stream, *bw);
            return true;
        }
        return false;
    }
    if constexpr (for_float) {
        if (!backward) hipLaunchKernelGGL((fast_fw_kernel<float, P, kFastFwRows>), grid, block, 0, stream, *fw);
        else if (two_rows) hipLaunchKernelGGL((fast_bw_kernel<float, P, 2>), grid, block, 0, stream, *bw);
        else hipLaunchKernelGGL((fast_bw_kernel<float, P>), grid, block, 0, stream, *bw);
        return true;
    }
    return false;
}

template <int L, bool INC>
void launch_fast4_t(bool backward, const Fast4Args &a, dim3 grid, hipStream_t stream)
{
    // row groups per backward iteration, which share its barriers: four fit the registers at any
    // length, but two are faster at 1024 (16384 rows, two blocks: 179.5 us a step against 194.8)
    constexpr int RB = L <= 8 ? 4 : 2;
    if (backward) hipLaunchKernelGGL((fast4_bw_kernel<L, INC, RB>), grid, dim3(kFastThreads), 0, stream, a);
    else hipLaunchKernelGGL((fast4_fw_kernel<L, INC, kFast4FwRows>), grid, dim3(kFastThreads), 0, stream, a);
}

template <typename T, int L, bool INC>
void launch_fast4g_t(bool backward, const Fast4GArgs &a, dim3 grid, hipStream_t stream)
{
    constexpr int R = sizeof(T) == 4 ? kFast4FwRows : kFast4GFwRowsComplex;
    // row groups per backward iteration: complex64 what the registers next to the factors allow, float
    // what is faster.  At 512 four, where a workgroup has as many (32768 rows: 94.7 us a step with two, 88.0
    // with four; backward call of 2048 rows 21.2, 21.0), two below that (1024 rows 19.2, 20.5; two blocks 43.8, 46.7)
    constexpr int RB = sizeof(T) == 4 ? (L <= 9 ? 4 : 2) : (L <= 6 ? 2 : 1);
    if constexpr (sizeof(T) == 4 && L == 9) {
        if (backward && a.groups_per_wg < RB) {
            hipLaunchKernelGGL((fast4g_bw_kernel<T, L, INC, 2>), grid, dim3(kFastThreads), 0, stream, a);
            return;
        }
    }
    if (backward) hipLaunchKernelGGL((fast4g_bw_kernel<T, L, INC, RB>), grid, dim3(kFastThreads), 0, stream, a);
    else hipLaunchKernelGGL((fast4g_fw_kernel<T, L, INC, R>), grid, dim3(kFastThreads), 0, stream, a);
}

}  // namespace bf

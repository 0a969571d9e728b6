// Launchers of the register-resident kernels.  Their definitions (launch_impl.hpp) and with them the
// kernels are instantiated in the kernels_*.hip files, which compile in parallel.
#pragma once

#include "fast.hpp"
#include "wide.hpp"
#include "fast4.hpp"
#include "fast4g.hpp"
#include "stream.hpp"

namespace bf {

constexpr int kFastFwRows = 4;         // row groups in flight per forward workgroup
constexpr int kFastFwRowsComplex = 2;  // complex64: half as many (LDS and registers double)
constexpr int kFast4FwRows = 4;
constexpr int kFast4GFwRowsComplex = 2;

// widest span: tiles of 32 consecutive floats (16 consecutive complex64: the same 128 bytes) per
// setting of the span's bits
constexpr int kSpanMaxBits = 5;
constexpr int kSpanMaxBitsComplex = 6;
constexpr int kSpanMaxStagesComplex = 10;  // stages one complex64 span pass can hold (registers + parked factors)

// (The 64-register variant of the two-block forward kernel for 512-element rows, decreasing
// stride first, does not fit its registers -- the build refuses kernels that spill -- so that
// plan always runs one workgroup per CU.)
constexpr bool fw_pairable(int L, bool inc) { return !(L == 9 && !inc); }

template <int L, int NB, bool INC>
void launch_fast_fw_t(bool cplx, bool paired, const FastFwArgs &a, dim3 grid, hipStream_t stream);

template <int L, int NB, bool INC>
void launch_fast_bw_t(bool cplx, bool two_rows, const FastBwArgs &a, dim3 grid, hipStream_t stream);

template <int H, int MODE>
bool launch_span_t(bool cplx, bool backward, bool two_rows, const FastFwArgs *fw, const FastBwArgs *bw, dim3 grid,
                   hipStream_t stream);

// EdgePlan passes (complex64)
void launch_edge(bool inc, const FastFwArgs *fw, const FastBwArgs *bw, dim3 grid, hipStream_t stream);

template <int L, bool INC>
void launch_fast4_t(bool backward, const Fast4Args &a, dim3 grid, hipStream_t stream);

template <typename T, int L, bool INC>
void launch_fast4g_t(bool backward, const Fast4GArgs &a, dim3 grid, hipStream_t stream);

// waves, planes: W and RB of stream_fw_kernel; false where there is no such kernel
bool launch_stream_fw(bool cplx, int waves, int planes, const StreamArgs &a, dim3 grid, hipStream_t stream);

void launch_wide_fw(bool cplx, int L, bool inc, const FastFwArgs &a, dim3 grid, hipStream_t stream);

}  // namespace bf

// Kernels on spans of 4 to 6 high bits (fast.hpp, SpanPlan) and at column tables (EdgePlan).
#include "launch_impl.hpp"

namespace bf {

#define BF_ONE(H, MODE) \
    template bool launch_span_t<H, MODE>(bool, bool, bool, const FastFwArgs *, const FastBwArgs *, dim3, hipStream_t);
#define BF_INST(H) BF_ONE(H, 0) BF_ONE(H, 1) BF_ONE(H, 2)
BF_INST(4) BF_INST(5) BF_INST(6)

void launch_edge(bool inc, const FastFwArgs *fw, const FastBwArgs *bw, dim3 grid, hipStream_t stream)
{
    const dim3 block(kFastThreads);
    if (fw && inc) hipLaunchKernelGGL((fast_fw_kernel<float2, EdgePlan<true>, kFastFwRowsComplex>), grid, block, 0, stream, *fw);
    else if (fw) hipLaunchKernelGGL((fast_fw_kernel<float2, EdgePlan<false>, kFastFwRowsComplex>), grid, block, 0, stream, *fw);
    else if (inc) hipLaunchKernelGGL((fast_bw_kernel<float2, EdgePlan<true>>), grid, block, 0, stream, *bw);
    else hipLaunchKernelGGL((fast_bw_kernel<float2, EdgePlan<false>>), grid, block, 0, stream, *bw);
}

}  // namespace bf

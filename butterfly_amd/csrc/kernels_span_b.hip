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
#define BF_EDGE(INC)                                                                                              \
    do {                                                                                                         \
        using P = EdgePlan<INC>;                                                                                 \
        if (fw && (fw->in_real || fw->out_real))                                                                 \
            hipLaunchKernelGGL((fast_fw_kernel<float2, P, kFastFwRowsComplex, 4, true>), grid, block, 0, stream, *fw);  \
        else if (fw)                                                                                             \
            hipLaunchKernelGGL((fast_fw_kernel<float2, P, kFastFwRowsComplex>), grid, block, 0, stream, *fw);    \
        else if (bw->x_real || bw->g_real)                                                                       \
            hipLaunchKernelGGL((fast_bw_kernel<float2, P, 1, true>), grid, block, 0, stream, *bw);               \
        else                                                                                                     \
            hipLaunchKernelGGL((fast_bw_kernel<float2, P>), grid, block, 0, stream, *bw);                        \
    } while (0)
    if (inc) BF_EDGE(true);
    else BF_EDGE(false);
#undef BF_EDGE
}

}  // namespace bf

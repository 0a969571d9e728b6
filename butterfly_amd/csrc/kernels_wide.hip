// Whole-block forward kernels (wide.hpp).
#include "launch_impl.hpp"

namespace bf {

void launch_wide_fw(bool cplx, int L, bool inc, const FastFwArgs &a, dim3 grid, hipStream_t stream)
{
    const dim3 block(kFastThreads);
    if (L == 12 && inc) hipLaunchKernelGGL((wide_fw_kernel<float, 12, true>), grid, block, 0, stream, a);
    else if (L == 12) hipLaunchKernelGGL((wide_fw_kernel<float, 12, false>), grid, block, 0, stream, a);
    else if (cplx && inc) hipLaunchKernelGGL((wide_fw_kernel<float2, 11, true>), grid, block, 0, stream, a);
    else if (cplx) hipLaunchKernelGGL((wide_fw_kernel<float2, 11, false>), grid, block, 0, stream, a);
    else if (inc) hipLaunchKernelGGL((wide_fw_kernel<float, 11, true>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((wide_fw_kernel<float, 11, false>), grid, block, 0, stream, a);
}

}  // namespace bf

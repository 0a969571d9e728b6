// Factor-streaming base-4 forward kernels (stream.hpp).
#include "launch_impl.hpp"

namespace bf {

template <typename T>
static bool launch_stream_t(int waves, int planes, const StreamArgs &a, dim3 grid, hipStream_t stream)
{
    const dim3 block(64 * waves);
#define BF_STREAM(W, RB)                                                                        \
    if (waves == W && planes == RB) {                                                           \
        hipLaunchKernelGGL((stream_fw_kernel<T, W, RB>), grid, block, 0, stream, a);            \
        return true;                                                                            \
    }
    BF_STREAM(8, 1)
    if constexpr (sizeof(T) == 4) { BF_STREAM(8, 2) BF_STREAM(16, 1) BF_STREAM(16, 2) }
#undef BF_STREAM
    return false;
}

bool launch_stream_fw(bool cplx, int waves, int planes, const StreamArgs &a, dim3 grid, hipStream_t stream)
{
    return cplx ? launch_stream_t<float2>(waves, planes, a, grid, stream)
                : launch_stream_t<float>(waves, planes, a, grid, stream);
}

}  // namespace bf

// Base-4 kernels: aligned float rows (fast4.hpp), the rest up to one workgroup's reach (fast4g.hpp).
#include "launch_impl.hpp"

namespace bf {

#define BF_INST(LL)                                                                          \
    template void launch_fast4_t<LL, false>(bool, const Fast4Args &, dim3, hipStream_t);     \
    template void launch_fast4_t<LL, true>(bool, const Fast4Args &, dim3, hipStream_t);
BF_INST(2) BF_INST(4) BF_INST(6) BF_INST(8) BF_INST(10)

#define BF_INST_G(T, LL)                                                                         \
    template void launch_fast4g_t<T, LL, false>(bool, const Fast4GArgs &, dim3, hipStream_t);    \
    template void launch_fast4g_t<T, LL, true>(bool, const Fast4GArgs &, dim3, hipStream_t);
BF_INST_G(float, 3) BF_INST_G(float, 5) BF_INST_G(float, 7) BF_INST_G(float, 9) BF_INST_G(float, 10)
BF_INST_G(float2, 2) BF_INST_G(float2, 3) BF_INST_G(float2, 4) BF_INST_G(float2, 5) BF_INST_G(float2, 6)
BF_INST_G(float2, 7) BF_INST_G(float2, 8)

}  // namespace bf

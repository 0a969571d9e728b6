// Backward kernels on whole rows and chunks, two blocks (fast.hpp).
#include "launch_impl.hpp"

namespace bf {

#define BF_INST(LL)                                                                                              \
    template void launch_fast_bw_t<LL, 2, false>(bool, bool, const FastBwArgs &, dim3, hipStream_t);           \
    template void launch_fast_bw_t<LL, 2, true>(bool, bool, const FastBwArgs &, dim3, hipStream_t);
BF_INST(1) BF_INST(2) BF_INST(3) BF_INST(4) BF_INST(5) BF_INST(6) BF_INST(7) BF_INST(8) BF_INST(9) BF_INST(10)

}  // namespace bf

// Forward kernels on whole rows and chunks (fast.hpp).
#include "launch_impl.hpp"

namespace bf {

#define BF_ONE(LL, NB, INC) template void launch_fast_fw_t<LL, NB, INC>(bool, bool, const FastFwArgs &, dim3, hipStream_t);
#define BF_INST(LL) BF_ONE(LL, 1, false) BF_ONE(LL, 1, true) BF_ONE(LL, 2, false) BF_ONE(LL, 2, true)
BF_INST(1) BF_INST(2) BF_INST(3) BF_INST(4) BF_INST(5) BF_INST(6) BF_INST(7) BF_INST(8) BF_INST(9) BF_INST(10)

}  // namespace bf

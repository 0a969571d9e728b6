// Kernels on spans of 1 to 3 high bits (fast.hpp, SpanPlan).
#include "launch_impl.hpp"

namespace bf {

#define BF_ONE(H, MODE) \
    template bool launch_span_t<H, MODE>(bool, bool, bool, const FastFwArgs *, const FastBwArgs *, dim3, hipStream_t);
#define BF_INST(H) BF_ONE(H, 0) BF_ONE(H, 1) BF_ONE(H, 2)
BF_INST(1) BF_INST(2) BF_INST(3)

}  // namespace bf

// The Q4_1 forms of the MFMA linear kernel (moe_leaf.hpp), in a file of their
// own: the compiler crashes on some of them with the scheduler that
// moe_mfma.hip is built with.
#include "moe_leaf.hpp"

namespace moe {

hipError_t launch_linear_mfma_q41(const LinearMfmaQ41Args &a, hipStream_t s) {
    if (a.q8) launch_linear_mfma_t<true, 4, true>(a, s);
    else launch_linear_mfma_t<false, 4, true>(a, s);
    return hipGetLastError();
}

}  // namespace moe

// The 64-block form of the fp16-operand gate / up kernel (moe_half.hpp), built
// with the iterative ILP machine scheduler (Makefile).
#include "moe_half.hpp"

namespace moe {

hipError_t launch_gate_up_half_full(const FfnArgs &a, unsigned grid, hipStream_t s) {
    k_gate_up_half<true, false><<<grid, kHtThreads, 0, s>>>(a);
    return hipGetLastError();
}

hipError_t launch_linear_half_full(const LinearMfmaArgs &a, unsigned grid, hipStream_t s) {
    if (a.q8) k_linear_half<true, true><<<grid, kHtThreads, 0, s>>>(a);
    else k_linear_half<true, false><<<grid, kHtThreads, 0, s>>>(a);
    return hipGetLastError();
}

}  // namespace moe

// Launchers of the fp16-operand projections (moe_half.hpp), and every form of
// them but the 64-block one, which moe_half_full.hip builds with its own
// scheduler.
#include "moe_half.hpp"

namespace moe {

hipError_t launch_gate_up_half(const FfnArgs &a, hipStream_t s) {
    if (!a.xhalf) return hipErrorInvalidValue;
    const bool dbg = a.middle_f32 || a.gate_dots || a.up_dots;
    const int nb = a.shape.H / 32;
    const unsigned grid = chunk_grid(a, (a.shape.I / 32 + kGuTiles - 1) / kGuTiles * kSubs, kGuChunkRows / kGuTiles);
    if (nb == kGuMaxBlocks && !dbg) return launch_gate_up_half_full(a, grid, s);
    const auto run = [&](auto kernel) { kernel<<<grid, kHtThreads, 0, s>>>(a); };
    if (nb == kGuMaxBlocks) run(k_gate_up_half<true, true>);
    else if (nb < kGuMaxBlocks) dbg ? run(k_gate_up_half<false, true>) : run(k_gate_up_half<false, false>);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_linear_half(const LinearMfmaArgs &a, hipStream_t s) {
    if (a.nb > kHalfMaxBlocks || !(a.q8 || (a.xq.codes && a.xq.heads))) return hipErrorInvalidValue;
    const unsigned groups = static_cast<unsigned>((a.row_tiles + kHtWaves - 1) / kHtWaves);
    const unsigned grid = (groups + 7u) / 8u * 8u * static_cast<unsigned>(a.col_tiles);
    if (a.nb == kGuMaxBlocks) return launch_linear_half_full(a, grid, s);
    if (a.q8) k_linear_half<false, true><<<grid, kHtThreads, 0, s>>>(a);
    else k_linear_half<false, false><<<grid, kHtThreads, 0, s>>>(a);
    return hipGetLastError();
}

}  // namespace moe

// b2_waves.hpp - the step for Models and States of any dimensions and layout with the worlds per wave fixed at compile
// time (k_step_waves<S>, S = 1, 2, 4, 8: one translation unit each, goi_b2_w*.hip).
#pragma once

#include "b2_launch.hpp"

namespace goi {
namespace {

// What bounds the step is its count of instructions on a world's serial path, so the constants count: with S known,
// every workspace index is a shift, the lane groups (64 / S lanes) and their exchanges unroll, and no debug code is
// carried (launches with debug arrays take k_step). kPlain as in k_step_fixed: revolute joints under the v2.4.1 solver
// and no edge shapes. The dimensions stay run-time values and the State any layout. By the compiler's report the instances
// spill at most 4 vector registers (16 to 32 B of scratch a lane) and 426 to 555 scalar ones, whose reloads are a
// v_readlane each (the 71 leaf pointers and the dimensions; the rig's fixed instance spills 202 to 246); k_step spills
// 121 vector registers (496 B) and 653 scalar ones. When they were added, the 4-body rig with 41 slots (no fixed
// instance): 16,384 worlds, S = 8: 620 -> 497 us a step; 1,024 worlds, S = 1: 435 -> 311 us; the instance for the rig's
// exact dimensions took 450 us at 16,384 worlds.
template <int kS, bool kMulti, bool kPlain>
__global__ void __launch_bounds__(kBlock, 2) k_step_waves(DModel m, Launch L) {
    L.wpw = kS;
    L.dbg = GoiDebug{};
    if (kPlain) {
        m.rev_only = 1;
        m.no_edges = 1;
        L.s.revolute_v24 = 1;
    }
    step_block<kMulti, true>(m, L);  // SolveTOI's views re-derived in each event iteration
}

template <int kS>
hipError_t launch_wave_instance(const DModel& d, const Launch& L, bool multi, bool plain, dim3 grid, size_t lds,
                                hipStream_t st) {
    const dim3 b(kBlock);
    if (!multi && plain) hipLaunchKernelGGL((k_step_waves<kS, false, true>), grid, b, lds, st, d, L);
    else if (!multi) hipLaunchKernelGGL((k_step_waves<kS, false, false>), grid, b, lds, st, d, L);
    else if (plain) hipLaunchKernelGGL((k_step_waves<kS, true, true>), grid, b, lds, st, d, L);
    else hipLaunchKernelGGL((k_step_waves<kS, true, false>), grid, b, lds, st, d, L);
    return hipGetLastError();
}

}  // namespace
}  // namespace goi

// goi_b2_w1.hip - the step for any dimensions, 1 world per wave (b2_waves.hpp).
#define GOI_LANE_ROWS 1  // contact rows a lane holds (b2_step.hpp)
#include "b2_waves.hpp"

namespace goi {

hipError_t launch_step_w1(const DModel& d, const Launch& L, bool multi, bool plain, dim3 grid, size_t lds,
                          hipStream_t st) {
    return launch_wave_instance<1>(d, L, multi, plain, grid, lds, st);
}

}  // namespace goi

// goi_b2_w2.hip - the step for any dimensions, 2 worlds per wave (b2_waves.hpp).
#define GOI_LANE_ROWS 1  // contact rows a lane holds (b2_step.hpp)
#include "b2_waves.hpp"

namespace goi {

hipError_t launch_step_w2(const DModel& d, const Launch& L, bool multi, bool plain, dim3 grid, size_t lds,
                          hipStream_t st) {
    return launch_wave_instance<2>(d, L, multi, plain, grid, lds, st);
}

}  // namespace goi

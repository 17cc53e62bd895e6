// nyl_stagelin32.hip -- the stage kernels of the model variants and of the
// linear upwind branches in single precision.
#include "nyl_stage.h"

namespace nyl {

template <>
hipError_t launch_stage_lin<float>(const Geo &g, const StageArgs<float> &a, int mode, hipStream_t s) {
    NYL_STAGE_GEO(stage_lin, float)
}

}  // namespace nyl

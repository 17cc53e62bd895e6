// nyl_stagelin64.hip -- the stage kernels of the model variants and of the
// linear upwind branches in double precision.
#include "nyl_stage.h"

namespace nyl {

template <>
hipError_t launch_stage_lin<double>(const Geo &g, const StageArgs<double> &a, int mode, hipStream_t s) {
    NYL_STAGE_GEO(stage_lin, double)
}

}  // namespace nyl

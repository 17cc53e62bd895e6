// nyl_stage32.hip -- the stage kernels in single precision (a source of its own:
// the instantiations of the two precisions compile side by side).
#include "nyl_stage.h"

namespace nyl {

template <>
hipError_t launch_stage<float>(const Geo &g, const StageArgs<float> &a, int mode, hipStream_t s) {
    if (a.flags || a.upw_a || a.upw_vf) return launch_stage_lin<float>(g, a, mode, s);
    NYL_STAGE_GEO(stage_les, float)
}

}  // namespace nyl

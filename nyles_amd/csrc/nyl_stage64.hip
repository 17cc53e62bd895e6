// nyl_stage64.hip -- the stage kernels in double precision (a source of its own:
// the instantiations of the two precisions compile side by side).
#include "nyl_stage.h"

namespace nyl {

template <>
hipError_t launch_stage<double>(const Geo &g, const StageArgs<double> &a, int mode, hipStream_t s) {
    if (a.flags || a.upw_a || a.upw_vf) return launch_stage_lin<double>(g, a, mode, s);
    NYL_STAGE_GEO(stage_les, double)
}

}  // namespace nyl

// nyl_stage64.hip -- the stage kernels in double precision (a source of its own:
// the instantiations of the two precisions compile side by side).
#include "nyl_stage.h"

namespace nyl {

template hipError_t launch_stage<double>(const Geo &, const StageArgs<double> &, int, hipStream_t);

}  // namespace nyl

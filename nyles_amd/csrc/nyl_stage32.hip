// nyl_stage32.hip -- the stage kernels in single precision (a source of its own:
// the instantiations of the two precisions compile side by side).
#include "nyl_stage.h"

namespace nyl {

template hipError_t launch_stage<float>(const Geo &, const StageArgs<float> &, int, hipStream_t);

}  // namespace nyl

// cbm_run_fp64.hip -- the resident plain step of the FP64 path, a launch of
// several steps (compiled as the other FP64 kernels, without hoisting out of the
// loop over the steps).
#include "cbm_kernel.h"

namespace cbm {

hipError_t launch_run_fp64(const StepArgs &a, int64_t mp, hipStream_t stream) {
  return launch_cbm<double, false, true>(a, mp, stream);
}

}  // namespace cbm

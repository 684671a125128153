// cbm_run_mixed.hip -- the resident plain step of the mixed path, a launch of
// several steps (compiled as the other mixed kernels, without hoisting out of
// the loop over the steps).
#include "cbm_kernel.h"

namespace cbm {

hipError_t launch_run_mixed(const StepArgs &a, int64_t mp, hipStream_t stream) {
  return launch_cbm<float, false, true>(a, mp, stream);
}

}  // namespace cbm

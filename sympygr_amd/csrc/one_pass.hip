// The kernels of one_pass.h that evaluate the BSSN right-hand side.
#include "one_pass.h"

namespace sgr {

hipError_t launch_one_pass(const LaunchArgs &a, hipStream_t s) { return launch_pass<Pass::BSSN>(a, s); }

}  // namespace sgr

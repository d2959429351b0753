// The kernels of one_pass.h that evaluate the CCZ4 right-hand side: one field
// more, Gamma-hat and Z^i in the folds, and the K and Theta equations complete
// only after the divergence of Gamma-hat.  A 192^3 block with flagged faces:
// 5.1 ms in two passes, 3.7 ms here.  Parking
// Z^i and those two equations in LDS instead of registers removed the scratch
// reloads of the field loops and still took 7% longer (4.02 -> 4.32 ms).
#include "one_pass.h"

namespace sgr {

hipError_t launch_one_pass_ccz4(const LaunchArgs &a, hipStream_t s) { return launch_pass<Pass::CCZ4>(a, s); }

}  // namespace sgr

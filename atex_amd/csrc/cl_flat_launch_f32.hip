// Flat channels-last kernels, f32 storage.
#include "cl_flat_launch_impl.hip.h"

namespace atexn {
ATEXN_INSTANTIATE_FLAT(float)
}  // namespace atexn

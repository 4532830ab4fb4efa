// Flat channels-last kernels, f16 storage.
#include "cl_flat_launch_impl.hip.h"

namespace atexn {
ATEXN_INSTANTIATE_FLAT(f16_t)
}  // namespace atexn

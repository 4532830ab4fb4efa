// Flat channels-last kernels, bf16 storage.
#include "cl_flat_launch_impl.hip.h"

namespace atexn {
ATEXN_INSTANTIATE_FLAT(bf16_t)
}  // namespace atexn

// The numbers that mark what the workgroups of one launch exchange (ExchangeTag in status.h).  Host
// tags are odd, those of recorded launches even, and none is 0: scratch memory that a caller has
// zeroed must not look claimed.
#pragma once

#ifdef __HIPCC__
#define ATEXN_TAG_FN __host__ __device__ inline
#else
#define ATEXN_TAG_FN inline
#endif

namespace atexn {

ATEXN_TAG_FN unsigned host_call_tag(unsigned n) { return n << 1 | 1u; }

// draw() returns the next number of a counter.  One number in 2^31 would make 0 and is passed over.
template <typename Draw>
ATEXN_TAG_FN unsigned recorded_call_tag(unsigned origin, Draw&& draw) {
  const unsigned tag = (origin + draw()) << 1;
  return tag != 0 ? tag : (origin + draw()) << 1;
}

}  // namespace atexn

// Host-only check of the exchange tags (atex_amd/csrc/call_tag.h); built and run by
// tests/test_call_tags.py.  Exit status 0 and "ok" on success.
#include <cstdio>

#include "call_tag.h"

int main() {
  // counters that pass the numbers whose tag would be 0 (origin + count = 0 and 2^31), and one that does not
  const unsigned origins[] = {0u - 5u, 0x80000000u - 5u, 12345u};
  for (const unsigned origin : origins) {
    unsigned count = 0, before = 1;
    for (int i = 0; i < 64; ++i) {
      const unsigned tag = atexn::recorded_call_tag(origin, [&] { return count++; });
      if (tag == 0 || tag % 2 != 0 || tag == before) {
        std::printf("recorded tag %u after %u, origin %u\n", tag, before, origin);
        return 1;
      }
      before = tag;
    }
  }
  for (unsigned n = 0u - 40u; n != 40u; ++n) {
    if (atexn::host_call_tag(n) % 2 != 1 || atexn::host_call_tag(n) == atexn::host_call_tag(n + 1)) {
      std::printf("host tag of %u\n", n);
      return 1;
    }
  }
  std::printf("ok\n");
  return 0;
}

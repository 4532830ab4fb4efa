// Host-only check of the plans of the flat and hold channels-last kernels (atex_amd/csrc/plan.h): what the kernels
// assume of them, and that threads, steps and slabs cover every element of an instance once.  Built and run
// by tests/test_flat_plans.py.  "ok <plans> <with several slabs> <plans that hold
// more>" on success.
#include <cstdio>
#include <vector>

#include "plan.h"

namespace atexn {
static Tuning g_tuning;
const Tuning& tuning() { return g_tuning; }
}  // namespace atexn
using namespace atexn;

static long g_plans = 0, g_split = 0, g_held = 0, g_failed = 0;
#define EXPECT(cond)                                                                                              \
  do {                                                                                                            \
    if (!(cond) && ++g_failed < 50)                                                                               \
      std::printf("FAIL %s: bwd=%d V=%d N=%lld C=%lld D=%lld cus=%d U=%d threads=%d S=%d\n", #cond, int(bwd), V,  \
                  (long long)N, (long long)C, (long long)D, cus, p.U, p.threads, p.S);                            \
  } while (0)

static void check(bool hold, bool bwd, int V, int64_t N, int64_t C, int64_t D, int cus) {
  const FlatPlan p = hold ? plan_hold(bwd, V, N, C, D, cus) : plan_flat(bwd, V, N, C, D, cus);
  if (!p.on) return;
  ++(hold ? g_held : g_plans);
  if (!hold && p.S > 1) ++g_split;
  EXPECT(p.threads == 256 || p.threads == 512);
  EXPECT(p.A <= p.threads && p.A % p.P == 0 && int64_t(p.P) * V == C * p.pix && V % p.pix == 0);
  bool built = false;
  for (const int u : kPlanFlatUs) built = built || (p.U == u && (u <= 8 || !bwd));
  EXPECT(p.hold == hold && (built || hold));
  if (hold) {  // every vector but the last one is whole, and the passes are what the kernel of that kind has
    const int Q = bwd ? kPlanHoldBwdPass : kPlanHoldFwdPass, B = bwd ? kPlanHoldBwdBatch : kPlanHoldFwdBatch;
    const HoldKind k = bwd ? kPlanHoldBwd[p.kind] : kPlanHoldFwd[p.kind];
    const int before = k.HA + (k.lds ? Q : 0) + p.R;  // vectors before the last pass
    EXPECT(p.S > 1 && C <= p.threads && p.R >= 0 && p.R % Q == 0 && (k.lds || p.R == 0) && Q % B == 0 && k.HA % B == 0);
    EXPECT(before < p.U && p.U <= before + Q && p.U >= Q);
    EXPECT(p.hold_at % 4 == 0 && p.hold_at >= p.k_at + int(bwd ? 4 : 3) * C);
    EXPECT(p.lds == size_t(4) * p.hold_at + (k.lds ? size_t(Q) * p.threads * 16 * (bwd ? 2 : 1) : 0) && p.lds <= 160 * 1024 - 512);
    EXPECT(int64_t(p.U) * p.A * 16 < (int64_t(1) << 32));
  }
  // the slabs are the instance's periods; every step of every slab but the last is whole
  const int64_t E = D * C, step = int64_t(p.A) * V;
  int64_t at = 0, least = E;
  for (int s = 0; s < p.S; ++s) {
    const int64_t p0 = int64_t(s) * p.base + std::max(s - (p.S - p.extra), 0), k = p.base + (s >= p.S - p.extra ? 1 : 0);
    const int64_t px0 = p0 * p.pix, px1 = std::min(px0 + k * p.pix, D);
    EXPECT(px0 * C == at && px1 > px0);
    const int64_t n = (px1 - px0) * C;
    EXPECT(n <= p.U * step && n >= (p.U - 1) * step && (hold || n < (int64_t(1) << 24)) && (k * p.pix < (1 << 24) || hold));
    // pixel counts as the fold takes them
    const int64_t said = s == p.S - 1 ? D - (int64_t(p.S - 1) * p.base + std::max(p.extra - 1, 0)) * p.pix
                                      : (int64_t(p.base) + (s >= p.S - p.extra ? 1 : 0)) * p.pix;
    EXPECT(said == px1 - px0);
    at += n;
    least = std::min(least, n);
  }
  EXPECT(at == E && least > 0);
  // an instance's slabs are on the chip (the XCD) together; 32-bit positions in its pairs
  const int64_t slots = int64_t(cus) * ((hold ? 512 : 1024) / p.threads);
  EXPECT(p.S <= (p.local ? slots / 8 : slots) && 4 * int64_t(p.S) * C < (int64_t(1) << 32));
  EXPECT(p.grid == (p.local ? round_up(N, 8) : N) * p.S && p.grid * p.threads < (int64_t(1) << 32));
  EXPECT(size_t(p.k_at) >= 2 * size_t(step) + 2 * size_t(std::max<int64_t>(p.threads, C)));
  EXPECT(p.lds >= sizeof(float) * (size_t(p.k_at) + size_t(bwd ? 4 : 3) * size_t(C)) && (hold || p.lds + 2048 <= 65536 + 1536));
  const size_t pairs = p.S > 1 ? size_t(16) * N * p.S * C : 0, finals = p.S > 1 ? size_t(16) * N * C : 0;
  EXPECT(p.off_tagged == 0 && p.off_finals >= pairs && p.off_claims >= p.off_finals + finals);
  EXPECT(p.off_part >= p.off_claims + (p.S > 1 ? size_t(4) * N * p.S : 0));
  EXPECT(p.off_tag >= p.off_part + (bwd && N > 1 ? size_t(8) * N * C : 0) && p.ws_bytes >= p.off_tag + 4);
  EXPECT(p.off_finals % 16 == 0 && p.off_claims % 16 == 0 && p.off_part % 16 == 0 && p.off_tag % 4 == 0);
  // the call's plan has room for it and for the kernels that serve y == x
  const ClPlan c = plan_cl(bwd, V, N, C, D, cus);
  EXPECT(!c.flat.on || c.flat.hold || !bwd || V == 8);  // (the product has no other flat backward)
  EXPECT(!c.flat.on || (c.ws_bytes >= c.flat.ws_bytes && c.ws_bytes >= plan_cl_slabs(bwd, V, N, C, D, cus).ws_bytes));
}

// Calls that stay on the slab kernels are told by their sizes, before a plan is made that would be refused.
static void check_refused_early(int V, int64_t N, int64_t C, int64_t D) {
  for (const bool bwd : {false, true}) {
    const int cus = 256;
    const ClPlan c = plan_cl(bwd, V, N, C, D, cus);
    const FlatPlan& p = c.flat;
    EXPECT(!p.on && !flat_may(c, bwd, V, N, C, D) && !hold_may(c, bwd, V, N, C, D));
  }
}

// The kernels of shapes that the rules' comments quote, forward and backward: slabs, flat or held.
static void check_kernel(int V, int64_t N, int64_t D, int64_t C, const char* want) {
  for (const bool bwd : {false, true}) {
    const int cus = 256;
    const FlatPlan p = plan_cl(bwd, V, N, C, D, cus).flat;
    const char got = !p.on ? 's' : (p.hold ? 'h' : 'f');
    EXPECT(got == want[bwd]);
  }
}
static void check_quoted() {
  check_kernel(8, 22, 14280, 17, "ff");
  check_kernel(8, 51, 7684, 87, "fh");
  check_kernel(8, 28, 1275, 162, "ff");
  check_kernel(8, 48, 304, 74, "ss");
  check_kernel(8, 1, 598464, 17, "fh");
  check_kernel(8, 2, 85000, 133, "fh");
  check_kernel(8, 4, 1664, 428, "ss");
  check_kernel(8, 3, 14016, 428, "ss");
  check_kernel(8, 5, 75264, 116, "hh");
  check_kernel(8, 38, 3328, 85, "ff");
  check_kernel(8, 50, 1248, 53, "fs");
  check_kernel(8, 20, 2920, 175, "fs");
  check_kernel(8, 11, 7104, 190, "fh");
  check_kernel(8, 33, 23808, 64, "fh");
  check_kernel(4, 15, 5488, 104, "fh");
  check_kernel(8, 12, 3408, 448, "ss");
  check_kernel(8, 64, 16384, 64, "ff");
  check_kernel(8, 32, 65536, 32, "fh");
  check_kernel(8, 11, 20592, 128, "hh");
  check_kernel(8, 17, 30940, 57, "fh");
  check_kernel(8, 28, 92880, 16, "sh");
  check_kernel(8, 36, 30000, 32, "sh");
  check_kernel(4, 5, 15779, 192, "sh");
  check_kernel(8, 1, 89514, 125, "fh");
  check_kernel(4, 2, 12673, 124, "ss");
  check_kernel(8, 38, 3168, 100, "ff");
  check_kernel(8, 2, 50000, 320, "ss");
  check_kernel(8, 3, 100000, 300, "sh");
  check_kernel(8, 36, 57624, 16, "sh");
  check_kernel(4, 8, 16384, 64, "ss");
  check_kernel(8, 16, 8192, 128, "ss");
  check_kernel(8, 24, 16384, 48, "sh");
  check_kernel(8, 20, 16384, 64, "sh");
  check_kernel(8, 9, 72447, 32, "hh");
  check_kernel(8, 16, 65536, 64, "hh");
  check_kernel(8, 8, 524288, 32, "hh");
  check_kernel(8, 2, 2097152, 32, "hh");
}

int main() {
  check_quoted();
  check_refused_early(8, 8, 64, 16384);
  check_refused_early(8, 2, 320, 216);
  check_refused_early(8, 100, 64, 2048 / 2);
  check_refused_early(8, 5, 57, 800);
  check_refused_early(4, 16, 64, 4096);
  check_refused_early(4, 46, 60, 100);
  std::vector<int64_t> channels;
  for (int64_t c = 4; c <= 80; ++c) channels.push_back(c);
  for (int64_t c = 81; c <= 2100; c += c < 600 ? 5 : 61) channels.push_back(c);
  for (const int64_t c : {127, 128, 129, 255, 256, 257, 511, 512, 513, 1024, 2047, 2048, 2049, 4096}) channels.push_back(c);
  const int64_t pixels[] = {1, 2, 7, 8, 9, 31, 100, 441, 1000, 2047, 4096, 5917, 16384, 30940, 100003, 268800, 1000000, 2097152, 6782976};
  const int64_t batches[] = {1, 2, 3, 7, 8, 9, 13, 17, 24, 59, 64, 300, 5000};
  for (const int64_t C : channels)
    for (const int64_t D : pixels)
      for (const int64_t N : batches)
        for (const int cus : {256, 304, 64, 8, 7})
          for (const int V : {8, 4}) {
            if (C < V) continue;
            for (const bool hold : {false, true})
              for (const bool bwd : {false, true}) check(hold, bwd, V, N, C, D, cus);
          }
  if (g_failed) return 1;
  std::printf("ok %ld %ld %ld\n", g_plans, g_split, g_held);
  return 0;
}

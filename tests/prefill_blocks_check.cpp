// Host check of the prefill attention's block ranges
// (fastdms_amd/csrc/fdms_prefill_blocks.h) over every workgroup and wave of all
// small sequence lengths.  Built with g++ by tests/test_prefill_dispatch.py;
// prints "ok" and exits 0 when every check holds.
#include <algorithm>
#include <cstdio>

#include "fdms_prefill_blocks.h"

using namespace fdms;

static int failures = 0;
#define CHECK(c)                                                                                              \
  do {                                                                                                        \
    if (!(c) && ++failures < 20)                                                                              \
      std::printf("FAIL %s: len %d klen %d q0 %d positions %d wq0 %d\n", #c, len, klen, q0, positions, wq0); \
  } while (0)

// The kernel's loops over the blocks: barriers passed, and blocks multiplied
// unmasked by the first one.
static int barriers(const PrefillBlocks& b, int* unmasked) {
  int n = 0, t = 0;
  *unmasked = 0;
  for (; t + 2 < b.whole; t += 2) n += 2, *unmasked += 2;
  for (; t < b.loaded; t += 2) {
    if (t + 1 < b.loaded) ++n;
    if (t + 1 < b.loaded && t + 2 < b.loaded) ++n;
  }
  return n;
}

int main() {
  for (int positions : {32, 64, 128})
    for (int klen = 1; klen <= 420; ++klen)
      for (int len = 1; len <= klen; ++len)
        for (int q0 = 0; q0 < len; q0 += positions) {
          int first = -1;
          for (int wq0 = q0; wq0 < q0 + positions; wq0 += kPrefillWaveRows) {
            const PrefillBlocks b = prefill_blocks(len, klen, q0, positions, wq0);
            const int off = klen - len, last = std::min(wq0 + kPrefillWaveRows, len) - 1;
            CHECK(0 <= b.whole && b.whole <= b.seen && b.seen <= b.loaded);
            CHECK(b.loaded * kPrefillKeys - klen < kPrefillKeys);  // every loaded block holds a key
            int unmasked;
            const int n = barriers(b, &unmasked);
            if (first < 0) first = n;
            CHECK(n == first);  // every wave of the workgroup passes the same barriers
            if (wq0 >= len) {
              CHECK(b.seen == 0 && unmasked == 0);  // nothing of the wave is stored: it multiplies nothing
            } else {
              CHECK(b.whole * kPrefillKeys <= off + wq0 + 1 && b.whole * kPrefillKeys <= klen);
              CHECK((b.seen - 1) * kPrefillKeys <= off + last && b.seen * kPrefillKeys > off + last);
            }
          }
        }
  if (!failures) std::printf("ok\n");
  return failures != 0;
}

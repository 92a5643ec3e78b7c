// Which 64-key blocks of a sequence a prefill attention workgroup loads and
// each of its waves multiplies.
#pragma once

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define FDMS_PREFILL_HD __host__ __device__
#else
#define FDMS_PREFILL_HD
#endif

namespace fdms {

constexpr int kPrefillKeys = 64;      // keys per block
constexpr int kPrefillWaveRows = 32;  // query positions per wave

struct PrefillBlocks {
  int loaded;  // blocks the workgroup loads: all a row of it sees
  int seen;    // blocks a valid row of the wave sees; 0 for a wave past the sequence's end
  int whole;   // leading blocks every row of the wave sees whole (no mask needed), at most `seen`
};

// The workgroup's queries are positions q0 .. q0 + positions - 1 of len (those
// past the end are not stored), the last len of the sequence's klen >= len keys;
// the wave's are wq0 .. wq0 + kPrefillWaveRows - 1, q0 <= wq0 < q0 + positions, q0 < len.
FDMS_PREFILL_HD inline PrefillBlocks prefill_blocks(int len, int klen, int q0, int positions, int wq0) {
  const int off = klen - len;  // position i sees keys 0 .. off + i
  const auto least = [](int a, int b) { return a < b ? a : b; };
  PrefillBlocks b;
  b.loaded = (least(klen, off + q0 + positions) + kPrefillKeys - 1) / kPrefillKeys;
  if (wq0 >= len) {
    b.seen = b.whole = 0;
  } else {
    b.seen = (off + least(wq0 + kPrefillWaveRows - 1, len - 1)) / kPrefillKeys + 1;
    b.whole = least((off + wq0 + 1) / kPrefillKeys, klen / kPrefillKeys);
  }
  return b;
}

}  // namespace fdms

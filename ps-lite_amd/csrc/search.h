// Searching sorted keys with a wavefront (the slicer's boundaries, the stretches of the ordered match).
#ifndef PSKV_SEARCH_H_
#define PSKV_SEARCH_H_
#include "device_common.h"

namespace pskv {

// A 64-ary lower_bound by one wavefront. Each round the 64 lanes probe evenly spaced keys of
// the remaining interval, a ballot counts how many are below the target (the probes are
// sorted, so the votes are a prefix of ones) and the interval shrinks 64-fold:
// ceil(log64 n) dependent loads instead of ceil(log2 n). Every lane returns the answer.
__device__ __forceinline__ uint64_t wave_lower_bound(const uint64_t* __restrict__ keys, uint64_t n,
                                                     uint64_t target, unsigned lane) {
  uint64_t lo = 0, hi = n;  // the answer lies in [lo, hi]; keys[lo..hi) are undecided
  while (hi > lo) {
    const uint64_t len = hi - lo;
    if (len <= 64) {
      const bool below = lane < len && keys[lo + lane] < target;
      lo += __popcll(__ballot(below));
      break;
    }
    const uint64_t step = (len + 63) / 64;
    const uint64_t idx = lo + (uint64_t)(lane + 1) * step - 1;
    const bool below = idx < hi && keys[idx] < target;
    const uint64_t c = __popcll(__ballot(below));
    // probes 0..c-1 are below the target, probe c (if any) is not
    const uint64_t new_lo = lo + c * step;
    const uint64_t cap = lo + (c + 1) * step - 1;
    hi = cap < hi ? cap : hi;
    lo = new_lo < hi ? new_lo : hi;
  }
  return lo;
}

}  // namespace pskv
#endif  // PSKV_SEARCH_H_

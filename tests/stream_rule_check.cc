// Which pushes stream through the slot array and in which shape (csrc/stream_rule.h).
#include <stdio.h>

#include "stream_rule.h"

using namespace pskv;

int main() {
  int bad = 0;
  auto fail = [&](const char* what, uint64_t n, uint64_t cap) {
    printf("%s: %llu keys, %llu slots\n", what, (unsigned long long)n, (unsigned long long)cap), ++bad;
  };
  // the shape: whatever is accepted fits what the kernels hold
  const uint64_t most = (uint64_t)kMostBins * kBinMean;
  uint64_t accepted = 0;
  for (uint64_t cap = 16; cap <= (1ull << 34); cap *= 2) {
    const uint64_t sizes[] = {1, 2, kSplitTile - 1, kSplitTile, kSplitTile + 1, cap / 64, cap / 7, cap / 2, cap - cap / 8, kBinMean * 2, kBinMean * 2 + 1,
                              most - 1, most, most + 1, 1ull << 24, 1ull << 31};
    for (uint64_t n : sizes) {
      if (n == 0) continue;
      const StreamShape s = stream_shape(n, cap);
      const uint64_t slots = (uint64_t)s.bins * s.images * kImageSlots;
      if (!s.bins) {
        // refused: an array of less than two bins, too many keys for the bins there can be, or too many images for a bin
        const uint64_t bins = cap / kImageSlots < kMostBins ? cap / kImageSlots : kMostBins;
        const bool few = cap / kImageSlots < 4, many = n > bins * kBinMean, large = cap / kImageSlots > (uint64_t)kMostBins * kMostImages;
        if (!few && !many && !large) fail("refused", n, cap);
        continue;
      }
      ++accepted;
      if (slots != cap) fail("the bins do not cover the array", n, cap);
      if (s.bins % 2 || s.bins > kMostBins || s.bins != 1u << s.bin_bits) fail("bins", n, cap);
      if (s.images < 1 || s.images > kMostImages) fail("images", n, cap);
      if (n > (uint64_t)s.bins * kBinMean) fail("more keys than the bins hold", n, cap);
      if ((n + kSplitTile - 1) / kSplitTile > kMostTiles) fail("more tiles than a workgroup looks at", n, cap);
    }
  }
  if (accepted < 100) fail("few sizes accepted", accepted, 0);
  if (!stream_shape(most, 1ull << 24).bins || stream_shape(most + 1, 1ull << 24).bins) fail("the most keys", most, 1ull << 24);
  if (stream_shape(1000, 8192).bins || !stream_shape(1000, 16384).bins) fail("the smallest array", 1000, 16384);
  if (!stream_shape(2000, 8192).bins || stream_shape(2000, 4096).bins) fail("the smallest array for its keys", 2000, 8192);
  if ((most + kSplitTile - 1) / kSplitTile * 2 <= kMostTiles) fail("a workgroup looks at more tiles than there can be", most, kMostTiles);
  if (!stream_shape(1000, 1ull << 28).bins || stream_shape(1000, 1ull << 29).bins) fail("the largest array", 1000, 1ull << 28);
  // four images a bin and more: arrays of 64M slots
  if (stream_shape(1000, 1ull << 26).images != 4 || stream_shape(1000, 1ull << 28).images != 16) fail("images of large arrays", 1000, 1ull << 26);

  // the gain: what the figures beside the rule say, by themselves
  auto pays = [&](bool yes, uint64_t n, uint64_t cap, double fresh, bool grows) {
    if ((stream_gain(n, cap, fresh, grows) >= kStreamLaunches) != yes) fail(yes ? "does not pay" : "pays", n, cap);
  };
  const uint64_t M = 1 << 20;
  pays(true, 4'000'000, 16 * M, 0.5, false);
  pays(true, 1'500'000, 4 * M, 0.5, false);
  pays(false, 3'000'000, 16 * M, 0.0, false);
  pays(false, 800'000, 4 * M, 1.0, false);
  pays(false, 1'000'000, 8 * M, kFreshGuess, false);  // (a table four times as large as the request, as far as is known)
  pays(true, 4'000'000, 16 * M, kFreshGuess, true);
  pays(true, 4'000'000, 64 * M, kFreshGuess, true);  // (a growth is paid for anyway)
  pays(false, 200'000, 2 * M, 1.0, true);
  if (!bad) printf("ok\n");
  return bad != 0;
}

// Which pushes stream through the slot array (stream_push.h), and in which shape. (No GPU code.)
#ifndef PSKV_STREAM_RULE_H_
#define PSKV_STREAM_RULE_H_
#include <stdint.h>

namespace pskv {

constexpr unsigned kSplitTile = 8192;   // keys of a tile
constexpr unsigned kTileWords = kSplitTile + kSplitTile / 2;  // 8-byte words it leaves: keys, and values behind them
constexpr unsigned kMostBins = 4096;
constexpr unsigned kStartsPad = 2;      // 16-bit words behind a tile's row of starts: the number of its keys
constexpr unsigned kImageSlots = 4096;
constexpr unsigned kMostImages = 16;    // per bin: every image looks at all keys of the bin
constexpr unsigned kBinKeys = 2048;     // that a workgroup holds
constexpr unsigned kBinMean = kBinKeys - 64;  // keys of a bin on average, at most (a few bins then have some more than are held)
constexpr unsigned kMostTiles = 1024;
static_assert((uint64_t)kMostBins * kBinMean <= (uint64_t)kMostTiles * kSplitTile, "the keys of the most bins lie in the most tiles");

struct StreamShape {
  uint32_t bins = 0;  // 0: the request does not fit
  uint32_t bin_bits = 0;
  uint32_t images = 0;
};

// The bins for n keys and an array of `cap` slots (a power of two): two images each, one where the bins would have too many
// keys, more where there would be too many bins.
inline StreamShape stream_shape(uint64_t n, uint64_t cap) {
  StreamShape s;
  uint64_t bins = cap / kImageSlots / 2;
  if (bins > kMostBins) bins = kMostBins;
  if (bins * kBinMean < n) bins *= 2;
  if (bins < 2 || bins > kMostBins || bins * kBinMean < n) return s;
  const uint64_t images = cap / kImageSlots / bins;
  if (images > kMostImages) return s;
  s.bins = (uint32_t)bins;
  while ((1ull << s.bin_bits) < bins) ++s.bin_bits;
  s.images = (uint32_t)images;
  return s;
}

// What streaming gains a table's share of a push, in us. Through the slots a million held keys take 48 and new ones
// 88; here a million keys take 18 and a million slots of an array that stays 6.4 (a table that grows is streamed through
// anyway), and a push has three launches more, one behind the other. Measured, us per call, through the slots -> here: 4M
// keys of which half are new in 16M slots 264 -> 173, 1.5M in 4M 162 -> 118, 3M in 16M 200 -> 163, held ones 144 -> 150 (they
// go through the slots); 800,000 new ones in 4M 92 -> 104 (likewise), 4M in 32M 310 -> 257.
// `fresh`: the share of new keys, as far as it is known (kFreshGuess: pushes of held keys are not to pay for the guess).
constexpr double kStreamLaunches = 35.0;
constexpr double kFreshGuess = 0.25;
inline double stream_gain(uint64_t n, uint64_t cap, double fresh, bool grows) {
  return 1e-6 * (double)n * (48.0 + 40.0 * fresh - 18.0) - (grows ? 0.0 : 6.4e-6 * (double)cap);
}

}  // namespace pskv
#endif  // PSKV_STREAM_RULE_H_

// The words in which the slicer's workgroups tell the host what they have found, and what the host makes of them (slice.hip).
// (No GPU code: the host's tests run it over words of their own.)
#ifndef PSKV_PARTS_H_
#define PSKV_PARTS_H_
#include <chrono>
#include <cstddef>
#include <cstdint>

namespace pskv {

// What the host reads goes to pinned memory, every word with a mark of its own that it is there (the host has cleared it):
// the host watches all of them, nothing has to arrive before anything else, and no fence writes back what the requests that
// run meanwhile have left in the L2. Positions and sums are below 2^62 in size.
constexpr uint64_t kHere = 1ull << 63;
constexpr uint64_t told(uint64_t word) { return (uint64_t)((int64_t)(word << 1) >> 1); }  // (sums of lens may be negative)

constexpr unsigned kFusedTargets = 32;  // boundaries that one launch searches

// A part of a request with lens, and the words it tells: lens in the lower kPartLensBits (2,048 of 32 bits, a sign), and above
// them for the part the first of its boundaries and their number, for a boundary its place in the part.
constexpr unsigned kFewSumsBlock = 256, kFewSumsItems = 8;  // (larger workgroups find no place on a busy GPU)
constexpr uint64_t kFewSumsPart = (uint64_t)kFewSumsBlock * kFewSumsItems;
constexpr unsigned kFewSumsParts = 512;
constexpr uint64_t kFewSumsKeys = kFewSumsParts * kFewSumsPart;
constexpr unsigned kPartLensBits = 45, kPartCountAt = kPartLensBits + 6;
static_assert(kFewSumsPart <= 1u << 11 && kFusedTargets < 64, "a place and two numbers of boundaries fit above the lens");
constexpr unsigned long long part_word(unsigned long long lens, unsigned long long upper) {
  return (lens & ((1ull << kPartLensBits) - 1)) | upper << kPartLensBits;
}
constexpr uint64_t part_lens(uint64_t word) {
  return (uint64_t)((int64_t)(word << (64 - kPartLensBits)) >> (64 - kPartLensBits));
}

// When a call that has been made now stops watching for its words and waits for its stream instead: whatever their number,
// for a GPU that is busy with something else leaves all of them out.
typedef std::chrono::steady_clock::time_point WatchEnd;
inline WatchEnd watch_end(std::chrono::steady_clock::time_point now) { return now + std::chrono::microseconds(200); }

// Watches `count` marked words; false when one was not there in the end.
inline bool all_here(const uint64_t* words, size_t count, WatchEnd end) {
  for (size_t i = 0; i < count; ++i) {
    if (__atomic_load_n(words + i, __ATOMIC_ACQUIRE) != 0) continue;
    for (bool here = false; !here;) {
      for (int spin = 0; spin < 256 && !here; ++spin) here = __atomic_load_n(words + i, __ATOMIC_ACQUIRE) != 0;
      if (!here && std::chrono::steady_clock::now() > end) return false;
    }
  }
  return true;
}

// What the parts of k_bounds_sums_few have told: the positions of the boundaries and the sums of the slices between them.
// False at the first word that did not show up, or when keys that are not sorted have left a boundary without an owner, or
// with two: what comes late may then still be on its way.
inline bool join_parts(const uint64_t* parts, const uint64_t* bounds, uint64_t n, size_t S, uint64_t* pos, uint64_t* sums,
                       WatchEnd end) {
  uint64_t before = 0, below[kFusedTargets], seen = 0;
  bool clear = true;  // no boundary has two owners
  for (size_t i = 0; i <= S; ++i) pos[i] = below[i] = 0;
  for (uint64_t b = 0; b * kFewSumsPart < n; ++b) {
    if (!all_here(parts + b, 1, end)) return false;
    const uint64_t word = parts[b];
    const unsigned first = (unsigned)(word >> kPartLensBits) & 63u, count = (unsigned)(word >> kPartCountAt) & 63u;
    for (unsigned i = first; i < first + count; ++i) {
      if (!all_here(bounds + i, 1, end)) return false;
      clear = clear && !(seen >> i & 1u);
      seen |= 1ull << i;
      pos[i] = b * kFewSumsPart + ((bounds[i] & ~kHere) >> kPartLensBits);
      below[i] = before + part_lens(bounds[i]);
    }
    before += part_lens(word);
  }
  for (size_t i = 1; i <= S; ++i) {
    if (pos[i] < pos[i - 1]) pos[i] = pos[i - 1], below[i] = below[i - 1];
    sums[i - 1] = below[i] - below[i - 1];
  }
  return clear && seen == (2ull << S) - 1;
}

}  // namespace pskv
#endif  // PSKV_PARTS_H_

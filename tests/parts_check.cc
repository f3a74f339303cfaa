// The host's half of a slice with lens (csrc/parts.h) over words of its own: what they are joined to, against sums taken
// directly; and how long the host looks for words that do not come, which is what a thread that calls the slicer burns while
// the GPU is busy with something else.
#include <stdio.h>
#include <stdlib.h>

#include <algorithm>
#include <vector>

#include "parts.h"

using namespace pskv;

struct Words {
  std::vector<uint64_t> parts, bounds;
};

// What the workgroups tell of keys 0, 1, .. n-1 with `lens`, cut at `cut` (ascending).
static Words tell(uint64_t n, const std::vector<int32_t>& lens, const std::vector<uint64_t>& cut) {
  Words w;
  w.bounds.assign(kFusedTargets, 0);
  for (uint64_t c0 = 0; c0 < n; c0 += kFewSumsPart) {
    const uint64_t c1 = std::min(n, c0 + kFewSumsPart);
    uint64_t first = 0, count = 0;
    for (size_t i = 0; i < cut.size(); ++i) {
      if (!(c0 == 0 || cut[i] > c0 - 1) || !(c1 == n || cut[i] <= c1 - 1)) continue;
      if (!count++) first = i;
      uint64_t below = 0;
      for (uint64_t j = c0; j < std::min(cut[i], c1); ++j) below += (uint64_t)(int64_t)lens[j];
      w.bounds[i] = kHere | part_word(below, std::min(cut[i], c1) - c0);
    }
    uint64_t all = 0;
    for (uint64_t j = c0; j < c1; ++j) all += (uint64_t)(int64_t)lens[j];
    w.parts.push_back(kHere | part_word(all, first | count << 6));
  }
  return w;
}

static bool check(uint64_t n, const std::vector<int32_t>& lens, const std::vector<uint64_t>& cut) {
  const size_t S = cut.size() - 1;
  const Words w = tell(n, lens, cut);
  std::vector<uint64_t> pos(S + 1), sums(S);
  if (!join_parts(w.parts.data(), w.bounds.data(), n, S, pos.data(), sums.data(), watch_end(std::chrono::steady_clock::now()))) return printf("not joined\n"), false;
  for (size_t i = 0; i < S; ++i) {
    uint64_t want = 0;
    for (uint64_t j = std::min(cut[i], n); j < std::min(cut[i + 1], n); ++j) want += (uint64_t)(int64_t)lens[j];
    if (pos[i] != std::min(cut[i], n) || sums[i] != want) return printf("slice %zu of %zu, n %llu\n", i, S, (unsigned long long)n), false;
  }
  return true;
}

int main() {
  srand(7);
  for (uint64_t n : {(uint64_t)1, kFewSumsPart - 1, kFewSumsPart, kFewSumsPart + 1, 5 * kFewSumsPart + 3, kFewSumsKeys}) {
    std::vector<int32_t> lens(n);
    for (auto& l : lens) l = rand() % 2001 - 1000;
    for (unsigned S : {1u, 3u, kFusedTargets - 1}) {
      std::vector<uint64_t> cut(S + 1);
      for (auto& c : cut) c = (uint64_t)rand() * 77 % (n + 3);
      std::sort(cut.begin(), cut.end());
      if (!check(n, lens, cut)) return 1;
    }
  }
  // no word, then all but the last: a look, however many words there are to look for
  const uint64_t n = kFewSumsKeys;
  const Words all = tell(n, std::vector<int32_t>(n, 1), {0, n / 2, n});
  for (int missing = 0; missing < 2; ++missing) {
    Words w = all;
    if (missing) w.parts.back() = 0; else std::fill(w.parts.begin(), w.parts.end(), 0), std::fill(w.bounds.begin(), w.bounds.end(), 0);
    uint64_t pos[3], sums[2];
    const auto t0 = std::chrono::steady_clock::now();
    if (join_parts(w.parts.data(), w.bounds.data(), n, 2, pos, sums, watch_end(t0))) return printf("joined what is not there\n"), 1;
    const double ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    if (ms > 20) return printf("looked for %.1f ms\n", ms), 1;
  }
  printf("ok\n");
  return 0;
}

// Whether a var-len request starts with one launch (k_var_push_start, k_var_pull_start of one_launch.h) or with two. (No GPU
// code: the host's tests run it.)
#ifndef PSKV_START_RULE_H_
#define PSKV_START_RULE_H_
#include <stdint.h>

namespace pskv {

struct StartOf {
  uint64_t keys = 0, floats = 0;  // of all its tables
  uint64_t parts = 0;             // workgroups that have to meet
  unsigned tables = 1;
  bool push = false;
  bool compared = false;  // may repeat the cached request
  bool shortcut = false;  // and if it does, the row kernel of a push need not look for the rows (no ragged rows in it)
};

constexpr unsigned kVarParts = 256;

// What one launch saves is 5 to 8 us. What it costs:
// Workgroups that wait for each other (200,000 rows in 391 of them, other rows in every step, three tables in turn: 233 us
// with two launches, 243 with one). A row kernel that also cleans up behind it is slower by up to a tenth where it moves much
// (us per push of other rows in every step, two launches -> one: 65,536 rows of 256 floats 64.3 -> 60.8, 20,000 of 1,024 72.3
// -> 69.8, 130,000 of 256 106.4 -> 108.4, 65,536 of 700 132 -> 137).
constexpr uint64_t kStartFloats = 24u << 20;
// Of a request that repeats the cached one two launches are short, for the second returns at once (100,000 rows over 16
// tables, push and pull: 51 us against 54; pulls of 65,536 rows of 64 floats 16.3 -> 15.0 with one, of 256 31.1 -> 33.3; pushes
// of 65,536 ragged rows of 45 in one table 23.9 -> 25.4 and 33.0 -> 35.2 with a wait behind each, of 40,000 20.3 -> 19.2 and
// 28.8 -> 29.9, of 65,536 over 16 27.5 -> 23.8 and 37.1 -> 37.0).
constexpr uint64_t kStartRepeatKeys = 1u << 16, kStartRepeatFloats = 1u << 23;
constexpr unsigned kStartFewTables = 4;
constexpr uint64_t kStartRepeatKeysFew = 3u << 14;  // of a push
// And k_var_push_start does not compare: it looks the keys up again, and the row kernel has no shortcut then (one table:
// 65,536 rows of 64 floats 22.1 -> 26.6 us, of 1,024 153 -> 197, 20,000 of 256 22.7 -> 28.2). That pays only where the
// launches are most of a request: push and pull of 5,000 rows of 64 in one table 21.6 -> 19.7 and 32.1 -> 32.5 with a wait
// behind each, over four 23.3 -> 19.6, slice, push and pull of 40,000 of 12 over three 26.5 -> 24.0 and 44.7 -> 46.3, but a
// push of 20,000 of 50 over four 11.8 -> 15.4; over 16, whose launches carry 3.8 KB, push and pull of 1,000 of 64 23 -> 18,
// pushes of 5,000 of 256 15.7 -> 15.6, of 20,000 of 64 15.3 -> 16.6.
constexpr uint64_t kStartShortcutFloatsFew = 1u << 19, kStartShortcutFloats = 1u << 20;

constexpr bool one_start(const StartOf& r) {
  if (r.parts > kVarParts || r.floats > kStartFloats) return false;
  if (!r.compared) return true;
  const bool few = r.tables <= kStartFewTables;
  if (r.keys > (r.push && few ? kStartRepeatKeysFew : kStartRepeatKeys) || r.floats > kStartRepeatFloats) return false;
  return !r.push || !r.shortcut || r.floats <= (few ? kStartShortcutFloatsFew : kStartShortcutFloats);
}

}  // namespace pskv
#endif  // PSKV_START_RULE_H_

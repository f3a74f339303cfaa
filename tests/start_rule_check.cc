// Which var-len requests start with one launch (csrc/start_rule.h).
#include <stdio.h>

#include <initializer_list>

#include "start_rule.h"

using namespace pskv;

static StartOf of(uint64_t keys, uint64_t row, unsigned tables, bool push, bool compared, bool shortcut) {
  StartOf r;
  r.keys = keys, r.floats = keys * row, r.parts = (keys + 511) / 512, r.tables = tables;
  r.push = push, r.compared = compared, r.shortcut = shortcut;
  return r;
}

int main() {
  int bad = 0;
  auto want = [&](bool one, const StartOf& r, const char* what) {
    if (one_start(r) != one) printf("%s: %d\n", what, !one), ++bad;
  };
  for (uint64_t keys : {1, 1000, 20'000, 65'536}) {
    want(true, of(keys, 64, 4, true, false, false), "a push of other keys");
    want(true, of(keys, 64, 4, false, true, false), "a pull that repeats the cached request");
    want(keys <= 3u << 14, of(keys, 45, 1, true, true, false), "a push that repeats it, with ragged rows, one table");
    want(true, of(keys, 45, 16, true, true, false), "a push that repeats it, with ragged rows, sixteen tables");
    // what the row kernel of a repeat saves is more than a launch
    want(keys * 64 <= 1u << 19, of(keys, 64, 1, true, true, true), "a push that repeats it, one table");
    want(keys * 64 <= 1u << 19, of(keys, 64, 4, true, true, true), "a push that repeats it, four tables");
    want(keys * 64 <= 1u << 20, of(keys, 64, 16, true, true, true), "a push that repeats it, sixteen tables");
  }
  want(false, of(20'000, 256, 16, true, true, true), "a push of many floats that repeats it, sixteen tables");
  want(false, of(20'000, 64, 1, true, true, true), "a push of some floats that repeats it, one table");
  want(false, of(65'537, 8, 16, true, true, false), "a push of many keys that repeats it");
  want(false, of(65'536, 256, 4, false, true, false), "a pull of many floats that repeats it");
  want(true, of(65'536, 256, 4, false, false, false), "a pull of other keys");
  want(false, of(65'536, 700, 1, true, false, false), "a push of very many floats");
  want(true, of(131'072, 8, 1, true, false, false), "as many workgroups as may meet");
  want(false, of(131'073, 8, 1, true, false, false), "one more");
  if (!bad) printf("ok\n");
  return bad != 0;
}

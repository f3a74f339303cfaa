// What the row kernels read of a request's values (csrc/quads.h): every quad of every row, of a push by workgroups that each
// take some rows (k_fixed_own) and of one that is cut quad by quad (rows_quads_fixed). Nothing is read past the values.
// --any-row: whatever the length of the row that follows.
#include <stdio.h>
#include <string.h>

#include <algorithm>

#include "quads.h"

using namespace pskv;

static bool inside(const char* who, uint64_t at, unsigned floats, uint64_t k, uint64_t n) {
  if (at + floats <= n * k) return true;
  printf("%s: floats %llu..%llu of %llu (k %llu, n %llu)\n", who, (unsigned long long)at, (unsigned long long)at + floats - 1,
         (unsigned long long)(n * k), (unsigned long long)k, (unsigned long long)n);
  return false;
}

int main(int argc, char** argv) {
  const bool any_row = argc > 1 && !strcmp(argv[1], "--any-row");
  for (uint64_t k = 1; k <= 13; ++k) {
    const uint64_t quads = (k + 3) / 4, rest = k & 3;
    for (uint64_t n = 1; n <= 3 * 256 + 5; ++n) {
      for (uint64_t row = 0; row < n; ++row) {
        for (uint64_t c = 0; c < quads; ++c) {
          const unsigned count = rest && c + 1 == quads ? (unsigned)rest : 4u;
          const uint64_t at = row * k + c * 4;
          const bool whole = count == 4 || (any_row ? row + 1 < n : whole_quads(row + 1, k, n));
          if (!inside("a quad", at, whole ? 4 : count, k, n)) return 1;
        }
      }
      for (uint64_t share : {(uint64_t)1, (uint64_t)2, (uint64_t)3, (uint64_t)64, (uint64_t)256}) {
        for (uint64_t first = 0; first < n; first += share) {
          const uint64_t mine = std::min(share, n - first);
          const bool whole = any_row ? !rest || first + mine < n : whole_quads(first + mine, k, n);
          for (uint64_t q = 0; whole && q < mine * quads; ++q)
            if (!inside("a share", (first + q / quads) * k + q % quads * 4, 4, k, n)) return 1;
        }
      }
    }
  }
  printf("ok\n");
  return 0;
}

// The bookkeeping of csrc/devpool.hip on the CPU (compiled against tests/include/host_hip): an array that is handed
// out is never one that queued work of another stream still uses, unless the taker was made to wait for it.
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include "devpool.h"
#include "host_common.h"

namespace pskv {
int set_error(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vfprintf(stderr, fmt, ap);
  va_end(ap);
  return code;
}
void clear_error() {}
}  // namespace pskv

using namespace pskv;

#define CHECK(x) do { if (!(x)) { printf("%s:%d: %s\n", __FILE__, __LINE__, #x); return 1; } } while (0)

// Whether `stream` may use an array whose former user was at `at` of `former`: it is past it, or was made to wait.
static bool safe(hipStream_t stream, hipStream_t former, unsigned long at) {
  if (stream == former || former->done >= at) return true;
  for (const auto& w : host_hip().waits)
    if (w.first == stream && w.second.stream == former && w.second.at >= at) return true;
  return false;
}

// Two tables on one stream, in two threads: one of them waits for the stream and settles, the other gives an array
// up between the two.
static int settle() {
  HostStream shared, other;
  void *before = nullptr, *between = nullptr, *got = nullptr;
  CHECK(array_alloc(&before, 1 << 20, &shared) == PSKV_OK);
  CHECK(array_alloc(&between, 8 << 20, &shared) == PSKV_OK);
  shared.queued = 5;
  CHECK(array_release(before, &shared) == PSKV_OK);
  const unsigned long long mark = array_mark();
  CHECK(hipStreamSynchronize(&shared) == hipSuccess);
  shared.queued = 9;  // (the kernel of a growth that reads the old array)
  CHECK(array_release(between, &shared) == PSKV_OK);
  array_settle(&shared, mark);
  CHECK(array_alloc(&got, 8 << 20, &other) == PSKV_OK && got == between);
  CHECK(safe(&other, &shared, 9));
  const size_t waits = host_hip().waits.size();
  CHECK(array_alloc(&got, 1 << 20, &other) == PSKV_OK && got == before);
  CHECK(host_hip().waits.size() == waits);  // settled: nothing to wait for, the stream may be gone
  CHECK(array_release(before, &other, true) == PSKV_OK && array_release(between, &other, true) == PSKV_OK);
  array_trim(0);
  CHECK(host_hip().live.empty());
  return 0;
}

int main(int argc, char** argv) {
  const char* what = argc > 1 ? argv[1] : "";
  int bad = 2;
  if (!strcmp(what, "settle")) bad = settle();
  if (!bad) printf("ok\n");
  return bad;
}

// The bookkeeping of csrc/devpool.hip on the CPU (compiled against tests/include/host_hip): an array that is handed
// out is never one that queued work of another stream still uses, unless the taker was made to wait for it.
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <chrono>
#include <thread>

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
  const unsigned long long mark = array_mark(0);
  CHECK(hipStreamSynchronize(&shared) == hipSuccess);
  shared.queued = 9;  // (the kernel of a growth that reads the old array)
  CHECK(array_release(between, &shared) == PSKV_OK);
  array_settle(0, &shared, mark);
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

static void sleep_ms(int ms) { std::this_thread::sleep_for(std::chrono::milliseconds(ms)); }

static size_t allocated() {
  std::lock_guard<std::mutex> lk(host_hip().mu);
  return host_hip().live_bytes;
}

// What tables leave is kept while there are tables, and for a while after the last one: then it goes back.
static int linger() {
  HostStream s;
  void *a = nullptr, *b = nullptr;
  auto give_back = [](int device) { array_trim(device); };
  device_tables(0, 1, give_back);
  device_tables(0, 1, give_back);
  CHECK(array_alloc(&a, 64 << 20, &s) == PSKV_OK && array_alloc(&b, 256 << 20, &s) == PSKV_OK);
  s.queued = 3;
  CHECK(array_release(a, &s) == PSKV_OK);
  device_tables(0, -1, give_back);  // (another one is there)
  sleep_ms(kLingerMs + 500);
  CHECK(allocated() > 0);
  CHECK(array_release(b, &s) == PSKV_OK);
  device_tables(0, -1, give_back);
  sleep_ms(kLingerMs / 2);
  CHECK(allocated() == (320u << 20));
  device_tables(0, 1, give_back);  // one comes in time: it finds what the last one has left
  sleep_ms(kLingerMs);
  void* again = nullptr;
  CHECK(array_alloc(&again, 256 << 20, &s) == PSKV_OK && again == b);
  CHECK(array_release(again, &s) == PSKV_OK);
  device_tables(0, -1, give_back);
  sleep_ms(kLingerMs + 500);
  CHECK(allocated() == 0);
  return 0;
}

// PSKV_NO_ASYNC_ALLOC: nothing is kept, and an array is freed when the work that uses it is done.
static int unkept() {
  HostStream s;
  void* a = nullptr;
  CHECK(!arrays_are_kept());
  CHECK(array_alloc(&a, 64 << 20, &s) == PSKV_OK && allocated() > 0);
  s.queued = 3;
  CHECK(array_release(a, &s) == PSKV_OK && s.done == 3 && allocated() == 0);
  CHECK(array_alloc(&a, 64 << 20, &s) == PSKV_OK);
  CHECK(array_release(a, &s, true) == PSKV_OK && allocated() == 0);
  return 0;
}

// More than the list may hold: the oldest arrays go.
static int bound() {
  HostStream s;
  std::vector<void*> all(12);
  for (void*& p : all) CHECK(array_alloc(&p, (size_t)1 << 30, &s) == PSKV_OK);
  for (void* p : all) CHECK(array_release(p, &s) == PSKV_OK);
  for (int i = 0; i < 100 && allocated() > ((size_t)8 << 30); ++i) sleep_ms(20);
  CHECK(allocated() == ((size_t)8 << 30));
  host_hip().room = (size_t)8 << 30;  // the memory is full: what the list holds makes room
  void* big = nullptr;
  CHECK(array_alloc(&big, (size_t)6 << 30, &s) == PSKV_OK && allocated() == ((size_t)6 << 30));
  return 0;
}

int main(int argc, char** argv) {
  const char* what = argc > 1 ? argv[1] : "";
  int bad = 2;
  if (!strcmp(what, "settle")) bad = settle();
  if (!strcmp(what, "linger")) bad = linger();
  if (!strcmp(what, "unkept")) bad = unkept();
  if (!strcmp(what, "bound")) bad = bound();
  if (!bad) printf("ok\n");
  return bad;
}

// pskv::StreamChoice (csrc/stream_choice.h) over calls whose times are given: on a quiet GPU it stays where it is, whatever
// the sizes of the calls and in whatever order they come; where calls wait behind others on some of the streams it finds one
// on which they do not.
#include <stdio.h>

#include <vector>

#include "stream_choice.h"

using namespace pskv;

struct Call {
  uint64_t n;
  size_t S;
  bool lens;
  float us;  // as measured on a quiet GPU
};
static const std::vector<Call> kQuiet = {
    {1000, 1, false, 8.5f},       {1000, 31, false, 9.7f},        {1u << 26, 31, false, 10.8f}, {1000, 1, true, 10.5f},
    {1000, 32, false, 16.0f},     {1u << 24, 100, false, 25.0f},  {100, 31, true, 19.8f},
    {1000, 16, true, 12.1f},      {300000, 1, true, 11.9f},       {1u << 20, 16, true, 15.2f},  {(1u << 20) + 1, 1, true, 15.4f},
    {(1u << 20) + 1, 31, true, 18.8f}, {1u << 21, 1, true, 15.6f}, {1u << 21, 31, true, 19.4f}, {1u << 22, 16, true, 17.7f},
    {1u << 23, 31, true, 23.7f},  {1u << 24, 1, true, 24.6f},     {1u << 24, 31, true, 30.6f},  {1u << 25, 16, true, 34.9f},
    {1u << 26, 1, true, 54.9f},   {1u << 26, 31, true, 66.9f}};

// `waits`: what a call waits for on each stream. Returns how often the stream changed in `count` calls.
static int moves(StreamChoice& c, const std::vector<Call>& calls, const float (&waits)[kSliceStreams], int count) {
  int n = 0;
  for (int i = 0; i < count; ++i) {
    const Call& x = calls[(size_t)(i * 7) % calls.size()];
    const float noise = 1.0f + 0.01f * (float)(i * 13 % 21);
    const int next = c.note(x.us * noise + waits[c.at], own_slice_us(x.n, x.S, x.lens));
    n += next != c.at;
    c.at = next;
  }
  return n;
}

int main() {
  const float none[kSliceStreams] = {0, 0, 0, 0};
  for (const Call& x : kQuiet) {
    StreamChoice c;
    if (const int n = moves(c, {x}, none, 2000))
      return printf("%d moves on a quiet GPU: %llu keys, %zu ranges, lens %d\n", n, (unsigned long long)x.n, x.S, (int)x.lens), 1;
  }
  StreamChoice mixed;
  if (const int n = moves(mixed, kQuiet, none, 2000)) return printf("%d moves on a quiet GPU, calls of all sizes\n", n), 1;
  for (int free = 0; free < kSliceStreams; ++free) {
    float waits[kSliceStreams] = {70, 70, 70, 70};
    waits[free] = 0;
    StreamChoice c;
    moves(c, {kQuiet[0], kQuiet[4]}, waits, 40);
    if (c.at != free) return printf("on stream %d, and stream %d is free\n", c.at, free), 1;
    if (moves(c, {kQuiet[0], kQuiet[4]}, waits, 500)) return printf("leaves the stream that is free\n"), 1;
  }
  for (float wait = 0; wait < 8; wait += 1) {  // a GPU with enough to do
    const float waits[kSliceStreams] = {wait, wait, wait, wait};
    StreamChoice c;
    if (moves(c, {kQuiet[0]}, waits, 500)) return printf("goes round the streams of a busy GPU\n"), 1;
  }
  // short waits, as behind a push and a pull that are short themselves
  for (int free = 0; free < kSliceStreams; ++free) {
    float waits[kSliceStreams] = {9, 9, 9, 9};
    waits[free] = 0;
    StreamChoice c;
    moves(c, {{59'225, 16, true, 12.6f}}, waits, 40);
    if (c.at != free) return printf("on stream %d with short waits, and stream %d is free\n", c.at, free), 1;
  }
  printf("ok\n");
  return 0;
}

// Which of a slicer context's streams the next call takes. (No GPU code: the host's tests run it over times of their own.)
#ifndef PSKV_STREAM_CHOICE_H_
#define PSKV_STREAM_CHOICE_H_
#include <cstddef>
#include <cstdint>

namespace pskv {

// What a call takes that waits for nobody, in us: 8.5 to 10.5 without lens, whatever the number of keys; with lens 10.5 for
// 1,000 keys over one range, 12.1 over 16, 13.7 and 15.2 for 1M, 16.3 and 17.7 for 4M, 55 and 58 for 64M (66.9 over 31).
inline float own_slice_us(uint64_t n, size_t S, bool lens) {
  return 10.0f + (lens ? 1.0f + 0.125f * (float)S + 7.5e-7f * (float)n : 0.0f);
}

// A process has few hardware queues (four), and a stream shares its one with others: where those are tables with
// requests queued, every call waits behind them (20 pushes of 1M keys, sliced one by one: 2,250 us, or 2,040 where it
// does not). Nothing says which queue a stream is on, but the calls themselves: a context whose calls take long, next to
// what they would take by themselves, tries other streams and keeps to the one on which they took least. (A limit in us
// for calls of any size had calls of millions of keys with lens go round the streams of a quiet GPU, a stream wait each.)
constexpr int kSliceStreams = 4;
constexpr float kSliceSlow = 2.0f;  // times as long as by itself

struct StreamChoice {
  float took[kSliceStreams] = {0.0f};  // times its own time, lately; forgotten little by little while another one is in use
  int at = 0;                          // the stream in use
  // A call has taken `us` on it, by itself it would take `own`: the stream of the next one.
  int note(float us, float own) {
    const float x = us / own;
    float& mine = took[at];
    mine = mine == 0.0f ? x : 0.75f * mine + 0.25f * x;
    for (int i = 0; i < kSliceStreams; ++i)
      if (i != at) took[i] *= 0.995f;
    if (mine < kSliceSlow) return at;
    // (by a good margin: a stream wait comes with it, and where the GPU itself is what calls wait for all are alike)
    int best = at;
    for (int i = 0; i < kSliceStreams; ++i)
      if (took[i] < 0.75f * mine && took[i] < took[best]) best = i;
    return best;
  }
};

}  // namespace pskv
#endif  // PSKV_STREAM_CHOICE_H_

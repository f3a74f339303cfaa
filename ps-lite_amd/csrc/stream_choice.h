// Which of a slicer context's streams the next call takes. (No GPU code: the host's tests run it over times of their own.)
#ifndef PSKV_STREAM_CHOICE_H_
#define PSKV_STREAM_CHOICE_H_
#include <cstddef>
#include <cstdint>

namespace pskv {

// What a call takes that waits for nobody, in us (to about a tenth): 8.5 to 10.5 without lens, whatever the number of keys, up to
// 31 ranges, 16 for 32 and 24.5 for 100; with lens 10.5 for 1,000 keys over one range, 12.4 over 16, 15.9 over 31, 14.0 and
// 15.0 for 1M over one and 16, 15.4 and 16.6 for one key more (another kernel), 18.0 and 22.4 for 8M, 55 and 58 for 64M.
inline float own_slice_us(uint64_t n, size_t S, bool lens) {
  if (!lens) return S < 32 ? 10.0f : 16.0f + 0.125f * (float)(S - 32);
  return 11.0f + 0.17f * (float)S + (n > (1u << 20) ? 3.0f : 0.0f) + 7e-7f * (float)n;
}

// A process has few hardware queues (four), and a stream shares its one with others: where those are tables with
// requests queued, every call waits behind them (20 pushes of 1M keys, sliced one by one: 2,250 us, or 2,040 where it
// does not). Nothing says which queue a stream is on, but the calls themselves: a context whose calls take long, next to
// what they would take by themselves, tries other streams and keeps to the one on which they took least. (A limit in us
// for calls of any size had calls of millions of keys with lens go round the streams of a quiet GPU, a stream wait each. Twice
// a call's own time is too long: calls that wait behind a push and a pull of some 10 us each take 15 to 25, and stay. us per
// slice, push and pull of 3 sets of 59,225 rows of 12 floats over 16 tables in turn, six runs: 118-134, with 1.5 times 91-113.
// Calls of 10 us take 15 to 20 on any stream of a GPU that has enough to do, so below 20 none is slow: 8 pushes of 200,000 new
// keys into four tables, sliced one by one, 279 us, and 287 with 15 as the limit.)
constexpr int kSliceStreams = 4;
constexpr float kSliceSlow = 1.5f, kSliceSlowUs = 20.0f;  // so many times its own time, and so long

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
    if (mine < kSliceSlow || mine * own < kSliceSlowUs) return at;
    // (by a good margin: a stream wait comes with it, and where the GPU itself is what calls wait for all are alike)
    int best = at;
    for (int i = 0; i < kSliceStreams; ++i)
      if (took[i] < 0.75f * mine && took[i] < took[best]) best = i;
    return best;
  }
};

}  // namespace pskv
#endif  // PSKV_STREAM_CHOICE_H_

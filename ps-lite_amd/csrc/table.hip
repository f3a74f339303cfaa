// Host side of the HBM-resident key-value store: owns the slot array, the row
// arena and the per-request workspace, sizes them, and enqueues the kernels of
// table_kernels.h in request order on one stream. This is what a ps-lite server
// calls in place of KVServerDefaultHandle (include/ps/kv_app.h:440-463).
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <thread>
#include <tuple>
#include <type_traits>
#include <vector>

#include <hip/hip_ext.h>

#include "devpool.h"
#include "growths.h"
#include "host_common.h"
#include "one_launch.h"
#include "scan.h"
#include "stager.h"
#include "stream_push.h"
#include "stream_rule.h"
#include "table_kernels.h"

namespace pskv {

static thread_local std::string g_last_error;

int set_error(int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_last_error = buf;
  return code;
}
void clear_error() { g_last_error.clear(); }

namespace {

constexpr uint64_t kDefaultCapacity = 1u << 20;
constexpr uint64_t kMinSlots = 1024;
constexpr unsigned kMaxGrid = 1u << 20;
// The write-back of the SCALAR key cache mostly finds nothing to do (the request in flight repeats
// the cached keys, or the slots are up to date), and a launch costs by the workgroup even then:
// 62,500 workgroups that leave at once took 15 us. It strides over the keys with this many.
constexpr unsigned kFlushGrid = 4096;
constexpr size_t kMaxProfSamples = 65536;
constexpr uint64_t kSlackBytes = 256ull << 20;  // tables up to this size trade memory for fewer waits
// A slot array that could run short is replaced without asking the device first while the larger
// one stays below this size; beyond it the host waits for exact counters before it spends the memory.
constexpr uint64_t kGrowUnaskedBytes = 4096ull << 20;
constexpr uint64_t kKeepInFlight = 2;  // requests the host leaves unaccounted for when it lets the device catch up
// ... unless the array that the uncertainty would cost is this large: then it lets the device catch up all the way
constexpr uint64_t kLargeArrayBytes = 1024ull << 20;
constexpr uint64_t kSpareMaxBytes = 16384ull << 20;  // no array larger than this is allocated ahead of need
// Host-resident requests up to this size (per direction) skip the copy commands: the kernels
// read the request from, and write the response to, pinned host memory mapped into the GPU.
constexpr size_t kSmallBytes = 1024u << 10;
// Requests up to a quarter of that take their room in turn, so that several can be in flight (small_room).
constexpr int kSmallParts = 4;
constexpr size_t kSmallPart = kSmallBytes / kSmallParts;
// Host-resident buffers from this size on travel piece by piece through the ring of pinned memory
// (stager.h), copying, transfer and kernels overlapping; smaller ones take one copy command.
constexpr size_t kPipeBytes = 4u << 20;
// The fill a slot array never exceeds, whatever the host assumed about the requests in flight (reserve()).
constexpr double kHardLoad = 0.85;

// A device buffer that only grows. Contents are not kept across growth.
struct GrowBuf {
  void* ptr = nullptr;
  size_t bytes = 0;
};

struct EventPair {
  hipEvent_t a, b;
};

// What the host reads back of the device state, written by the device into pinned host memory
// (a one-wavefront kernel is quicker than a copy command for these few words).
struct StateView {
  uint64_t count;       // keys held, the side slot included
  uint64_t arena_top;
  uint64_t scan_total;
  uint64_t same_epoch;
  unsigned error, req_error, special_present, pad;
  unsigned long long seq;  // written last: the number of the reading (StateBatch::seq)
};

// A new table: its device state all zero, the side slot's payload unset, its slots all ones (key = empty
// marker). One launch: a memset command behind a kernel of its own left the GPU idle for 5 to 12 us per table.
__global__ __launch_bounds__(kBlock) void k_init_table(DevState* st, Slot* slots, uint64_t cap) {
  unsigned long long* w = reinterpret_cast<unsigned long long*>(st);
  constexpr unsigned kAt = offsetof(DevState, special_payload) / 8;
  static_assert(sizeof(DevState) % 8 == 0, "the state is cleared word by word");
  if (blockIdx.x == 0)
    for (unsigned i = threadIdx.x; i < sizeof(DevState) / 8; i += kBlock) w[i] = i == kAt ? kPayloadUnset : 0ull;
  const u64x2 empty = {kEmptyKey, kPayloadUnset};
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < cap; i += stride)
    *reinterpret_cast<u64x2*>(&slots[i]) = empty;
}

// One wavefront per table (blockIdx.x).
struct StateBatch {
  const DevState* st[kMaxBatch];
  StateView* out[kMaxBatch];
  unsigned long long seq;
};
__global__ void k_read_state(StateBatch sb) {
  const DevState* st = sb.st[blockIdx.x];
  StateView* out = sb.out[blockIdx.x];
  unsigned long long c = threadIdx.x < kCountShards ? st->count_shard[threadIdx.x * kShardStride] : 0ull;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
  if (threadIdx.x != 0) return;
  out->count = c;
  out->arena_top = st->arena_top;
  out->scan_total = st->scan_total;
  out->same_epoch = st->same_epoch;
  out->error = st->error;
  out->req_error = st->req_error;
  out->special_present = st->special_present;
  __hip_atomic_store(&out->seq, sb.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The parts of a table that have one size whatever the table holds: device state, the pinned words and
// request buffers, events, its stream. Creating them costs the calling thread about a millisecond (every
// pinned allocation and its release go through the driver), so a table that goes leaves its shell to
// the next one: up to kShellsKept per device (2.1 MiB of pinned memory each), given back by pskv_device_trim, and
// some time after the last table of the device has gone.
struct Shell {
  DevState* st = nullptr;
  char* pinned = nullptr;  // StateView, Snapshot, outcome word, done word (256 bytes each), small_in, small_out
  hipEvent_t done[kSmallParts] = {nullptr};
};
constexpr size_t kShellsKept = 32;

struct ShellPool {
  std::mutex mu;
  std::vector<Shell*> idle;
};
ShellPool g_shells[64];

void shell_free(Shell* sh) {
  if (!sh) return;
  if (sh->st) (void)hipFree(sh->st);
  if (sh->pinned) (void)hipHostFree(sh->pinned);
  for (hipEvent_t e : sh->done)
    if (e) (void)hipEventDestroy(e);
  delete sh;
}

// A shell for a table on `device` (current): one whose last table is gone (nothing on the GPU uses it any
// more) if there is one.
Shell* shell_take(int device) {
  Shell* sh = nullptr;
  if (device < 64) {
    ShellPool& p = g_shells[device];
    std::lock_guard<std::mutex> lk(p.mu);
    if (!p.idle.empty()) {
      sh = p.idle.back();
      p.idle.pop_back();
    }
  }
  if (!sh) {
    sh = new (std::nothrow) Shell();
    if (!sh) return nullptr;
    // coherent: the GPU does not cache this memory, so each request sees what the host just wrote
    bool ok = hipMalloc(reinterpret_cast<void**>(&sh->st), sizeof(DevState)) == hipSuccess &&
              hipHostMalloc(reinterpret_cast<void**>(&sh->pinned), 1024 + 2 * kSmallBytes, hipHostMallocCoherent) ==
                  hipSuccess;
    for (int q = 0; ok && q < kSmallParts; ++q)
      ok = hipEventCreateWithFlags(&sh->done[q], hipEventDisableTiming) == hipSuccess;
    if (!ok) {
      shell_free(sh);
      return nullptr;
    }
  }
  return sh;
}

void shell_give(int device, Shell* sh) {
  if (!sh) return;
  if (device < 64 && arrays_are_kept()) {
    ShellPool& p = g_shells[device];
    std::lock_guard<std::mutex> lk(p.mu);
    if (p.idle.size() < kShellsKept) {
      p.idle.push_back(sh);
      return;
    }
  }
  shell_free(sh);
}

// With `device` current: idle shells go.
void shell_trim(int device) {
  std::vector<Shell*> go;
  {
    ShellPool& p = g_shells[device];
    std::lock_guard<std::mutex> lk(p.mu);
    go.swap(p.idle);
  }
  for (Shell* sh : go) shell_free(sh);
}

// The streams of tables that were not given one. A process has four hardware queues, and a stream is put on the one that
// the fewest streams are on when it is made, used or not: streams that are made one by one, as tables come and go, end
// up anywhere, and tables whose streams share a queue run one after the other. Four that are made together lie on one
// queue each, so they are, and a new table gets a stream of the place among the four that the fewest tables are on.
// (Three tables of 200,000 rows in turn, other rows in every step: 196 us a step on a queue each, 223 on the same one.)
// They stay when their tables go: they are no memory, and the ones that took their place might lie elsewhere.
constexpr int kQueues = 4;
struct StreamPool {
  std::mutex mu;
  struct Entry {
    hipStream_t stream;
    int place;
    bool used;
  };
  std::vector<Entry> all;
};
StreamPool g_streams[64];

// A stream for a table on `device` (current), or null.
hipStream_t stream_take(int device) {
  hipStream_t alone = nullptr;
  if (device >= 64) return hipStreamCreateWithFlags(&alone, hipStreamNonBlocking) == hipSuccess ? alone : nullptr;
  StreamPool& p = g_streams[device];
  std::lock_guard<std::mutex> lk(p.mu);
  int used[kQueues] = {0};
  for (const StreamPool::Entry& e : p.all) used[e.place] += e.used ? 1 : 0;
  auto best = [&]() -> StreamPool::Entry* {
    StreamPool::Entry* b = nullptr;
    for (StreamPool::Entry& e : p.all)
      if (!e.used && (!b || used[e.place] < used[b->place])) b = &e;
    return b;
  };
  StreamPool::Entry* e = best();
  if (!e || used[e->place] > *std::min_element(used, used + kQueues)) {
    for (int q = 0; q < kQueues; ++q) {
      hipStream_t s = nullptr;
      if (hipStreamCreateWithFlags(&s, hipStreamNonBlocking) == hipSuccess)
        p.all.push_back({s, q, false});
      else
        (void)hipGetLastError();
    }
    e = best();
  }
  if (!e) return nullptr;
  e->used = true;
  return e->stream;
}

void stream_give(int device, hipStream_t stream) {
  if (device >= 64) {
    (void)hipStreamDestroy(stream);
    return;
  }
  StreamPool& p = g_streams[device];
  std::lock_guard<std::mutex> lk(p.mu);
  for (StreamPool::Entry& e : p.all)
    if (e.stream == stream) e.used = false;
}

// With `device` current: the streams that no table has go.
void stream_trim(int device) {
  if (device >= 64) return;
  StreamPool& p = g_streams[device];
  std::lock_guard<std::mutex> lk(p.mu);
  for (size_t i = p.all.size(); i-- > 0;) {
    if (p.all[i].used) continue;
    (void)hipStreamDestroy(p.all[i].stream);
    p.all.erase(p.all.begin() + (ptrdiff_t)i);
  }
}

// What tables that are gone have left (`device` is current).
void give_back(int device) {
  array_trim(device);
  if (device < 64) shell_trim(device);
}

}  // namespace
}  // namespace pskv

using namespace pskv;

struct pskv_table {
  int device = 0;
  int mode = PSKV_MODE_SCALAR;
  hipStream_t stream = nullptr;
  hipStream_t own_stream = nullptr;  // the same, where the table was not given one
  float max_load = 0.5f;

  Slot* slots = nullptr;
  uint64_t cap = 0;        // slots, a power of two
  // The array the next growth will move into, allocated ahead of need (once the table is 40 % of
  // the way to that growth) at the end of a request, while the GPU is busy with that request:
  // allocating costs the host 50-100 us, which would otherwise be spent with the GPU idle.
  Slot* spare = nullptr;
  uint64_t spare_cap = 0;
  std::shared_ptr<AllocJob> spare_job;  // the allocation of `spare` while it is under way
  // what the sizing logic did, printed when the table goes if PSKV_STATS is set in the environment
  struct Stats {
    uint64_t requests = 0, waits = 0, growths = 0, growths_unasked = 0, spare_used = 0, records = 0, catch_ups = 0;
    double alloc_us = 0, release_us = 0, catch_up_us = 0;  // host time spent allocating, releasing, catching up
    double ahead_us = 0;  // time the allocating thread spent on this table's arrays
  } stats;
  uint64_t count = 0;      // key count at the last read_state()

  // Host-side bounds of what the device counters can have reached. Requests are enqueued
  // without waiting, so the host only knows exact counters (`base_*`) as of request
  // `base_seq` and must assume that every key of a later request was new (`pend_*`).
  // A published snapshot (below) moves the base forward without a stream wait.
  uint64_t seq = 0;        // requests begun so far
  uint64_t base_seq = 0;   // base_count / base_top hold after all requests < base_seq
  uint64_t base_count = 0, base_top = 0;
  uint64_t pend_keys = 0, pend_units = 0;  // sums of the log over [base_seq, seq)
  static const int kLog = 64;
  uint64_t log_keys[kLog] = {0}, log_units[kLog] = {0};
  Snapshot* snap = nullptr;  // pinned host memory the device publishes into
  uint64_t record_seq = ~0ull;  // the newest request that was asked to publish its counters (all ones: none yet)
  uint64_t unrecorded_keys = 0;  // keys that requests behind it have named
  double new_share = 0.0;  // share of the keys named by requests that were new, over the latest records
  bool share_known = false;  // (a record has said so)
  DevState* st = nullptr;  // device
  StateView* st_host = nullptr;  // pinned: what read_state() last read of the device state

  // row modes
  float* arena = nullptr;
  uint64_t arena_cap = 0;  // floats
  uint64_t row_len = 0;    // FIXED

  GrowBuf ws;         // per-request workspace (row references, offsets; SCALAR: keys by bin, stream_push.h)
  GrowBuf tiles;      // VARLEN: first key of every request-side tile
  GrowBuf tiles_aff;  // VARLEN: one TileNote per tile
  Shell* shell = nullptr;     // what st, st_host, snap, outcome and small_* belong to
  char* small_in = nullptr;   // pinned, kSmallBytes: small host-resident requests, read in place
  char* small_out = nullptr;  // pinned, kSmallBytes: their responses, written in place
  // A small host-resident SCALAR push returns once its kernel is queued: nothing comes back from
  // it. Requests of up to kSmallPart bytes take their room in small_in one behind the other, so that
  // as many pushes as fit can be in flight. An event is left when a part has been used up and
  // waited for when the part comes round again: one event for 21 pushes of 1,000 keys (an event behind
  // every push cost the calling thread 3.6 us of its 11.5).
  hipEvent_t small_done[kSmallParts] = {nullptr};
  bool small_pending[kSmallParts] = {false};  // the part's event has been recorded and not been waited for
  int small_part = 0;             // the part that is being used up,
  size_t small_at = 0;            // and the bytes of it that have been given away
  bool small_in_flight = false;   // requests that nobody has waited for may still be reading small_in
  unsigned long long* done = nullptr;  // pinned: done_seq of the newest request that had to tell its end
  unsigned long long done_seq = 0;
  GrowBuf stage;      // device copies of host-resident request buffers
  GrowBuf stage_out;  // device-side response of a host-resident or undersized pull
  bool no_growth = false;  // set while dumping: every key is known to be present
  // Recorded requests (pskv_replay_*): `gen` counts the requests that went the ordinary way, each
  // of which may move a buffer, refill the key cache or write cached values back, so a recording
  // only runs while `gen` is what it was when the recording was made. `capturing`: the table's
  // stream is being captured into a HIP graph, nothing may be allocated, waited for or timed.
  uint64_t gen = 0;
  bool capturing = false;

  // Row modes: the workspace keeps the row references, offsets and tile table of the last
  // request that computed them, and the key cache keeps that request's keys and lens, so a
  // request with the same keys (the usual case for a parameter server) can skip the lens
  // scan and every hash probe. The device decides whether the keys match; these fields only
  // say whether the buffers still have the shape the cached request gave them.
  GrowBuf cache_keys, cache_lens;
  bool cache_valid = false;
  uint64_t cache_n = 0, cache_nvals = 0;
  uint64_t known_n = 0;  // FIXED: positions of cache_keys whose reference in the workspace belongs to the key there
  uint64_t epoch = 0;  // number of the last request that took part in this

  // SCALAR: the same idea with the VALUES of the cached keys kept in request order (and the
  // slot number of every key), so that a request which repeats the cached key set streams
  // through `sc_vals` and touches no slot; the slots are brought up to date before anything
  // else reads or changes them (`sc_dirty`: they may be behind).
  GrowBuf sc_vals, sc_slots;
  bool sc_dirty = false;
  uint64_t sc_last_n = 0;   // keys of the previous request: a size that repeats is worth recording
  int sc_last_kind = -1;    // and its kind (0: push or push+pull, 1: pull)
  unsigned sc_pairs = 0;    // pulls in a row (up to 2) that came right behind a push of their own size
  // What the comparisons of the two kinds of requests (0: pushes and push+pulls, 1: pulls) have
  // come to lately: pushes that bring new keys every time may still leave a cache behind that the
  // pull after each of them is served from.
  struct ScTrack {
    unsigned fail = 0;  // comparisons in a row that found other keys
    unsigned skip = 0;  // requests of this kind left to run without a comparison after such failures
    bool hit = false;   // the newest comparison of this kind found the cached keys
  } sc_track[2];
  static const int kScKinds = 64;
  unsigned char sc_kind[kScKinds] = {0};  // kind of the request with number e, at e % kScKinds
  unsigned long long* outcome = nullptr;  // pinned: epoch << 1 | same of the newest comparison; VARLEN: whether pushes have ragged rows
  unsigned long long sc_seen = 0;         // the value of *outcome the host last looked at
  unsigned push_looks = 0;                // k_fixed_own: how often a workgroup looks for the verdict
  uint64_t sc_min_keys = 0;               // requests below this size leave the cache alone; 0 = no cache
  // which pushes stream through the slot array (stream_push.h); PSKV_STREAM=0 and =1, read when a table is created, are for tests
  enum class Streams { kNever, kWhereItPays, kWhereItFits } streams = Streams::kWhereItPays;
  uint64_t pack_min_keys = 0;             // cached keys of at least this many are packed
  bool packing = false;                   // a comparison has been asked to pack the cached keys (PackedKeys)
  unsigned stream_turn = 0;               // the counter of left keys that the newest of them used

  bool prof = false;
  std::vector<EventPair> pending[PSKV_KERNEL_COUNT];
  std::vector<EventPair> free_events;
  uint64_t launches[PSKV_KERNEL_COUNT] = {0};
  double total_ms[PSKV_KERNEL_COUNT] = {0};
  std::vector<float> samples[PSKV_KERNEL_COUNT];  // per-launch durations, bounded
};

namespace {

// ---- profiling -------------------------------------------------------------------
// Launches `kernel` on the table's stream. While profiling is on, the launch carries
// a start and a stop event of its own (hipExtLaunchKernel), which take the
// begin/end timestamps of that very dispatch: the same clock a profiler reads,
// without the idle time that events recorded around a launch would add.
hipError_t launch_args(pskv_table* t, int prof_kernel, const void* kernel, dim3 grid, dim3 block, size_t lds,
                       void** args) {
  if (t->prof && prof_kernel >= 0 && !t->capturing) {
    EventPair ev;
    bool have = false;
    if (!t->free_events.empty()) {
      ev = t->free_events.back();
      t->free_events.pop_back();
      have = true;
    } else if (hipEventCreate(&ev.a) == hipSuccess) {
      if (hipEventCreate(&ev.b) == hipSuccess) {
        have = true;
      } else {
        (void)hipEventDestroy(ev.a);
      }
    }
    if (have) {
      t->pending[prof_kernel].push_back(ev);
      return hipExtLaunchKernel(kernel, grid, block, args, lds, t->stream, ev.a, ev.b, 0);
    }
  }
  return hipLaunchKernel(kernel, grid, block, args, lds, t->stream);
}

template <typename... KArgs, typename... Args>
int launch(pskv_table* t, int prof_kernel, void (*kernel)(KArgs...), dim3 grid, dim3 block, size_t lds,
           Args... given) {
  std::tuple<KArgs...> as_declared(static_cast<KArgs>(given)...);
  return std::apply(
      [&](KArgs&... a) {
        void* args[] = {static_cast<void*>(&a)...};
        PSKV_HIP(launch_args(t, prof_kernel, reinterpret_cast<const void*>(kernel), grid, block, lds, args));
        return PSKV_OK;
      },
      as_declared);
}

int prof_collect(pskv_table* t) {
  PSKV_HIP(hipStreamSynchronize(t->stream));
  for (int k = 0; k < PSKV_KERNEL_COUNT; ++k) {
    for (const EventPair& ev : t->pending[k]) {
      float ms = 0.f;
      if (hipEventElapsedTime(&ms, ev.a, ev.b) == hipSuccess) {
        t->total_ms[k] += ms;
        t->launches[k] += 1;
        if (t->samples[k].size() < kMaxProfSamples) t->samples[k].push_back(ms);
      }
      t->free_events.push_back(ev);
    }
    t->pending[k].clear();
  }
  return PSKV_OK;
}

// ---- memory ----------------------------------------------------------------------
// Carves aligned pieces out of a GrowBuf that was grown to the total beforehand.
struct Carver {
  char* base;
  size_t at = 0;
  explicit Carver(void* p) : base(static_cast<char*>(p)) {}
  template <typename T>
  T* take(size_t count) {
    T* r = reinterpret_cast<T*>(base + at);
    at += (count * sizeof(T) + 255) & ~(size_t)255;
    return r;
  }
  static size_t need(size_t count, size_t elem) { return (count * elem + 255) & ~(size_t)255; }
};

// What the host keeps of a state that k_read_state has just written (the stream is idle).
void adopt_state(pskv_table* t) {
  const uint64_t c = t->st_host->count;
  t->count = c;
  // everything enqueued so far is complete: the bounds become exact
  t->base_seq = t->seq;
  t->base_count = c;
  t->base_top = t->st_host->arena_top;
  t->pend_keys = t->pend_units = 0;
}

// Reads the device state of up to kMaxBatch tables on one stream, with one launch and one wait. `watch`: what the
// caller wants to see afterwards lies in pinned memory (the state itself, answers that kernels have written
// there): it is enough that this kernel, the last one on the stream, has run.
std::atomic<unsigned long long> g_readings{0};
int read_states(pskv_table* const* tables, size_t count, bool watch) {
  StateBatch sb;
  sb.seq = ++g_readings;
  for (size_t i = 0; i < count; ++i) {
    sb.st[i] = tables[i]->st;
    sb.out[i] = tables[i]->st_host;
  }
  k_read_state<<<dim3((unsigned)count), dim3(64), 0, tables[0]->stream>>>(sb);
  PSKV_HIP(hipGetLastError());
  bool seen = watch;
  for (size_t i = 0; seen && i < count; ++i) seen = seen_in_time(&tables[i]->st_host->seq, sb.seq);
  if (!seen) PSKV_HIP(hipStreamSynchronize(tables[0]->stream));
  for (size_t i = 0; i < count; ++i) adopt_state(tables[i]);
  return PSKV_OK;
}

int read_state(pskv_table* t, bool watch = false) { return read_states(&t, 1, watch); }

// Turns device error bits into a status, clearing them on the device.
int report_device_errors(pskv_table* t) {
  const unsigned bits = t->st_host->error | t->st_host->req_error;
  if (!bits) return PSKV_OK;
  PSKV_HIP(hipMemsetAsync(&t->st->error, 0, 2 * sizeof(unsigned), t->stream));
  PSKV_HIP(hipStreamSynchronize(t->stream));
  if (bits & kDevErrFull) return set_error(PSKV_ENOMEM, "slot array full (internal sizing error)");
  if (bits & kDevErrReplay)
    return set_error(PSKV_ESTALE, "a replayed request no longer named the keys it was recorded with (or was held up for "
                                  "good): that run of it changed and answered nothing on this table");
  if (bits & kDevErrBadLen)
    return set_error(PSKV_EINVAL, "a length is negative or above PSKV_MAX_VARLEN_ROW");
  if (bits & kDevErrSizeMismatch)
    return set_error(PSKV_ESIZE_MISMATCH, "lens do not add up to the number of values");
  if (bits & kDevErrDuplicate)
    return set_error(PSKV_EINVAL, "a request held the same key twice (keys must be unique)");
  if (bits & kDevErrNoRoom)
    return set_error(PSKV_ESIZE_MISMATCH, "a var-len pull response did not fit the caller's buffer");
  return set_error(PSKV_ELEN_CHANGED, "a pushed row length differs from the stored length");
}

// (not filled: whoever asks for the array writes every slot of it)
int alloc_slots(uint64_t cap, Slot** out, hipStream_t stream) {
  return array_alloc(reinterpret_cast<void**>(out), cap * sizeof(Slot), stream);
}

int grow(pskv_table* t, GrowBuf* b, size_t bytes) {
  if (bytes <= b->bytes) return PSKV_OK;
  if (t->capturing) return set_error(PSKV_ESTALE, "a recorded request needs a buffer that its first run did not leave");
  // An eighth to spare (up to 32 MB): the slices of a worker's requests differ by a few keys from one
  // request to the next, and a reallocation costs the calling thread several requests' worth when the
  // pool has to ask the system, every time a table sees its largest slice so far.
  size_t want = std::max(bytes + std::min<size_t>(bytes / 8, (size_t)32 << 20), b->bytes + b->bytes / 2);
  want = (want + 4095) & ~(size_t)4095;
  if (b == &t->ws || b == &t->tiles || b == &t->tiles_aff || b == &t->cache_keys ||
      b == &t->cache_lens || b == &t->sc_vals || b == &t->sc_slots)
    t->cache_valid = false;  // the contents do not survive a reallocation
  // (earlier requests on the stream may still read the old buffer)
  int rc = array_release(b->ptr, t->stream);
  if (rc) return rc;
  b->ptr = nullptr;
  b->bytes = 0;
  rc = array_alloc(&b->ptr, want, t->stream);
  if (rc) return rc;
  // the staging buffers are filled and read by copy streams, which know nothing of this stream's order
  if (b == &t->stage || b == &t->stage_out) PSKV_HIP(hipStreamSynchronize(t->stream));
  b->bytes = want;
  return PSKV_OK;
}

// Gives back what grow() took.
int drop(pskv_table* t, GrowBuf* b) {
  void* const gone = b->ptr;
  b->ptr = nullptr;
  b->bytes = 0;
  return array_release(gone, t->stream);
}

// Moves the base of the bounds forward to the newest record the device has published: the
// counters after request `s1`.
void adopt_snapshot(pskv_table* t) {
  const Snapshot* sn = t->snap;
  const uint64_t s1 = sn->seq, count = sn->count, units = sn->arena_top;
  if (count >> kRecordTagAt != (record_word(0, s1) >> kRecordTagAt) || units >> kRecordTagAt != count >> kRecordTagAt) return;
  if (s1 < t->base_seq || s1 >= t->seq) return;  // (the initial record is all ones)
  const uint64_t c = count & (((uint64_t)1 << kRecordTagAt) - 1), top = units & (((uint64_t)1 << kRecordTagAt) - 1);
  uint64_t named = 0;
  for (uint64_t r = t->base_seq; r <= s1; ++r) {
    named += t->log_keys[r % pskv_table::kLog];
    t->pend_keys -= t->log_keys[r % pskv_table::kLog];
    t->pend_units -= t->log_units[r % pskv_table::kLog];
  }
  // which share of the keys that requests named turned out to be new, lately (a moving average)
  if (named) {
    const double share = c > t->base_count ? std::min(1.0, (double)(c - t->base_count) / (double)named) : 0.0;
    t->new_share = t->share_known ? 0.5 * t->new_share + 0.5 * share : share;
    t->share_known = true;
  }
  t->base_seq = s1 + 1;
  t->base_count = c;
  t->base_top = top;
}

// SCALAR: brings the slots up to date with the values of the key cache. Enqueued before
// anything but the kernels of a request that repeats the cached keys looks at the slots.
int flush_scalar_cache(pskv_table* t) {
  if (!t->sc_dirty) return PSKV_OK;
  HeadBatch<1> rb;
  std::memset(&rb, 0, sizeof(rb));
  TableHead& d = rb.t[0];
  d.slots = t->slots;
  d.mask = t->cap - 1;
  d.st = t->st;
  d.n = t->cache_n;
  d.arena = static_cast<float*>(t->sc_vals.ptr);
  d.tile_key = static_cast<uint32_t*>(t->sc_slots.ptr);
  d.nblk = grid_for(t->cache_n, kBlock, kFlushGrid);
  hipLaunchKernelGGL(k_scalar_flush, dim3(d.nblk, 1), dim3(kBlock), 0, t->stream, rb);
  PSKV_HIP(hipGetLastError());
  t->sc_dirty = false;
  return PSKV_OK;
}

// Takes over the array that the allocating thread was asked for, if it is there (`wait`: or
// once it is there).
void collect_spare(pskv_table* t, bool wait) {
  if (!t->spare_job) return;
  if (wait) {
    const auto w0 = std::chrono::steady_clock::now();
    alloc_wait(t->spare_job);
    t->stats.alloc_us += std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - w0).count();
  } else if (!alloc_finished(t->spare_job)) {
    return;
  }
  t->stats.ahead_us += t->spare_job->took_us;
  if (t->spare_job->rc == PSKV_OK && t->spare_job->ptr) {
    t->spare = static_cast<Slot*>(t->spare_job->ptr);
  } else {
    t->spare_cap = 0;  // (the growth will ask again itself and report)
  }
  t->spare_job.reset();
}

// The slots a growth goes to when the table has to hold `keys_needed` keys: at least twice the
// slots; four or eight times while that stays a small array (a table that starts at the default size and
// keeps growing then moves its keys a half or a third as often on the way up).
uint64_t grown_cap(const pskv_table* t, uint64_t keys_needed) {
  const uint64_t want = next_pow2((uint64_t)((double)keys_needed / t->max_load) + 1);
  uint64_t factor = 2;
  while (factor < (uint64_t)kRegrowMaxFactor && t->cap * factor * 2 * sizeof(Slot) <= kSlackBytes) factor *= 2;
  return std::max(want, t->cap * factor);
}

// The slot arrays that are to move for a request (growths.h). They do so before anything else of it, when move() is called or,
// where it ends early, when the list goes.
struct Growths {
  std::vector<Growth<pskv_table, Slot>> list;
  int move();
  ~Growths() { (void)move(); }
};

struct GrowthLaunches {
  int scatter(const Growth<pskv_table, Slot>& g) {  // (a small table that a large request makes much larger)
    pskv_table* t = g.t;
    PSKV_HIP(hipMemsetAsync(t->slots, 0xFF, t->cap * sizeof(Slot), t->stream));
    return launch(t, PSKV_KERNEL_REHASH, k_rehash, dim3(grid_for(g.cap, kBlock, kMaxGrid)), dim3(kBlock), 0,
                  (const Slot*)g.from, g.cap, t->slots, t->cap - 1, t->st);
  }
  // two streaming passes: the new array is written whole, slot by slot, from LDS
  int stream(Growth<pskv_table, Slot>* const* some, unsigned count, bool& begun) {
    RegrowBatch b;
    std::memset(&b, 0, sizeof(b));
    pskv_table* lead = some[0]->t;
    uint64_t most = 0, factors = 0;
    for (unsigned i = 0; i < count; ++i) {
      const Growth<pskv_table, Slot>& g = *some[i];
      const uint64_t factor = g.t->cap / g.cap;
      b.t[i] = RegrowOf{g.from, g.t->slots, g.cap - 1, g.t->cap - 1, g.t->st, factor, kRegrowOld};
      most = std::max(most, g.cap);
      factors = std::max(factors, factor);
    }
    const unsigned nblk = (unsigned)(most / kRegrowOld);
    const size_t lds = (size_t)kRegrowOld * factors * 2 * sizeof(unsigned long long);
    int rc = launch(lead, PSKV_KERNEL_REHASH, k_regrow, dim3(nblk, count), dim3(kBlock), lds, b);
    if (rc) return rc;
    begun = true;
    return launch(lead, PSKV_KERNEL_REHASH, k_regrow_rest, dim3((nblk * kRestLanes + kBlock - 1) / kBlock, count),
                  dim3(kBlock), 0, b);
  }
  int release(pskv_table* t, Slot* slots) {
    const auto r0 = std::chrono::steady_clock::now();
    const int rc = array_release(slots, t->stream);
    t->stats.release_us += std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - r0).count();
    return rc;
  }
};

int Growths::move() {
  if (list.empty()) return PSKV_OK;
  std::vector<Growth<pskv_table, Slot>> todo;
  todo.swap(list);
  GrowthLaunches launches;
  return move_growths(todo, (unsigned)kMaxBatch, (uint64_t)kRegrowMaxFactor, launches);
}

int grow_slots(pskv_table* t, uint64_t keys_needed, Growths* growths) {
  uint64_t want = grown_cap(t, keys_needed);
  Slot* fresh = nullptr;
  int rc = PSKV_OK;
  if (t->mode == PSKV_MODE_SCALAR) {
    // the key cache holds slot numbers of the old array, and values the old array may lack
    rc = flush_scalar_cache(t);
    if (rc) return rc;
    t->cache_valid = false;
  }
  ++t->stats.growths;
  collect_spare(t, true);
  struct {
    pskv_table* t;
    bool allocated;
    int release(Slot* slots) { return array_release(slots, t->stream); }
    int allocate(uint64_t n, Slot** to) {
      allocated = true;
      const auto a0 = std::chrono::steady_clock::now();
      const int rc = alloc_slots(n, to, t->stream);
      t->stats.alloc_us += std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - a0).count();
      return rc;
    }
  } arrays{t, false};
  rc = next_array(t->spare, t->spare_cap, want, fresh, arrays);
  if (rc) return rc;
  if (!arrays.allocated) ++t->stats.spare_used;
  growths->list.push_back({t, t->slots, t->cap, false});
  t->slots = fresh;
  t->cap = want;
  return PSKV_OK;
}

// Called at the end of a request, with its kernels queued: allocates the array of the next growth
// once the keys the table is known to hold have come 40 % of the way to that growth.
void prepare_growth(pskv_table* t) {
  if (t->spare || t->spare_job || t->no_growth) return;
  adopt_snapshot(t);  // (a read of pinned memory)
  const double limit = (double)t->max_load * (double)t->cap;
  // the keys known to be held, plus, while requests have mostly been bringing new keys, the share of
  // the keys in flight that will be new if that goes on (a caller that runs far ahead of the device
  // would otherwise learn too late how full the table is)
  const double expected = (double)t->base_count + (t->new_share >= 0.5 ? t->new_share * (double)t->pend_keys : 0.0);
  if (expected <= 0.4 * limit) return;
  const uint64_t want = grown_cap(t, 0);
  if (want * sizeof(Slot) > kSpareMaxBytes) return;
  std::shared_ptr<AllocJob> job = std::make_shared<AllocJob>();
  job->device = t->device;
  job->bytes = want * sizeof(Slot);
  job->stream = t->stream;
  t->spare_cap = want;
  t->spare_job = job;
  alloc_submit(job);
}

// Room behind an arena's last row: the row kernels read a row's last quad whole.
constexpr size_t kArenaEnd = 16;

int grow_arena(pskv_table* t, uint64_t floats_needed, uint64_t live_floats) {
  uint64_t want = std::max(floats_needed, t->arena_cap + t->arena_cap / 2);
  want = (want + 1023) & ~(uint64_t)1023;
  float* fresh = nullptr;
  int rc = array_alloc(reinterpret_cast<void**>(&fresh), want * sizeof(float) + kArenaEnd, t->stream);
  if (rc) return rc;
  if (live_floats && t->arena) {
    PSKV_HIP(hipMemcpyAsync(fresh, t->arena, live_floats * sizeof(float), hipMemcpyDeviceToDevice,
                            t->stream));
  }
  rc = array_release(t->arena, t->stream);
  t->arena = fresh;
  t->arena_cap = want;
  return rc;
}

// Begins a request that may create up to `n` keys and take up to `units` allocation units
// of the arena (rows for FIXED, 16 bytes for VARLEN; `floats_per_unit` converts to floats).
// Grows the slot array / the arena first if the bounds say they could overflow. The fast
// path touches no device state; the next best reads the snapshot the device published;
// only then does it wait for the stream and read the counters.
//
// Close to a limit the device publishes its counters as they are after the request, so that a
// later request can move the base forward without waiting for the stream: `pub->snap` is
// set when a record is wanted, and the caller hands it to the kernel of the request that
// changes the counters.
struct PublishReq {
  Snapshot* snap = nullptr;
  uint64_t seq = 0;
};

// The share of the keys in flight that is taken to be new: what the latest records say, a quarter more and a
// tenth, to be on the safe side; all of them while no record has said anything.
double new_share_at_most(const pskv_table* t) {
  return t->share_known ? std::min(1.0, 1.25 * t->new_share + 0.1) : 1.0;
}

int reserve(pskv_table* t, uint64_t n, uint64_t units, uint64_t floats_per_unit, PublishReq* pub, Growths* growths) {
  if (t->no_growth) return PSKV_OK;
  // Two limits. `limit` is the fill the table is kept below; `hard` (0.85 unless max_load is higher) is
  // the fill it must never exceed. The keys in flight count in full against the second, and against the
  // first with the share of them that is going to be new if requests go on as the latest records say
  // (new_share_at_most).
  // A server whose requests mostly name keys it holds, the steady state of a parameter server, then does
  // not grow, or wait, for keys that are not coming, however far ahead of the device its caller runs; if
  // the requests change their ways the table runs fuller than `limit` for as long as it takes the next
  // records to say so, never fuller than `hard`.
  const double limit = (double)t->max_load * (double)t->cap;
  const double hard = std::max((double)t->max_load, kHardLoad) * (double)t->cap;
  auto slots_short = [&]() {
    // (looked up on every call: a record adopted further down may have changed it)
    const double in_flight = (double)(t->pend_keys + n);
    return (double)t->base_count + in_flight > hard ||
           (double)t->base_count + new_share_at_most(t) * in_flight > limit;
  };
  auto arena_short = [&]() {
    return units && (t->base_top + t->pend_units + units) * floats_per_unit > t->arena_cap;
  };
  // an ageing base is refreshed from the newest record whenever one has arrived (a host read)
  if (t->seq - t->base_seq >= (uint64_t)pskv_table::kLog / 4) adopt_snapshot(t);
  if (slots_short() || arena_short() || t->seq - t->base_seq >= (uint64_t)pskv_table::kLog - 1) {
    adopt_snapshot(t);
    const bool old_log = t->seq - t->base_seq >= (uint64_t)pskv_table::kLog - 1;
    // (two requests of 16M keys that are left unaccounted for would make a 1 GiB array a 2 GiB one;
    // the host's lead is worth less than that: a few tens of microseconds of idle GPU, once)
    const uint64_t keep =
        grown_cap(t, t->base_count + t->pend_keys + n) * sizeof(Slot) >= kLargeArrayBytes ? 0 : kKeepInFlight;
    if (slots_short() && !arena_short() && !old_log && (double)(t->base_count + n) <= limit &&
        t->record_seq != ~0ull && t->record_seq >= t->base_seq && t->seq - t->base_seq > keep) {
      // The array is only short if the requests in flight create most of their keys, and some of
      // them are going to say how many they did create: the host lets the device catch up, but not
      // all the way (unless a large array is at stake). A caller that runs many requests ahead is held
      // back until only kKeepInFlight requests are unaccounted for (so the device never runs dry, as it would in a wait for the
      // stream, and the steps that follow do not run in lock-step with the host); if the array
      // still looks short then, it is replaced, at most that many requests early and sized for
      // at most that many requests of uncertainty.
      const auto t0 = std::chrono::steady_clock::now();
      unsigned spins = 0;
      while (slots_short() && (double)(t->base_count + n) <= limit && t->record_seq >= t->base_seq &&
             t->seq - t->base_seq > keep) {
        adopt_snapshot(t);
        if ((++spins & 63u) == 0) {
          if (std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(20)) break;
          std::this_thread::yield();
        }
      }
      ++t->stats.catch_ups;
      t->stats.catch_up_us += std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count();
    }
    if (slots_short() && !arena_short() && !old_log &&
        grown_cap(t, t->base_count + t->pend_keys + n) * sizeof(Slot) <= kGrowUnaskedBytes) {
      // Only the slots could run short, and the larger array is not a large one: it is taken now,
      // sized for what the requests in flight could create at most, without asking the device how
      // many keys they did create. The move is queued behind them; nothing waits.
      const uint64_t most = t->base_count + t->pend_keys + n;
      // (room for two more such requests while that keeps the array a small one)
      const uint64_t slack_n = grown_cap(t, most + 2 * n) * sizeof(Slot) <= kSlackBytes ? 2 * n : 0;
      int rc = grow_slots(t, most + slack_n, growths);
      if (rc) return rc;
      ++t->stats.growths_unasked;
    } else if (slots_short() || arena_short() || old_log) {
      int rc = read_state(t);  // exact counters, stream idle
      if (rc) return rc;
      ++t->stats.waits;
      // The wait happened because requests in flight had to be assumed to create all their
      // keys. Small tables get room for two more such requests, so that a caller who keeps
      // requests of this size in flight does not wait again on every one of them; for large
      // tables the wait is short next to their kernels and the memory is not.
      const uint64_t slack_n = grown_cap(t, t->base_count + 3 * n) * sizeof(Slot) <= kSlackBytes ? 2 * n : 0;
      const uint64_t slack_u = t->arena_cap * sizeof(float) <= kSlackBytes ? 2 * units : 0;
      if ((double)(t->base_count + n + slack_n) > limit) {
        rc = grow_slots(t, t->base_count + n + slack_n, growths);
        if (rc) return rc;
      }
      if (units && (t->base_top + units + slack_u) * floats_per_unit > t->arena_cap) {
        rc = grow_arena(t, (t->base_top + units + slack_u) * floats_per_unit,
                        t->base_top * floats_per_unit);
        if (rc) return rc;
      }
    }
  }
  const uint64_t q = t->seq++;
  t->log_keys[q % pskv_table::kLog] = n;
  t->log_units[q % pskv_table::kLog] = units;
  t->pend_keys += n;
  t->pend_units += units;
  // Close to a limit, as the latest records say how many of the keys in flight are going to be new, every
  // request leaves a record; from a third of the way to the next growth on, every fourth one does: the host then
  // knows how full the table is early enough to have the next array allocated by the time it is needed. The
  // election of a kernel's last workgroup costs a 1M-key launch about 6 us, so it is not made with every request for
  // the mere length of the queue: minibatches of keys that are all held left a record with 96 of 100 requests while
  // keys in flight counted in full here, as soon as the caller ran a dozen requests ahead (4 pushes and pulls of 1M of
  // 20M held keys: 281 us, with a record for every fourth 255). A long queue leaves them by the keys as well, one for
  // an eighth of the room below `hard`: a host that is held back there waits for the next record.
  const double limit_now = (double)t->max_load * (double)t->cap;
  const double hard_now = std::max((double)t->max_load, kHardLoad) * (double)t->cap;
  const double base = (double)t->base_count, ahead = (double)(t->pend_keys + 2 * n);
  t->unrecorded_keys += n;
  const bool tight_slots =
      base + new_share_at_most(t) * ahead > limit_now || (base + ahead > 0.35 * limit_now && q % 4 == 0) ||
      (base + ahead > limit_now && (double)t->unrecorded_keys > 0.125 * (hard_now - base));
  const bool tight_arena =
      units && (t->base_top + t->pend_units + 2 * units) * floats_per_unit > t->arena_cap;
  // (a base that merely grows old asks for a record every eighth request, not every one)
  const uint64_t age = t->seq - t->base_seq;
  const bool old_base = age >= (uint64_t)pskv_table::kLog / 4 && (age % 8 == 0 || age >= (uint64_t)pskv_table::kLog - 8);
  ++t->stats.requests;
  if (tight_slots || tight_arena || old_base) {
    pub->snap = t->snap;
    pub->seq = q;
    t->record_seq = q;
    t->unrecorded_keys = 0;
    ++t->stats.records;
  }
  return PSKV_OK;
}

// ---- request pipeline ------------------------------------------------------------
// One table's share of a request.
struct Request {
  bool push, pull;
  const uint64_t* keys;  // device
  uint64_t n;
  const float* vals;     // device
  uint64_t nvals;
  const int32_t* lens;   // device
  float* out;            // device
  uint64_t out_cap;
  int32_t* out_lens;     // device (VARLEN pull)
  uint64_t out_nvals;    // result
  bool lazy_out;         // VARLEN pull into host memory: `out` is allocated once the size is known
  bool need_total;       // VARLEN pull: the caller wants the response size back (forces a wait)
  char* small_out;       // lazy_out: pinned room the response may go to when it fits
  uint64_t small_out_floats;
  // Large host-resident requests (row modes). pipe_in: `vals` is room in device memory that the
  // row kernel fills itself, piece by piece, from `vals_host` while it works through the pieces
  // that have arrived. pipe_out: the gather kernel is not launched with the request; the caller
  // launches it piece by piece in step with the transfer of the response (gather_deferred says
  // that it is still owed, gather_varlen which kernel it is).
  bool pinned;               // keys, vals and lens lie in pinned host memory
  unsigned long long* done;  // SCALAR, pinned: the word that takes done_seq when the request is done, or null
  unsigned long long done_seq;
  const float* vals_host;
  bool pipe_in, pipe_out, gather_deferred, gather_varlen;
  // pskv_replay_record: kReplayPrime = the run that brings the tables into the state a repeat of the
  // request finds (the key cache is filled whatever the size of the request and whatever earlier
  // comparisons came to); kReplayCapture = the launches of such a repeat, recorded, not run.
  int replay;
};
constexpr int kReplayPrime = 1, kReplayCapture = 2;

// A request as the kernels see it: the shares of up to kMaxBatch tables that live on one device,
// work in one mode and run on one stream, served by ONE launch per step of the pipeline. The
// single-table entry points run a batch of one; pskv_push_multi / pskv_pull_multi hand over all
// key ranges of a sliced request at once.
struct Item {
  pskv_table* t = nullptr;
  Request r{};
  TableReq d{};
  PublishReq pub;
  ReqTag tag{};
  // var-len workspace of the request
  int32_t* tmp_lens = nullptr;
  uint64_t nparts = 0, tiles_cap = 0;
};
typedef std::vector<Item> Batch;

// The table whose stream the batch runs on and whose launch statistics it is booked to.
pskv_table* lead_of(Batch& bt) {
  for (Item& it : bt)
    if (it.t->prof) return it.t;
  return bt[0].t;
}

// One kernel of the store in its three sizes (ReqBatch, or HeadBatch: `head`).
struct KernelSet {
  const void* one;
  const void* four;
  const void* most;
  bool head;
};
template <typename B>
constexpr bool takes_heads(void (*)(B)) { return false; }
template <int TABLES>
constexpr bool takes_heads(void (*)(HeadBatch<TABLES>)) { return true; }
#define PSKV_KSET(name)                                                                                        \
  (KernelSet{reinterpret_cast<const void*>(&name<1>), reinterpret_cast<const void*>(&name<4>),                   \
             reinterpret_cast<const void*>(&name<kMaxBatch>), takes_heads(&name<1>)})
#define PSKV_KSET_OF(name, ...)                                                                                \
  (KernelSet{reinterpret_cast<const void*>(&name<__VA_ARGS__, 1>), reinterpret_cast<const void*>(&name<__VA_ARGS__, 4>), \
             reinterpret_cast<const void*>(&name<__VA_ARGS__, kMaxBatch>), takes_heads(&name<__VA_ARGS__, 1>)})

// A launch as pskv_replay_record keeps it: everything it takes to make it again.
struct SavedLaunch {
  const void* kernel;
  dim3 grid, block;
  union {  // (the kernel takes as much of it as its size says)
    ReqBatch<kMaxBatch> rb;
    HeadBatch<kMaxBatch> heads;
  };
};
// Where launch_batch leaves a copy of its launches while a request is being recorded (the thread
// that records is the thread that launches).
thread_local std::vector<SavedLaunch>* g_recording = nullptr;

// One launch for the whole batch: blockIdx.y selects the table, `nblk_of` says how many
// workgroups serve each (0: none, the table sits this step out).
template <typename F>
int launch_batch(Batch& bt, int prof_kernel, const KernelSet& kernels, F nblk_of, unsigned threads = kBlock) {
  SavedLaunch l;
  const size_t room = bt.size() <= 1 ? 1 : bt.size() <= 4 ? 4 : kMaxBatch;
  l.kernel = room == 1 ? kernels.one : room == 4 ? kernels.four : kernels.most;
  uint64_t gx = 0;
  for (size_t i = 0; i < bt.size(); ++i) {
    const uint64_t nb = nblk_of(bt[i]);
    if (nb > 0x7fffffffull) return set_error(PSKV_EINVAL, "request too large");
    bt[i].d.nblk = (uint32_t)nb;
    if (kernels.head) l.heads.t[i] = bt[i].d; else l.rb.t[i] = bt[i].d;
    gx = std::max(gx, nb);
  }
  if (!gx) return PSKV_OK;
  l.grid = dim3((unsigned)gx, (unsigned)bt.size());
  l.block = dim3(threads);
  void* args[] = {&l.rb};
  PSKV_HIP(launch_args(lead_of(bt), prof_kernel, l.kernel, l.grid, l.block, 0, args));
  if (g_recording) g_recording->push_back(l);
  return PSKV_OK;
}

int read_state_batch(Batch& bt, bool watch) {
  pskv_table* tables[kMaxBatch];
  for (size_t i = 0; i < bt.size(); ++i) tables[i] = bt[i].t;
  return read_states(tables, bt.size(), watch);
}

// What the device has reported about the comparisons of earlier requests with the cached keys
// (a pinned word, read whenever the host gets here, never waited for): comparisons that keep
// finding other keys switch the comparison off for 2, 4, ... 64 requests of that kind.
void note_outcomes(pskv_table* t) {
  const unsigned long long seen = *static_cast<volatile unsigned long long*>(t->outcome);
  if (seen == t->sc_seen) return;
  t->sc_seen = seen;
  const unsigned long long e = seen >> 1;
  if (e + pskv_table::kScKinds <= t->epoch) return;  // the note of its kind has been overwritten
  pskv_table::ScTrack& tr = t->sc_track[t->sc_kind[e % pskv_table::kScKinds] & 1];
  if (seen & 1ull) {
    tr.fail = 0;
    tr.hit = true;
  } else {
    tr.fail = std::min(tr.fail + 1u, 6u);
    tr.skip = 1u << tr.fail;
    tr.hit = false;
    t->packing = false;
  }
}

// Numbers a request that takes part in the key cache and says whether the key cache has the
// right shape for it. Row modes (`back_off`): a request of the right shape is still not compared
// while comparisons of its kind (pushes, pulls) are in a spell of finding other keys, as the
// requests of an embedding table do that names other rows in every batch; the request then goes
// the general way, which leaves its keys behind as the new cache all the same.
ReqTag next_tag(pskv_table* t, const Request& r, bool back_off = false) {
  ReqTag tag;
  tag.epoch = ++t->epoch;
  tag.replay = r.replay == kReplayCapture ? 1u : 0u;
  bool compare = t->cache_valid && t->cache_n == r.n;
  if (back_off && compare && !r.replay) {
    note_outcomes(t);
    const int kind = r.push ? 0 : 1;
    pskv_table::ScTrack& tr = t->sc_track[kind];
    if (tr.skip) {
      --tr.skip;
      compare = false;
    } else {
      t->sc_kind[tag.epoch % pskv_table::kScKinds] = (unsigned char)kind;
    }
  }
  tag.try_cache = compare ? kTryKeys : 0u;
  return tag;
}

// SCALAR requests of at least this many keys may use the key cache (below that a request is a
// single short launch either way, and the cache would add two). The environment variable
// PSKV_SCALAR_CACHE_MIN_KEYS, read when a table is created, overrides it (0 switches the cache off).
constexpr uint64_t kScalarCacheMinKeys = 1u << 17;

// Cached keys of at least this many are packed once a request has repeated them (12 MB of them: the time of smaller ones is the
// launches', and the comparison of packed ones starts a little later: push and pull of 1.06M keys 19.8 -> 21.9 us, of 1.25M 21.3 -> 21.5-22.2,
// of 1.5M 22.6 -> 22.4, of 1.75M 24.0 -> 23.8, of 2M 25.6 -> 24.9). The environment variable PSKV_PACK_MIN_KEYS, read when a table
// is created, is for tests. Figures: PackedKeys. Room for it, 6 B per key, is taken when such a request is recorded in the key cache; keys that a
// recorded step left there (pskv_replay_*, which never packs) have none.
constexpr uint64_t kPackKeys = 3u << 19;

// How a SCALAR request of one table relates to the table's key cache.
enum ScalarCacheUse {
  kScPlain,   // neither uses nor fills it
  kScRecord,  // served through the slots; leaves its keys, values and slot numbers as the new cache
  kScTry,     // compared with the cached keys on the device: served from the cache if they match,
              // like kScRecord otherwise
};

// Decides it from what the host knows without waiting for the device: a request whose size
// repeats the previous one is worth recording, a request of the cached size is worth comparing,
// and comparisons that keep finding other keys (reported by the device through a pinned word,
// read whenever the host gets here) switch the comparison off for a growing number of requests
// of that kind.
bool scalar_cache_eligible(const pskv_table* t, const Request& r) {
  return t->sc_min_keys && r.n >= t->sc_min_keys && t->cap < (1ull << 32);
}

// pulls have been following the pushes of their keys and are not in a spell of failed comparisons
bool pulls_follow(const pskv_table* t) { return t->sc_pairs >= 2 && t->sc_track[1].skip == 0; }

ScalarCacheUse scalar_cache_use(pskv_table* t, const Request& r) {
  note_outcomes(t);
  const int kind = r.push ? 0 : 1;
  // a worker that pushes gradients and pulls the weights of the same keys right away shows as a
  // pull behind a push of its own size, whatever that size is from one step to the next
  if (kind == 1 && t->sc_last_kind == 0)
    t->sc_pairs = r.n == t->sc_last_n ? std::min(t->sc_pairs + 1u, 2u) : 0u;
  ScalarCacheUse use = kScPlain;
  if (scalar_cache_eligible(t, r)) {
    pskv_table::ScTrack& tr = t->sc_track[kind];
    const bool compare = tr.skip == 0;
    if (!compare) --tr.skip;
    const bool size_repeats = r.n == t->sc_last_n;
    if (compare && t->cache_valid && t->cache_n == r.n) {
      use = kScTry;
    } else if (kind == 0) {
      // a push is worth recording when its size repeats (the same keys may be coming again) or
      // when pulls have been following the pushes
      if ((compare && size_repeats) || pulls_follow(t)) use = kScRecord;
    } else if (compare && size_repeats && t->sc_last_kind == 1) {
      use = kScRecord;  // a pull behind a pull of the same size
    }
  }
  t->sc_last_n = r.n;
  t->sc_last_kind = kind;
  return use;
}

// How a table's share of a SCALAR request is going to be served.
struct ScalarPlan {
  ScalarCacheUse use = kScPlain;
  int kind_before = -1;  // of the request in front of it (pskv_table::sc_last_kind)
  bool may_stream = false, streams = false;
};

// A table's share of a push that streams through its slot array.
struct Streamed {
  Item* it;
  Growth<pskv_table, Slot> g;  // of the table, if `grows`
  bool grows;
  StreamShape shape;
  uint32_t tiles() const { return (uint32_t)((it->r.n + kSplitTile - 1) / kSplitTile); }
};

size_t stream_room(const Streamed& s) {
  return Carver::need((size_t)s.tiles() * kTileWords, 8) +
         Carver::need((size_t)s.tiles() * (s.shape.bins + kStartsPad), 2) + Carver::need(s.it->r.n, sizeof(unsigned));
}

// Those tables' shares of a push; the slot arrays that move for it have been allocated, nothing has been moved.
int stream_push(Batch& bt, std::vector<Streamed>& todo) {
  pskv_table* lead = lead_of(bt);
  StreamBatch all;
  RegrowBatch rest;
  std::memset(&all, 0, sizeof(all));
  std::memset(&rest, 0, sizeof(rest));
  // the tables by what their arrays do: stay, become twice as large, or more
  struct Kind {
    StreamBatch b;
    unsigned tables = 0, most_bins = 0;
  } kinds[3];
  unsigned most_tiles = 0, n_grow = 0;
  uint64_t most_keys = 0, most_rest = 0;
  for (size_t i = 0; i < todo.size(); ++i) {
    Streamed& s = todo[i];
    Item& it = *s.it;
    pskv_table* t = it.t;
    StreamOf& d = all.t[i];
    d.slots = t->slots;
    d.mask = t->cap - 1;
    d.old_slots = s.grows ? s.g.from : t->slots;
    d.old_mask = (s.grows ? s.g.cap : t->cap) - 1;
    d.st = t->st;
    d.keys = it.r.keys;
    d.vals = it.r.vals;
    d.n = it.r.n;
    d.tiles = s.tiles();
    d.bins = s.shape.bins;
    d.bin_bits = s.shape.bin_bits;
    d.images = s.shape.images;
    Carver c(t->ws.ptr);
    d.parts = c.take<unsigned long long>((size_t)d.tiles * kTileWords);
    d.starts = c.take<uint16_t>((size_t)d.tiles * (d.bins + kStartsPad));
    d.left = c.take<unsigned>(it.r.n);
    d.snap = it.pub.snap;
    d.snap_seq = it.pub.seq;
    d.told = t->outcome + 1;
    d.turn = t->stream_turn ^= 1u;
    most_tiles = std::max(most_tiles, d.tiles);
    most_keys = std::max(most_keys, d.n);
    const uint64_t factor = s.grows ? t->cap / s.g.cap : 1;
    Kind& kind = kinds[factor == 1 ? 0 : factor == 2 ? 1 : 2];
    kind.b.t[kind.tables++] = d;
    kind.most_bins = std::max(kind.most_bins, d.bins);
    if (s.grows) {
      const uint64_t stretch = kImageSlots / factor;
      rest.t[n_grow++] = RegrowOf{s.g.from, t->slots, s.g.cap - 1, t->cap - 1, t->st, factor, stretch};
      most_rest = std::max(most_rest, s.g.cap / stretch);
    }
  }
  const unsigned tables = (unsigned)todo.size();
  int rc = launch(lead, PSKV_KERNEL_REHASH, k_split, dim3(most_tiles, tables), dim3(kSplitBlock), 0, all);
  void (*const kernels[3])(StreamBatch) = {k_stream_push<4>, k_stream_push<2>, k_stream_push<1>};
  bool begun[3] = {false, false, false};
  for (int k = 0; k < 3 && !rc; ++k) {
    if (!kinds[k].tables) continue;
    rc = launch(lead, PSKV_KERNEL_REHASH, kernels[k], dim3(kinds[k].most_bins, kinds[k].tables),
                dim3(kStreamBlock), 0, kinds[k].b);
    begun[k] = !rc;
  }
  if (!rc && n_grow)
    rc = launch(lead, PSKV_KERNEL_REHASH, k_regrow_rest, dim3((unsigned)((most_rest * kRestLanes + kBlock - 1) / kBlock), n_grow),
                dim3(kBlock), 0, rest);
  // (a lane for every 16th key would do where all of them were left; usually next to none is)
  if (!rc)
    rc = launch(lead, PSKV_KERNEL_REHASH, k_push_left, dim3(grid_for(most_keys, kBlock * 16, 512), tables), dim3(kBlock), 0, all);
  for (Streamed& s : todo) {
    pskv_table* t = s.it->t;
    if (rc) (void)hipMemsetAsync(t->st->left_keys, 0, sizeof(t->st->left_keys), t->stream);  // (what was left is not looked up)
    if (!s.grows) continue;
    Slot* gone = s.g.from;
    if (!begun[t->cap / s.g.cap == 2 ? 1 : 2]) {  // it keeps its old array, as in move_growths
      gone = t->slots;
      t->slots = s.g.from;
      t->cap = s.g.cap;
    }
    const int r = GrowthLaunches().release(t, gone);
    if (!rc) rc = r;
  }
  return rc;
}

// Picks the shares of a push that stream: out of `growths` the moves of their tables, which are part of it then. Takes
// the room they need; one that there is no room for goes through the slots.
std::vector<Streamed> pick_streamed(Batch& bt, const std::vector<ScalarPlan>& plan, Growths* growths) {
  std::vector<Streamed> some;
  double gain = 0.0;
  for (size_t i = 0; i < bt.size(); ++i) {
    pskv_table* t = bt[i].t;
    const uint64_t n = bt[i].r.n;
    if (!plan[i].may_stream || !n || t->streams == pskv_table::Streams::kNever) continue;
    Streamed s{&bt[i], {}, false, {}};
    for (const Growth<pskv_table, Slot>& g : growths->list)
      if (g.t == t && t->cap / g.cap <= (uint64_t)kRegrowMaxFactor) s.g = g, s.grows = true;
    s.shape = stream_shape(n, t->cap);
    if (!s.shape.bins) continue;
    const double its = t->streams == pskv_table::Streams::kWhereItFits
                           ? kStreamLaunches
                           : stream_gain(n, t->cap, t->share_known ? t->new_share : kFreshGuess, s.grows);
    if (its <= 0.0) continue;
    gain += its;
    some.push_back(s);
  }
  if (gain < kStreamLaunches) return {};
  std::vector<Streamed> todo;
  for (const Streamed& s : some) {
    if (grow(s.it->t, &s.it->t->ws, stream_room(s)) != PSKV_OK) {
      clear_error();
      continue;
    }
    todo.push_back(s);
    auto& list = growths->list;
    if (s.grows)
      list.erase(std::find_if(list.begin(), list.end(), [&](const Growth<pskv_table, Slot>& g) { return g.t == s.it->t; }));
  }
  return todo;
}

int run_scalar(Batch& bt, bool push, bool pull) {
  Growths growths;
  uint64_t n_largest = 0;
  bool any_cache = false, behind = false, packs = false, packed = false;
  std::vector<ScalarPlan> plan(bt.size());
  for (size_t i = 0; i < bt.size(); ++i) {
    Item& it = bt[i];
    pskv_table* t = it.t;
    Request& r = it.r;
    r.out_nvals = pull ? r.n : 0;
    it.d = TableReq{};
    if (r.n == 0) continue;
    // (a growth writes the cache back and drops it; a recorded repeat creates no key)
    int rc = r.replay == kReplayCapture ? PSKV_OK : reserve(t, r.n, 0, 0, &it.pub, &growths);
    if (rc) return rc;
    plan[i].kind_before = t->sc_last_kind;
    if (r.replay) {
      // a request that is being recorded fills the key cache, or is compared with it, whatever its size
      if (t->cap >= (1ull << 32))
        return set_error(PSKV_EINVAL, "a table of 2^32 slots keeps no key cache: its requests cannot be recorded");
      const bool fits = t->cache_valid && t->cache_n == r.n;
      if (r.replay == kReplayCapture && !fits)
        return set_error(PSKV_ESTALE, "the key cache does not hold the request that is being recorded");
      plan[i].use = fits ? kScTry : kScRecord;
      t->sc_last_n = r.n;
      t->sc_last_kind = r.push ? 0 : 1;
    } else {
      plan[i].use = scalar_cache_use(t, r);
      // A push that streams through the slots leaves no record. It gives way to one where pulls follow the pushes, and where the
      // newest push that streamed named the keys of the one before it (as far as the host has been told).
      const bool told_same = *static_cast<volatile unsigned long long*>(t->outcome + 1) != 0ull;
      plan[i].may_stream = push && !pull && !r.pinned &&
                      (plan[i].use == kScPlain || (plan[i].use == kScRecord && !pulls_follow(t) && !told_same));
    }
  }
  std::vector<Streamed> streamed = push && !pull ? pick_streamed(bt, plan, &growths) : std::vector<Streamed>();
  for (const Streamed& s : streamed) plan[s.it - bt.data()].streams = true;
  // (should the request end before they have: their arrays move with the others)
  struct GiveBack {
    std::vector<Streamed>& some;
    Growths& growths;
    ~GiveBack() {
      for (const Streamed& s : some)
        if (s.grows) growths.list.push_back(s.g);
    }
  } give_back_growths{streamed, growths};
  for (size_t i = 0; i < bt.size(); ++i) {
    Item& it = bt[i];
    pskv_table* t = it.t;
    Request& r = it.r;
    if (r.n == 0) continue;
    int rc = PSKV_OK;
    if (plan[i].streams) plan[i].use = kScPlain;
    // (17 B per key that a push that streamed has needed, and that nothing else of a SCALAR table does: a table that has been filled
    // may be pulled from for long)
    if (!plan[i].streams && t->ws.ptr && !t->capturing && (rc = drop(t, &t->ws))) return rc;
    if (plan[i].use != kScTry) {
      // the request goes through the slots, so they must be up to date; a push then makes the
      // cached values stale, a recording replaces them
      rc = flush_scalar_cache(t);
      if (rc) return rc;
      if (push || plan[i].use == kScRecord) t->cache_valid = false;
    }
    if (plan[i].streams) continue;
    TableReq& d = it.d;
    if (plan[i].use == kScRecord) {
      // Room for this request in the cache (it has been written back above; kScTry needs nothing:
      // the buffers have the cached request's size). Only a request that is going to be recorded
      // pays for it: a one-off pull of 16M keys would otherwise allocate 256 MB it never uses, and
      // wait for the stream to do so.
      rc = grow(t, &t->cache_keys, !r.replay && r.n >= t->pack_min_keys ? PackedKeys::bytes(r.n) : r.n * sizeof(uint64_t));
      if (rc) return rc;
      t->packing = false;
      rc = grow(t, &t->sc_vals, r.n * sizeof(float));
      if (rc) return rc;
      rc = grow(t, &t->sc_slots, r.n * sizeof(uint32_t));
      if (rc) return rc;
    }
    if (plan[i].use == kScPlain) {
      d.outcome = r.done;
      d.tag.epoch = r.done_seq;
    } else {
      it.tag = next_tag(t, r);
      t->sc_kind[it.tag.epoch % pskv_table::kScKinds] = r.push ? 0 : 1;
      d.tag = it.tag;
      d.cache_keys = static_cast<uint64_t*>(t->cache_keys.ptr);
      d.arena = static_cast<float*>(t->sc_vals.ptr);
      d.tile_key = static_cast<uint32_t*>(t->sc_slots.ptr);
      d.outcome = t->outcome;
      // A pull right behind a push, with the slots up to date (the push went through them and
      // recorded itself): the pull kernel compares key by key and needs no launch in front of it.
      // (not in a recording: keys that differ would go through the slots there)
      const bool per_key = plan[i].use == kScTry && !push && !t->sc_dirty && plan[i].kind_before == 0 && r.replay != kReplayCapture;
      d.cache_mode = per_key ? kCachePerKey : kCacheOn;
      any_cache = true;
      if (!per_key && it.tag.try_cache && !r.replay && r.n >= t->pack_min_keys && t->cache_keys.bytes >= PackedKeys::bytes(r.n)) {
        // (packed they are as soon as they have been asked for, further up the stream; the device looks, and says where it was not so)
        volatile unsigned long long* const told = t->outcome + 2;
        if (*told == kNotPacked) t->packing = false;
        if (t->packing) {
          if (*told != kNeverPacked) it.tag.try_cache = kTryPacked, packed = true;
        } else if (t->sc_track[r.push ? 0 : 1].hit) {
          it.tag.try_cache = kTryAndPack;
          t->packing = packs = true;
          *told = 0ull;
        }
        d.tag = it.tag;
      }
      // (a recorded repeat is served from the cache or not at all: nothing to write back)
      if (!per_key && it.tag.try_cache && t->sc_dirty && r.replay != kReplayCapture) {
        d.cache_mode = kCacheOnBehind;
        behind = true;
      }
    }
    d.slots = t->slots;
    d.mask = t->cap - 1;
    d.st = t->st;
    d.keys = r.keys;
    d.vals = r.vals;
    d.out = r.out;
    d.n = r.n;
    d.snap = it.pub.snap;  // the request's kernel leaves the counter record itself
    d.snap_seq = it.pub.seq;
    n_largest = std::max(n_largest, r.n);
  }
  if (!n_largest && streamed.empty()) return PSKV_OK;
  int rc = growths.move();
  if (rc) return rc;
  if (!streamed.empty()) {
    std::vector<Streamed> todo;
    todo.swap(streamed);
    rc = stream_push(bt, todo);
    if (rc || !n_largest) return rc;
  }
  // a recorded repeat, where the workgroups that compare it can wait for each other: one launch
  unsigned repeat_quads = 0;
  auto repeat_groups = [&](const Item& it) -> uint64_t {
    const uint64_t per = (uint64_t)kRepeatBlock * 4 * repeat_quads;
    return (it.d.n + per - 1) / per;
  };
  if (bt[0].r.replay == kReplayCapture) {
    for (unsigned quads : {kRepeatFew, kRepeatMany}) {
      uint64_t groups = 0;
      repeat_quads = quads;
      for (const Item& it : bt) groups += repeat_groups(it);
      if (groups <= kRepeatGroups) break;
      repeat_quads = 0;
    }
  }
  const bool one_launch = repeat_quads != 0;
  if (any_cache && !one_launch) {
    // (one kernel for all tables: the packed ones' compares the others' keys as they are, ReqTag::try_cache)
    const uint64_t per = packs || packed ? (uint64_t)kBlock * PackedKeys::kItems : (uint64_t)kBlock * kSameKeysItems;
    const KernelSet kernels = packs    ? PSKV_KSET_OF(k_same_packed, true)
                              : packed ? PSKV_KSET_OF(k_same_packed, false) : PSKV_KSET(k_same_keys);
    rc = launch_batch(bt, PSKV_KERNEL_SAME_KEYS, kernels, [&](const Item& it) {
      return ((it.d.cache_mode == kCacheOn || it.d.cache_mode == kCacheOnBehind) && it.tag.try_cache) ? (it.r.n + per - 1) / per : 0ull;
    });
    if (rc) return rc;
  }
  // The kernel strides over a table's keys, so a grid capped at kMaxGrid serves any request. A
  // request that is expected to repeat the cached keys gets a quarter of the workgroups: served
  // from the cache it moves four keys per lane (should it go through the slots after all, every
  // lane takes four turns).
  auto nblk = [&](const Item& it) -> uint64_t {
    if (!it.d.n) return 0;
    const bool four = (it.d.cache_mode == kCacheOn && it.tag.try_cache) || it.d.cache_mode == kCacheOnBehind ||
                      it.d.cache_mode == kCachePerKey;
    return grid_for(it.d.n, four ? kBlock * 4 : kBlock, kMaxGrid);
  };
  const bool pinned = bt[0].r.pinned;
  if (any_cache) {
    for (Item& it : bt) it.r.done = nullptr;  // (the word of such a launch says how the comparison went)
  }
  if (one_launch) {
    const bool few = repeat_quads == kRepeatFew;
    // (the environment variable, read when a request is recorded, is for tests of the wait that runs out)
    unsigned looks = kRepeatLooks;
    if (const char* e = std::getenv("PSKV_REPEAT_LOOKS")) looks = (unsigned)std::strtoul(e, nullptr, 10);
    for (Item& it : bt) it.d.cache_mode = looks;
    const KernelSet kernels =
        push && pull ? (few ? PSKV_KSET_OF(k_scalar_repeat, true, true, kRepeatFew) : PSKV_KSET_OF(k_scalar_repeat, true, true, kRepeatMany))
        : push       ? (few ? PSKV_KSET_OF(k_scalar_repeat, true, false, kRepeatFew) : PSKV_KSET_OF(k_scalar_repeat, true, false, kRepeatMany))
                     : (few ? PSKV_KSET_OF(k_scalar_repeat, false, true, kRepeatFew) : PSKV_KSET_OF(k_scalar_repeat, false, true, kRepeatMany));
    rc = launch_batch(bt, push ? PSKV_KERNEL_PUSH_SCALAR : PSKV_KERNEL_PULL_SCALAR, kernels, repeat_groups, kRepeatBlock);
  } else if (push && pull) {
    rc = behind    ? launch_batch(bt, PSKV_KERNEL_PUSH_SCALAR, PSKV_KSET_OF(k_scalar, true, true, true, false, true), nblk)
         : any_cache ? launch_batch(bt, PSKV_KERNEL_PUSH_SCALAR, PSKV_KSET_OF(k_scalar, true, true, true, false, false), nblk)
         : pinned  ? launch_batch(bt, PSKV_KERNEL_PUSH_SCALAR, PSKV_KSET_OF(k_scalar, true, true, false, true, false), nblk)
                   : launch_batch(bt, PSKV_KERNEL_PUSH_SCALAR, PSKV_KSET_OF(k_scalar, true, true, false, false, false), nblk);
  } else if (push) {
    rc = behind    ? launch_batch(bt, PSKV_KERNEL_PUSH_SCALAR, PSKV_KSET_OF(k_scalar, true, false, true, false, true), nblk)
         : any_cache ? launch_batch(bt, PSKV_KERNEL_PUSH_SCALAR, PSKV_KSET_OF(k_scalar, true, false, true, false, false), nblk)
         : pinned  ? launch_batch(bt, PSKV_KERNEL_PUSH_SCALAR, PSKV_KSET_OF(k_scalar, true, false, false, true, false), nblk)
                   : launch_batch(bt, PSKV_KERNEL_PUSH_SCALAR, PSKV_KSET_OF(k_scalar, true, false, false, false, false), nblk);
  } else {
    const int kind = bt[0].d.cache_mode == kCachePerKey ? PSKV_KERNEL_PULL_PER_KEY : PSKV_KERNEL_PULL_SCALAR;
    rc = behind    ? launch_batch(bt, kind, PSKV_KSET_OF(k_scalar, false, true, true, false, true), nblk)
         : any_cache ? launch_batch(bt, kind, PSKV_KSET_OF(k_scalar, false, true, true, false, false), nblk)
         : pinned  ? launch_batch(bt, PSKV_KERNEL_PULL_SCALAR, PSKV_KSET_OF(k_scalar, false, true, false, true, false), nblk)
                   : launch_batch(bt, PSKV_KERNEL_PULL_SCALAR, PSKV_KSET_OF(k_scalar, false, true, false, false, false), nblk);
  }
  if (rc) return rc;
  for (size_t i = 0; i < bt.size(); ++i) {
    if (plan[i].use == kScPlain || !bt[i].r.n) continue;
    pskv_table* t = bt[i].t;
    t->cache_valid = true;  // whichever way the device decides, the cache now stands for this request
    t->cache_n = bt[i].r.n;
    if (push && plan[i].use == kScTry) t->sc_dirty = true;  // served from the cache: the slots lag behind
  }
  return PSKV_OK;
}

// Requests at least this large (4 MiB) are streamed with non-temporal accesses: between two
// requests of a busy server they do not survive in the caches anyway.
constexpr uint64_t kStreamFloats = 1u << 20;

// FIXED: quads (see k_rows) that lie, whole (`started`: or in part), within the first `floats` floats of a
// request with rows of k floats.
uint64_t quads_within(uint64_t floats, uint64_t k, bool started) {
  const uint64_t in_row = floats % k;
  return floats / k * ((k + 3) / 4) + (started ? (in_row + 3) / 4 : in_row / 4);
}

// The row kernel over the request-side floats [first, first + floats) of the batch's only table (`first`
// is a multiple of a VARLEN workgroup's stretch): one piece of a request that is served as it arrives.
template <bool VARLEN>
int launch_rows_piece(Batch& bt, int op, uint64_t first, uint64_t floats) {
  Item& it = bt[0];
  const bool stream = it.d.total >= kStreamFloats;
  uint64_t blocks;
  if (VARLEN) {
    it.d.tile_base = (uint32_t)(first / kRowsVarPerBlock);
    blocks = (floats + kRowsVarPerBlock - 1) / kRowsVarPerBlock;
  } else {
    // a quad on the edge of two pieces goes with the second when it is read, with the first when written
    it.d.nvals = quads_within(first, it.d.k, op == kOpGather);
    it.d.ntiles = quads_within(first + floats, it.d.k, op == kOpGather);
    blocks = (it.d.ntiles - it.d.nvals + kQuadsFixed - 1) / kQuadsFixed;
  }
  auto nblk = [&](const Item&) { return blocks; };
  int rc;
  if (op == kOpAcc) {
    rc = stream ? launch_batch(bt, PSKV_KERNEL_ROWS_ACC, PSKV_KSET_OF(k_rows, kOpAcc, VARLEN, true, false, false), nblk)
                : launch_batch(bt, PSKV_KERNEL_ROWS_ACC, PSKV_KSET_OF(k_rows, kOpAcc, VARLEN, false, false, false), nblk);
  } else {
    rc = stream ? launch_batch(bt, PSKV_KERNEL_ROWS_GATHER, PSKV_KSET_OF(k_rows, kOpGather, VARLEN, true, false, false), nblk)
                : launch_batch(bt, PSKV_KERNEL_ROWS_GATHER, PSKV_KSET_OF(k_rows, kOpGather, VARLEN, false, false, false), nblk);
  }
  it.d.tile_base = 0;
  return rc;
}

// FIXED: whether all rows of a launch are wide ones, and the kernels for them. (A request that is served in pieces waits for the host
// link, whatever its kernel.)
bool all_wide(const Batch& bt) {
  return std::all_of(bt.begin(), bt.end(), [](const Item& it) { return !it.d.ntiles || it.d.k >= kWideRow; });
}
KernelSet wide_kernels(int op, bool stream) {
  if (op == kOpAcc) return stream ? PSKV_KSET_OF(k_rows_wide, kOpAcc, true) : PSKV_KSET_OF(k_rows_wide, kOpAcc, false);
  return stream ? PSKV_KSET_OF(k_rows_wide, kOpGather, true) : PSKV_KSET_OF(k_rows_wide, kOpGather, false);
}

// The row kernel over every table of the batch whose TableReq::total is not zero.
template <bool VARLEN>
int launch_rows(Batch& bt, int op) {
  uint64_t floats = 0;
  for (Item& it : bt) {
    floats += it.d.total;
    if (!VARLEN) {
      it.d.nvals = 0;
      it.d.ntiles = it.d.total ? it.d.n * ((it.d.k + 3) / 4) : 0;
    }
  }
  if (!floats) return PSKV_OK;
  if (bt.size() == 1 && op == kOpAcc && bt[0].r.pipe_in) {
    // the values are still in the caller's memory: every piece is accumulated as soon as it is here
    Item& it = bt[0];
    Stager* sg = Stager::get(it.t->device);
    if (!sg) return set_error(PSKV_ENOMEM, "no pinned memory to stage the request through");
    return sg->to_device(const_cast<float*>(it.r.vals), it.r.vals_host, it.d.total * sizeof(float),
                         it.t->stream, [&](size_t off, size_t len) {
                           return launch_rows_piece<VARLEN>(bt, kOpAcc, off / sizeof(float), len / sizeof(float));
                         });
  }
  if (bt.size() == 1 && op == kOpGather && bt[0].r.pipe_out) {
    bt[0].r.gather_deferred = true;  // launched piece by piece in step with the transfer to the host
    bt[0].r.gather_varlen = VARLEN;
    return PSKV_OK;
  }
  auto nblk = [&](const Item& it) {
    if (VARLEN) {
      uint64_t blocks = (it.d.total + kRowsVarPerBlock - 1) / kRowsVarPerBlock;
      if (op == kOpAcc && it.d.ragged) {
        const uint64_t rows = (uint64_t)kBlock >> by_row_shift(it.d.ragged);  // of a workgroup
        blocks = std::max(blocks, (it.d.n + rows - 1) / rows);
      }
      return blocks + (it.d.started ? 1 : 0);
    }
    return (it.d.ntiles + kQuadsFixed - 1) / kQuadsFixed;
  };
  const bool stream = floats >= kStreamFloats;
  const int kind = op == kOpAcc ? PSKV_KERNEL_ROWS_ACC : PSKV_KERNEL_ROWS_GATHER;
  if (!VARLEN && all_wide(bt)) return launch_batch(bt, kind, wide_kernels(op, stream), nblk);
  bool started = false;
  for (const Item& it : bt) started = started || (VARLEN && it.d.started);
  bool by_row = false;
  for (const Item& it : bt) by_row = by_row || (VARLEN && op == kOpAcc && it.d.ragged);
  auto pick = [&](auto op_, auto started_, auto by_row_) {
    constexpr int OP = decltype(op_)::value;
    constexpr bool STARTED = decltype(started_)::value, BY_ROW = decltype(by_row_)::value;
    return stream ? PSKV_KSET_OF(k_rows, OP, VARLEN, true, STARTED, BY_ROW) : PSKV_KSET_OF(k_rows, OP, VARLEN, false, STARTED, BY_ROW);
  };
  using Acc = std::integral_constant<int, kOpAcc>;
  using Gather = std::integral_constant<int, kOpGather>;
  using No = std::false_type;
  using Yes = std::integral_constant<bool, VARLEN>;
  const KernelSet kernels = op == kOpAcc ? (by_row ? (started ? pick(Acc(), Yes(), Yes()) : pick(Acc(), No(), Yes()))
                                                   : (started ? pick(Acc(), Yes(), No()) : pick(Acc(), No(), No())))
                                         : (started ? pick(Gather(), Yes(), No()) : pick(Gather(), No(), No()));
  return launch_batch(bt, kind, kernels, nblk);
}

// Starts a row-mode request on every table with keys: numbers it and (`compare`: a recorded one), where the
// key cache has the right shape, lets the device compare the request with the cached one. Call after every
// buffer the cache lives in has been grown for this request.
int begin_row_request(Batch& bt, bool compare) {
  for (Item& it : bt) {
    if (!it.r.n) continue;
    it.tag = next_tag(it.t, it.r, it.t->mode == PSKV_MODE_VARLEN);
    if (it.r.replay == kReplayCapture && !it.tag.try_cache)
      return set_error(PSKV_ESTALE, "the key cache does not hold the request that is being recorded%s",
                       it.t->mode == PSKV_MODE_VARLEN ? " (a PSKV_MODE_VARLEN pull leaves no key cache behind: record "
                                                        "it together with the push of its keys, or right behind one)"
                                                      : "");
    it.d.tag = it.tag;
    it.d.outcome = it.t->outcome;
  }
  if (!compare) return PSKV_OK;
  return launch_batch(bt, PSKV_KERNEL_SAME_KEYS, PSKV_KSET(k_same_keys), [](const Item& it) {
    return (it.r.n && it.tag.try_cache) ? (it.r.n + kBlock * kSameKeysItems - 1) / (kBlock * kSameKeysItems)
                                        : 0ull;
  });
}

// Whether a FIXED request is one launch (k_fixed_own): not where it arrives, or leaves, piece by piece or is being
// recorded, nor where a row is more than a workgroup takes. A push needs its workgroups on the GPU together. A pull of rows
// that do not end on a quad is better off with the lookup in front of it when it is large (500,000 rows of 33 floats,
// three tables in turn: 309 us per step against 298; 193,521 of 30: 120 against 126).
constexpr uint64_t kOwnRaggedFloats = 1u << 23;
bool fixed_in_one(const Batch& bt, bool push) {
  if (bt[0].r.replay || bt[0].r.pipe_in || bt[0].r.pipe_out) return false;
  uint64_t groups = 0, floats = 0;
  for (const Item& it : bt) {
    if (!it.r.n) continue;
    if ((it.d.k + 3) / 4 > kOwnQuads || it.r.n > ((uint64_t)1 << 40) / it.d.k) return false;
    groups += (it.r.n + own_keys(it.d.k) - 1) / own_keys(it.d.k);
    floats += it.d.k % 4 ? it.r.n * it.d.k : 0;
  }
  return push ? groups <= kOwnPushGroups : floats <= kOwnRaggedFloats;
}

// The same of longer rows (k_fixed_long, which says why the lines lie there).
bool fixed_long(const Batch& bt) {
  if (bt[0].r.replay || bt[0].r.pipe_in || bt[0].r.pipe_out) return false;
  uint64_t floats = 0;
  for (const Item& it : bt) {
    if (!it.r.n) continue;
    if ((it.d.k + 3) / 4 <= kOwnQuads || it.r.n > kLongKeys || it.d.k > kLongFloats) return false;
    floats += it.r.n * it.d.k;
  }
  return floats <= kLongFloats;
}

int run_fixed(Batch& bt, bool push, bool pull) {
  Growths growths;
  uint64_t n_largest = 0;
  for (Item& it : bt) {
    pskv_table* t = it.t;
    Request& r = it.r;
    const uint64_t k = t->row_len;
    r.out_nvals = pull ? r.n * k : 0;
    it.d = TableReq{};
    if (r.n == 0) continue;
    int rc = r.replay == kReplayCapture ? PSKV_OK : reserve(t, r.n, r.n, k, &it.pub, &growths);
    if (rc) return rc;
    rc = grow(t, &t->ws, Carver::need(r.n, sizeof(uint64_t)));
    if (rc) return rc;
    rc = grow(t, &t->cache_keys, r.n * sizeof(uint64_t));
    if (rc) return rc;
    if (!t->cache_valid) t->known_n = 0;
    Carver c(t->ws.ptr);
    TableReq& d = it.d;
    d.cached = (uint32_t)std::min<uint64_t>(t->known_n, 0xffffffffu);
    d.slots = t->slots;
    d.mask = t->cap - 1;
    d.st = t->st;
    d.keys = r.keys;
    d.n = r.n;
    d.arena = t->arena;
    d.ref = c.take<uint64_t>(r.n);
    d.cache_keys = static_cast<uint64_t*>(t->cache_keys.ptr);
    d.snap = it.pub.snap;
    d.snap_seq = it.pub.seq;
    d.k = k;
    n_largest = std::max(n_largest, r.n);
  }
  if (!n_largest) return PSKV_OK;
  int rc = growths.move();
  if (rc) return rc;
  rc = begin_row_request(bt, bt[0].r.replay == kReplayCapture);
  if (rc) return rc;
  const bool lengthy = fixed_long(bt), one = lengthy || fixed_in_one(bt, push);
  if (one) {
    uint64_t floats = 0;
    bool apart = true;  // (rows that share no line with their neighbours; the others go through the caches, see k_rows)
    for (Item& it : bt) {
      if (!it.r.n) continue;
      it.d.vals = it.r.vals;
      it.d.out = it.r.out;
      it.d.cache_mode = it.t->push_looks;
      floats += it.r.n * it.d.k;
      apart = apart && it.d.k >= 32 && (it.d.k % 4 == 0 || it.d.k >= 1024);
    }
    const bool stream = floats >= kStreamFloats && apart;
    const KernelSet kernels = lengthy ? (push && pull ? PSKV_KSET_OF(k_fixed_long, true, true)
                                         : push       ? PSKV_KSET_OF(k_fixed_long, true, false)
                                                      : PSKV_KSET_OF(k_fixed_long, false, true))
                              : push && pull ? PSKV_KSET_OF(k_fixed_own, true, true, false)
                              : push       ? stream ? PSKV_KSET_OF(k_fixed_own, true, false, true)
                                                    : PSKV_KSET_OF(k_fixed_own, true, false, false)
                              : stream     ? PSKV_KSET_OF(k_fixed_own, false, true, true)
                                           : PSKV_KSET_OF(k_fixed_own, false, true, false);
    rc = launch_batch(bt, push ? PSKV_KERNEL_ROWS_ACC : PSKV_KERNEL_ROWS_GATHER, kernels, [&](const Item& it) -> uint64_t {
      if (!it.r.n) return 0;
      return lengthy ? it.r.n * long_groups(it.d.k) : (it.r.n + own_keys(it.d.k) - 1) / own_keys(it.d.k);
    });
  } else if (bt[0].r.replay == kReplayCapture) {
    // a recorded repeat is compared as a whole and uses the references that are there: no lookup
  } else if (n_largest >= kLookupLargeKeys) {
    rc = launch_batch(bt, PSKV_KERNEL_LOOKUP, PSKV_KSET_OF(k_lookup_fixed, kLookupItemsLarge), [](const Item& it) {
      return it.r.n ? (uint64_t)grid_for(it.r.n, kBlock * kLookupItemsLarge, kMaxGrid) : 0ull;
    });
  } else {
    rc = launch_batch(bt, PSKV_KERNEL_LOOKUP, PSKV_KSET_OF(k_lookup_fixed, 1), [](const Item& it) {
      return it.r.n ? (uint64_t)grid_for(it.r.n, kBlock, kMaxGrid) : 0ull;
    });
  }
  if (rc) return rc;
  for (Item& it : bt) {
    if (!it.r.n) continue;
    // push and pull both create absent keys, so either leaves references for all n keys behind
    it.t->cache_valid = true;
    it.t->cache_n = it.r.n;
    it.t->cache_nvals = it.r.n * it.d.k;
    it.t->known_n = std::max(it.t->known_n, it.r.n);  // (what lies behind this request's last key holds still)
  }
  if (one) return PSKV_OK;
  if (push) {
    for (Item& it : bt) {
      if (!it.r.n) continue;
      it.d.req = const_cast<float*>(it.r.vals);
      it.d.total = it.r.n * it.d.k;
      it.d.ignore_new = 0;
    }
    rc = launch_rows<false>(bt, kOpAcc);
    if (rc) return rc;
  }
  if (pull) {
    for (Item& it : bt) {
      if (!it.r.n) continue;
      it.d.req = it.r.out;
      it.d.total = it.r.n * it.d.k;
      it.d.ignore_new = push ? 1u : 0u;
    }
    rc = launch_rows<false>(bt, kOpGather);
    if (rc) return rc;
  }
  return PSKV_OK;
}

// Room in the two tile tables for `floats` request-side floats.
int grow_tile_tables(pskv_table* t, uint64_t floats, uint64_t* ntiles_cap) {
  *ntiles_cap = (floats + kTileVar - 1) / kTileVar;
  int rc = grow(t, &t->tiles, (*ntiles_cap + 1) * sizeof(uint32_t));
  if (rc) return rc;
  return grow(t, &t->tiles_aff, (*ntiles_cap + 1) * sizeof(TileNote));
}

// Keys per thread of the creating lookup: 4 for long requests (fewer atomic adds on the arena counter), 1 for
// short ones so that even 100k keys spread over a few hundred workgroups.
constexpr uint64_t kVarLookupLargeKeys = 1u << 20;

// Workgroups for a kernel over `chunks` stretches of a request that returns at once when the request repeats
// the cached one: one per stretch, or a few hundred that stride over them where the newest comparison of
// requests of this kind has found the cached keys (a launch costs by the workgroup even then).
uint64_t may_return_at_once(const Item& it, bool push, uint64_t chunks, size_t tables) {
  const bool expected = it.tag.try_cache && it.t->sc_track[push ? 0 : 1].hit;
  return expected ? std::min<uint64_t>(chunks, std::max<uint64_t>(32, 512 / tables)) : chunks;
}

// Pass 2 of a pull's scan for every table with a response: the request-side offsets of the
// response and the tile table for Item::d.total floats of room (the row kernel fills the other
// table).
int make_tile_tables(Batch& bt, bool there = false) {
  for (Item& it : bt) {
    if (!it.d.total) continue;
    uint64_t ntiles_cap = 0;
    int rc = grow_tile_tables(it.t, it.d.total, &ntiles_cap);
    if (rc) return rc;
    it.d.tile_key = static_cast<uint32_t*>(it.t->tiles.ptr);
    it.d.tile_aff = static_cast<TileNote*>(it.t->tiles_aff.ptr);
    it.d.ntiles = ntiles_cap;
  }
  if (there || bt[0].r.replay == kReplayCapture) return PSKV_OK;  // (k_var_pull_start's; a recorded repeat's)
  return launch_batch(bt, -1, PSKV_KSET(k_var_offsets), [&](const Item& it) {
    return (it.r.n && it.d.total) ? may_return_at_once(it, false, it.nparts, bt.size()) : 0ull;
  });
}

// Whether a var-len request starts with one launch (start_rule.h): not where it is being recorded, or arrives piece by piece.
// The row kernel behind it cleans up, so every table has to have one (`floats`).
template <typename F>
bool start_together(const Batch& bt, bool push, F floats) {
  StartOf r;
  r.tables = (unsigned)bt.size();
  r.push = push;
  for (const Item& it : bt) {
    if (it.r.replay || it.r.pipe_in) return false;
    if (!it.r.n) continue;
    if (!floats(it)) return false;
    r.keys += it.r.n;
    r.floats += floats(it);
    r.parts += start_parts(it.r.n);
    r.compared = r.compared || it.tag.try_cache;
    r.shortcut = r.shortcut || (it.tag.try_cache && !const_cast<volatile unsigned long long*>(it.t->outcome)[1]);
  }
  return one_start(r);
}

// How the rows of a push are added should they be ragged (rows_by_row), where the table's pushes have been so far as the host has
// been told: so many lanes that two or three turns of them reach rows twice as long as the mean (lengths spread evenly from 1 on).
// Slice, push and pull, us: 2M rows of 1 to 20 floats in four tables 159 -> 146, 1M of 1 to 60 in one 163 -> 148. With a lane or more per
// quad of the mean and two turns always, the row kernel was no quicker than by tiles where the mean is a little above a power of two
// quads: 600,000 rows of 1 to 70 floats by tiles 56.6, so 60.2, with three turns of half the lanes 45.8; of 1 to 80 62.6, 63.6, 53.2; of 1
// to 180 129, 123, 107; 40,000 of 1 to 80 7.3, 8.6, 7.0.
// Not rows of a quad or two (300,000 of 1 to 10 in two tables 54 -> 56), of hundreds of floats, which fill wavefronts either way, nor
// requests that come in pieces, nor (the device sees to that) where a row takes sixteen times as long as the others. Nor requests that
// repeat the cached one, whose rows lie as the request has them and stay in the caches, of 1.5M to 3.5M floats, slice, push and pull by
// tiles and by the row: 55,000 rows of 1 to 100 34.4 and 36.0, 70,000 of 1 to 100 37.2 and 38.7, of 1 to 50 30.5 and 31.0; above and
// below it pays (90,000 of 1 to 100 43.4 and 42.7, 120,000 50.5 and 47.7; 30,000 of 1 to 80 27.3 and 26.9), and so it does for short rows
// (250,000 of 1 to 16 38.9 and 37.6). Whether a push repeats the cached one nobody knows that starts with one launch: 40,000 of 1
// to 100 take 30.7 and 32.3 repeated, 33.0 and 32.4 with other rows in every step.
constexpr uint64_t kByRowLeast = 8, kByRowMost = 128, kCachedLeast = 3ull << 19, kCachedMost = 7ull << 19, kCachedRow = 16;
// `floats`: of the whole request
uint64_t ragged_by_row(const Item& it, uint64_t floats) {
  const pskv_table* t = it.t;
  const Request& r = it.r;
  const uint64_t mean = r.nvals / r.n;
  const bool repeats = it.tag.try_cache && t->sc_track[0].hit;
  if (repeats && mean >= kCachedRow && floats >= kCachedLeast && floats < kCachedMost) return 0;
  if (!const_cast<volatile unsigned long long*>(t->outcome)[1] || r.pipe_in || mean < kByRowLeast || mean > kByRowMost) return 0;
  const uint64_t quads = (mean + 3) / 4;
  unsigned shift = 2;
  while ((3ull << shift) < quads * 2) ++shift;
  return by_row(shift, (1ull << shift) < quads, 16 * mean + 16);
}

// Launches per var-len request: a push takes three (compare + scan pass 1; scan pass 2 +
// find-or-create + counter record; rows), a pull three (compare + stored lengths + scan pass 1;
// scan pass 2 + tile table; rows), whatever the number of tables; a small one two (start_together).
int run_varlen(Batch& bt, bool push, bool pull) {
  uint64_t n_largest = 0;
  for (Item& it : bt) {
    it.r.out_nvals = 0;
    it.d = TableReq{};
    if (it.r.n > 0xfffffffeull) return set_error(PSKV_EINVAL, "too many keys in one request");
    n_largest = std::max(n_largest, it.r.n);
  }
  if (!n_largest) return PSKV_OK;
  // (keys per thread of the key-by-key kernels: by the keys of the whole launch, not of its largest table)
  uint64_t n_launch = 0, floats = 0;
  for (const Item& it : bt) n_launch += it.r.n, floats += it.r.nvals;
  const bool large = n_launch >= kVarLookupLargeKeys;
  const uint64_t chunk = kBlock * (large ? 4 : 1);  // keys per workgroup of the creating lookup
  const uint64_t pad_chunk = std::min(chunk, kStartPart);  // (and of k_var_push_start)
  const bool async_pull = pull && !push && !bt[0].r.need_total;
  for (Item& it : bt) {
    pskv_table* t = it.t;
    Request& r = it.r;
    if (!r.n) continue;
    it.nparts = scan_num_parts(r.n);
    const size_t need = Carver::need(r.n, 8) + Carver::need(r.n + 1, 8) + Carver::need(it.nparts, 8) +
                        Carver::need(r.n, 4);
    // Every buffer the key cache lives in is grown BEFORE the request is compared with the
    // cached one: a reallocation loses the cached contents and must rule the fast path out.
    int rc = grow(t, &t->ws, need);
    if (rc) return rc;
    rc = grow(t, &t->cache_keys, r.n * sizeof(uint64_t));
    if (rc) return rc;
    rc = grow(t, &t->cache_lens, r.n * sizeof(int32_t));
    if (rc) return rc;
    const uint64_t tiles_for = push ? r.nvals : (async_pull ? r.out_cap : 0);
    rc = grow_tile_tables(t, tiles_for, &it.tiles_cap);
    if (rc) return rc;
    Carver c(t->ws.ptr);
    TableReq& d = it.d;
    d.ref = c.take<uint64_t>(r.n);
    d.off = c.take<uint64_t>(r.n + 1);
    d.part = c.take<unsigned long long>(it.nparts);
    it.tmp_lens = c.take<int32_t>(r.n);
    d.cache_keys = static_cast<uint64_t*>(t->cache_keys.ptr);
    d.cache_lens = static_cast<int32_t*>(t->cache_lens.ptr);
    d.keys = r.keys;
    d.n = r.n;
    d.st = t->st;
  }

  if (push) {
    Growths growths;
    for (Item& it : bt) {
      pskv_table* t = it.t;
      Request& r = it.r;
      if (!r.n) continue;
      // every key may round its row up to a 16-byte unit, every workgroup may pad its rows' start
      int rc = r.replay == kReplayCapture
                   ? PSKV_OK
                   : reserve(t, r.n, r.nvals / 4 + r.n + kArenaPadUnits * ((r.n + pad_chunk - 1) / pad_chunk), 4, &it.pub, &growths);
      if (rc) return rc;
      if (t->cache_nvals != r.nvals) t->cache_valid = false;  // same lens would mean the same total
      it.tag = next_tag(t, r, true);
      if (r.replay == kReplayCapture && !it.tag.try_cache)
        return set_error(PSKV_ESTALE, "the key cache does not hold the request that is being recorded");
      TableReq& d = it.d;
      d.outcome = t->outcome;
      d.slots = t->slots;
      d.mask = t->cap - 1;
      d.arena = t->arena;
      d.lens = r.lens;
      d.nvals = r.nvals;
      d.tag = it.tag;
      d.snap = it.pub.snap;
      d.snap_seq = it.pub.seq;
      // pass 2 also fills the tile table of the request side (tile sizes are those of nvals; a
      // request whose lens do not add up to nvals is refused before it gets there)
      d.tile_key = r.nvals ? static_cast<uint32_t*>(t->tiles.ptr) : nullptr;
      d.tile_aff = static_cast<TileNote*>(t->tiles_aff.ptr);
      d.ntiles = it.tiles_cap;
      d.ragged = ragged_by_row(it, floats);
    }
    int rc = growths.move();
    if (rc) return rc;
    const bool start = start_together(bt, push, [](const Item& it) { return it.r.nvals; });
    if (start) {
      for (Item& it : bt) {
        it.tag.try_cache = it.d.tag.try_cache = 0;
        it.d.started = (uint32_t)start_parts(it.r.n);
        it.d.cache_mode = it.t->push_looks;
      }
      rc = launch_batch(bt, PSKV_KERNEL_LOOKUP, PSKV_KSET(k_var_push_start), [](const Item& it) { return start_parts(it.r.n); });
    } else {
      rc = launch_batch(bt, -1, PSKV_KSET(k_var_push_begin), [](const Item& it) { return it.r.n ? it.nparts : 0ull; });
    }
    if (rc) return rc;
    // (a recorded repeat uses the offsets, tile table and references that are there)
    if (!start && bt[0].r.replay != kReplayCapture)
      rc = launch_batch(bt, PSKV_KERNEL_LOOKUP, large ? PSKV_KSET_OF(k_var_push_lookup, 4) : PSKV_KSET_OF(k_var_push_lookup, 1), [&](const Item& it) {
        return it.r.n ? may_return_at_once(it, true, (it.r.n + chunk - 1) / chunk, bt.size()) : 0ull;
      });
    if (rc) return rc;
    for (Item& it : bt) {
      if (!it.r.n) continue;
      it.t->cache_valid = true;  // whichever way the device decided, the cache now is this request
      if (!start) it.d.snap = nullptr;  // (its lookup leaves the counter record)
      it.t->cache_n = it.r.n;
      it.t->cache_nvals = it.r.nvals;
      it.d.req = const_cast<float*>(it.r.vals);
      it.d.total = it.r.nvals;
      it.d.ignore_new = 0;
      it.d.total_on_device = 0;
    }
    rc = launch_rows<true>(bt, kOpAcc);
    if (rc) return rc;
  }
  if (pull) {
    int rc;
    if (push) {
      // a refused push must not be followed by its pull half
      rc = read_state_batch(bt, true);
      if (rc) return rc;
      for (Item& it : bt) {
        rc = report_device_errors(it.t);
        if (rc) return rc;
      }
    }
    for (Item& it : bt) {
      if (!it.r.n) continue;
      it.d.slots = it.t->slots;
      it.d.mask = it.t->cap - 1;
      it.d.arena = it.t->arena;
      it.d.out_lens = it.r.out_lens ? it.r.out_lens : it.tmp_lens;
      it.d.total = 0;
      it.d.snap = nullptr;
      it.d.started = 0;
    }
    // A pull with the keys of the cached push finds every key present with the cached length
    // and reuses its references; any other pull recomputes them and so ends the cache.
    rc = begin_row_request(bt, bt[0].r.replay == kReplayCapture);
    if (rc) return rc;
    for (Item& it : bt)
      if (it.r.n && !it.tag.try_cache) it.t->cache_valid = false;
    const bool start = async_pull && start_together(bt, false, [](const Item& it) { return it.r.out ? it.r.out_cap : 0; });
    if (start) {
      for (Item& it : bt) {
        if (!it.r.n) continue;
        it.d.tile_key = static_cast<uint32_t*>(it.t->tiles.ptr);
        it.d.ntiles = it.tiles_cap;
        it.d.started = (uint32_t)start_parts(it.r.n);
        it.d.cache_mode = it.t->push_looks;
      }
    }
    rc = launch_batch(bt, PSKV_KERNEL_LOOKUP, start ? PSKV_KSET(k_var_pull_start) : PSKV_KSET(k_var_pull_lookup),
                      [&](const Item& it) { return start ? start_parts(it.r.n) : it.r.n ? it.nparts : 0ull; });
    if (rc) return rc;
    if (async_pull) {
      // No host round trip: the grid covers the caller's buffer, the kernels take the real
      // size from the scan, and a response that does not fit is reported by the next sync.
      for (Item& it : bt) {
        if (!it.r.n || !it.r.out_cap) continue;
        if (!it.r.out) return set_error(PSKV_EINVAL, "null out");
        it.d.req = it.r.out;
        it.d.total = it.r.out_cap;
        it.d.total_on_device = 1;
        it.d.ignore_new = 1;
      }
      rc = make_tile_tables(bt, start);
      if (rc) return rc;
      return launch_rows<true>(bt, kOpGather);
    }
    rc = read_state_batch(bt, true);  // the response sizes are data dependent
    if (rc) return rc;
    int fit = PSKV_OK;
    for (Item& it : bt) {
      pskv_table* t = it.t;
      Request& r = it.r;
      if (!r.n) continue;
      if (t->st_host->same_epoch != it.tag.epoch) t->cache_valid = false;  // the pull recomputed the workspace
      const uint64_t total = t->st_host->scan_total;
      r.out_nvals = total;
      if (total > r.out_cap && !fit)
        fit = set_error(PSKV_ESIZE_MISMATCH, "response needs %llu floats, buffer holds %llu",
                        (unsigned long long)total, (unsigned long long)r.out_cap);
    }
    if (fit) return fit;
    for (Item& it : bt) {
      pskv_table* t = it.t;
      Request& r = it.r;
      const uint64_t total = r.n ? r.out_nvals : 0;
      if (!total) continue;
      if (r.lazy_out) {
        if (r.small_out && total <= r.small_out_floats) {
          r.out = reinterpret_cast<float*>(r.small_out);
        } else {
          rc = grow(t, &t->stage_out, total * sizeof(float));
          if (rc) return rc;
          r.out = static_cast<float*>(t->stage_out.ptr);
        }
      }
      if (!r.out) return set_error(PSKV_EINVAL, "null out");
      it.d.req = r.out;
      it.d.total = total;
      it.d.total_on_device = 0;
      it.d.ignore_new = 1;
    }
    rc = make_tile_tables(bt);
    if (rc) return rc;
    rc = launch_rows<true>(bt, kOpGather);
    if (rc) return rc;
  }
  return PSKV_OK;
}

int run_batch(Batch& bt, bool push, bool pull) {
  int rc;
  const bool capturing = bt[0].t->capturing;
  if (!capturing)
    for (Item& it : bt) ++it.t->gen;
  switch (bt[0].t->mode) {
    case PSKV_MODE_SCALAR: rc = run_scalar(bt, push, pull); break;
    case PSKV_MODE_FIXED: rc = run_fixed(bt, push, pull); break;
    default: rc = run_varlen(bt, push, pull); break;
  }
  // the GPU is busy with the request now: the moment to allocate ahead of a coming growth
  if (!rc && !capturing)
    for (Item& it : bt) prepare_growth(it.t);
  return rc;
}

// Host-side checks that mirror the CHECKs of the reference and the frozen rules of
// the row modes; nothing is enqueued when they fail.
int validate(pskv_table* t, bool push, bool pull, uint64_t n, uint64_t nvals, const int32_t* lens,
             uint64_t nlens, int memkind) {
  switch (t->mode) {
    case PSKV_MODE_SCALAR:
      // kv_app.h:447 CHECK_EQ(n, req_data.vals.size()); with pull set the reference
      // indexes vals[i] unchecked, which this library refuses when the sizes differ
      if (push && n != nvals)
        return set_error(PSKV_ESIZE_MISMATCH, "%llu keys but %llu values", (unsigned long long)n,
                         (unsigned long long)nvals);
      return PSKV_OK;
    case PSKV_MODE_FIXED:
      if (push) {
        if (n == 0) {
          if (nvals) return set_error(PSKV_ESIZE_MISMATCH, "values without keys");
        } else {
          const uint64_t k = nvals / n;  // kv_app.h:548-549
          if (k * n != nvals || k == 0)
            return set_error(PSKV_ESIZE_MISMATCH, "%llu values do not divide over %llu keys",
                             (unsigned long long)nvals, (unsigned long long)n);
          if (t->row_len == 0) t->row_len = k;
          if (k != t->row_len)
            return set_error(PSKV_ESIZE_MISMATCH, "row length %llu, table holds rows of %llu",
                             (unsigned long long)k, (unsigned long long)t->row_len);
        }
      }
      if (n && t->row_len == 0) return set_error(PSKV_EINVAL, "pull before the row length is known");
      return PSKV_OK;
    default:
      if (push) {
        if (nlens != n)  // kv_app.h:489,551
          return set_error(PSKV_ESIZE_MISMATCH, "%llu keys but %llu lens", (unsigned long long)n,
                           (unsigned long long)nlens);
        if (n && !lens) return set_error(PSKV_EINVAL, "lens missing");
        if (n == 0 && nvals) return set_error(PSKV_ESIZE_MISMATCH, "values without keys");
        if (memkind == PSKV_MEM_HOST) {
          uint64_t total = 0;
          for (uint64_t i = 0; i < n; ++i) {
            if (lens[i] < 0 || (uint32_t)lens[i] > PSKV_MAX_VARLEN_ROW)
              return set_error(PSKV_EINVAL, "lens[%llu] = %d out of range", (unsigned long long)i,
                               lens[i]);
            total += (uint64_t)lens[i];
          }
          if (total != nvals)
            return set_error(PSKV_ESIZE_MISMATCH, "lens add up to %llu, %llu values given",
                             (unsigned long long)total, (unsigned long long)nvals);
        }
      }
      return PSKV_OK;
  }
}

// Everything enqueued on the table has been waited for: small_in is free.
void small_idle(pskv_table* t) {
  t->small_part = 0;
  t->small_at = 0;
  t->small_in_flight = false;
  for (bool& p : t->small_pending) p = false;
}

// Room for a small host-resident request of `bytes` bytes in small_in that no request in flight reads.
int small_room(pskv_table* t, size_t bytes, char** out) {
  if (bytes > kSmallPart) {  // all of it (such a request is waited for)
    if (t->small_in_flight) PSKV_HIP(hipStreamSynchronize(t->stream));
    small_idle(t);
  } else if (t->small_at + bytes > kSmallPart) {
    // the requests that lie in the part that is full now are queued
    PSKV_HIP(hipEventRecord(t->small_done[t->small_part], t->stream));
    t->small_pending[t->small_part] = true;
    t->small_part = (t->small_part + 1) % kSmallParts;
    t->small_at = 0;
    if (t->small_pending[t->small_part]) {
      PSKV_HIP(hipEventSynchronize(t->small_done[t->small_part]));
      t->small_pending[t->small_part] = false;
    }
  }
  *out = t->small_in + (size_t)t->small_part * kSmallPart + t->small_at;
  t->small_at = std::min(t->small_at + bytes, kSmallPart);
  t->small_in_flight = true;
  return PSKV_OK;
}

int request(pskv_table* t, bool push, bool pull, const uint64_t* keys, size_t n, const float* vals,
            size_t nvals, const int32_t* lens, size_t nlens, float* out, size_t out_cap,
            int32_t* out_lens, size_t* out_nvals, int memkind) {
  clear_error();
  if (!t) return set_error(PSKV_EINVAL, "null table");
  if (memkind != PSKV_MEM_HOST && memkind != PSKV_MEM_DEVICE)
    return set_error(PSKV_EINVAL, "bad memkind %d", memkind);
  if (n && !keys) return set_error(PSKV_EINVAL, "null keys");
  if (push && nvals && !vals) return set_error(PSKV_EINVAL, "null vals");
  if (out_nvals) *out_nvals = 0;
  DeviceGuard guard(t->device);
  if (!guard.ok()) return set_error(PSKV_EHIP, "cannot select device %d", t->device);
  int rc = validate(t, push, pull, n, nvals, lens, nlens, memkind);
  if (rc) return rc;
  const bool host = memkind == PSKV_MEM_HOST;
  const bool varlen = t->mode == PSKV_MODE_VARLEN;
  bool small = false;        // host-resident request served from the pinned buffers
  bool early = false;        // a small push that returns once its kernel is queued
  size_t small_out_at = 0;   // bytes of small_out already given away

  // SCALAR and FIXED know the response size up front. A response that does not fit is
  // still computed (into scratch) so that the store ends up as the reference's would:
  // a pull creates absent keys (kv_app.h:457).
  uint64_t fixed_out = 0;
  if (pull && !varlen) fixed_out = t->mode == PSKV_MODE_SCALAR ? n : n * t->row_len;
  const bool too_small = pull && !varlen && fixed_out > out_cap;
  if (pull && !varlen && fixed_out && !too_small && !out) return set_error(PSKV_EINVAL, "null out");

  Request r{};
  r.push = push;
  r.pull = pull;
  r.n = n;
  r.nvals = push ? nvals : 0;
  r.out_cap = out_cap;
  r.need_total = host || out_nvals != nullptr || push;
  if (!host) {
    r.keys = keys;
    r.vals = vals;
    r.lens = lens;
    r.out = out;
    r.out_lens = out_lens;
  } else {
    const bool want_lens = push && varlen;
    const bool want_out_lens = pull && varlen;
    const size_t in_need =
        Carver::need(n, 8) + Carver::need(r.nvals, 4) + Carver::need(want_lens ? n : 0, 4);
    const size_t out_lens_need = Carver::need(want_out_lens ? n : 0, 4);
    small = in_need <= kSmallBytes && out_lens_need <= kSmallBytes;
    char* base = nullptr;
    early = small && t->mode == PSKV_MODE_SCALAR && !pull && in_need <= kSmallPart;
    if (small) {
      rc = small_room(t, in_need, &base);
      if (rc) return rc;
    }
    if (!small) {
      rc = grow(t, &t->stage, in_need + out_lens_need);
      if (rc) return rc;
      base = static_cast<char*>(t->stage.ptr);
    }
    Carver c(base);
    uint64_t* dkeys = c.take<uint64_t>(n);
    float* dvals = c.take<float>(r.nvals);
    int32_t* dlens = c.take<int32_t>(want_lens ? n : 0);
    int32_t* dout_lens = nullptr;
    if (small) {
      if (n) std::memcpy(dkeys, keys, n * 8);
      if (r.nvals) std::memcpy(dvals, vals, r.nvals * 4);
      if (want_lens && n) std::memcpy(dlens, lens, n * 4);
      small_out_at = out_lens_need;
      if (want_out_lens) dout_lens = reinterpret_cast<int32_t*>(t->small_out);
    } else {
      dout_lens = c.take<int32_t>(want_out_lens ? n : 0);
      Stager* sg = Stager::get(t->device);
      auto copy_in = [&](void* dst, const void* src, size_t bytes) -> int {
        if (!bytes) return PSKV_OK;
        // (buffers of the pinned pool are within reach of the copy engines as they are)
        if (sg && bytes >= kPipeBytes && !host_pool_owns(src, bytes))
          return sg->to_device(dst, src, bytes, t->stream, nullptr);
        PSKV_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, t->stream));
        return PSKV_OK;
      };
      rc = copy_in(dkeys, keys, n * 8);
      if (rc) return rc;
      if (want_lens) {
        rc = copy_in(dlens, lens, n * 4);
        if (rc) return rc;
      }
      if (sg && t->mode != PSKV_MODE_SCALAR && r.nvals * 4 >= kPipeBytes && !host_pool_owns(vals, r.nvals * 4)) {
        // the values follow piece by piece while the lookup and the row kernel are already at work
        r.vals_host = vals;
        r.pipe_in = true;
      } else {
        rc = copy_in(dvals, vals, r.nvals * 4);
        if (rc) return rc;
      }
    }
    // a large response of a row mode into ordinary memory leaves piece by piece as well, each piece
    // gathered just before it travels
    const uint64_t out_room = varlen ? out_cap : fixed_out;
    r.pipe_out = pull && !too_small && t->mode != PSKV_MODE_SCALAR && out_room * 4 >= kPipeBytes &&
                 !host_pool_owns(out, out_room * 4) && Stager::get(t->device) != nullptr;
    r.keys = dkeys;
    r.vals = dvals;
    r.lens = dlens;
    r.out_lens = want_out_lens ? dout_lens : nullptr;
    r.pinned = small;
    r.lazy_out = pull && varlen;
    if (small && r.lazy_out) {
      r.small_out = t->small_out + small_out_at;
      r.small_out_floats = (kSmallBytes - small_out_at) / sizeof(float);
    }
  }
  if (pull && !varlen && (host || too_small) && fixed_out) {
    if (small && !too_small && fixed_out * sizeof(float) <= kSmallBytes - small_out_at) {
      r.out = reinterpret_cast<float*>(t->small_out + small_out_at);
      if (t->mode == PSKV_MODE_SCALAR) {  // the host watches for the end of the request
        r.done = t->done;
        r.done_seq = ++t->done_seq;
      }
    } else {
      rc = grow(t, &t->stage_out, fixed_out * sizeof(float));
      if (rc) return rc;
      r.out = static_cast<float*>(t->stage_out.ptr);
    }
    r.out_cap = fixed_out;
  }

  Batch bt(1);
  bt[0].t = t;
  bt[0].r = r;
  rc = run_batch(bt, push, pull);
  r = bt[0].r;
  if (out_nvals) *out_nvals = r.out_nvals;
  // Kernels of this request may still be reading the pinned request buffer, which the next
  // host-resident request overwrites from the host: no early return without a wait.
  if (small && (rc || too_small)) {
    (void)hipStreamSynchronize(t->stream);
    small_idle(t);
  }
  if (rc) {
    t->cache_valid = false;
    return rc;
  }
  if (too_small)
    return set_error(PSKV_ESIZE_MISMATCH, "response needs %llu floats, buffer holds %llu",
                     (unsigned long long)fixed_out, (unsigned long long)out_cap);

  if (host) {
    const bool out_pinned = pull && r.out_nvals && r.out >= reinterpret_cast<float*>(t->small_out) &&
                            r.out < reinterpret_cast<float*>(t->small_out + kSmallBytes);
    const bool lens_pinned = r.out_lens == reinterpret_cast<int32_t*>(t->small_out);
    Stager* sg = Stager::get(t->device);
    bool copying = false;  // a copy command of its own is on the stream
    if (pull && r.out_nvals && !out_pinned) {
      if (r.gather_deferred || (sg && r.out_nvals * 4 >= kPipeBytes && !host_pool_owns(out, r.out_nvals * 4))) {
        // piece by piece: the gather (when it is still owed), the transfer of a piece, and the copy
        // into the caller's buffer overlap with those of the neighbouring pieces
        if (!sg) return set_error(PSKV_ENOMEM, "no pinned memory to stage the response through");
        std::function<int(size_t, size_t)> gather;
        if (r.gather_deferred) {
          gather = [&](size_t off, size_t len) {
            return r.gather_varlen ? launch_rows_piece<true>(bt, kOpGather, off / 4, len / 4)
                                   : launch_rows_piece<false>(bt, kOpGather, off / 4, len / 4);
          };
        }
        rc = sg->to_host(out, r.out, r.out_nvals * 4, t->stream, gather);
        if (rc) return rc;
      } else {
        PSKV_HIP(hipMemcpyAsync(out, r.out, r.out_nvals * 4, hipMemcpyDeviceToHost, t->stream));
        copying = true;
      }
    }
    if (pull && varlen && out_lens && n && !lens_pinned) {
      PSKV_HIP(hipMemcpyAsync(out_lens, r.out_lens, n * 4, hipMemcpyDeviceToHost, t->stream));
      copying = true;
    }
    if (early) {
      // no device-detected errors in this mode and nothing to hand back: the caller's buffers have
      // been copied, the kernel is queued, later requests follow it on the stream
      return PSKV_OK;
    }
    if (t->mode == PSKV_MODE_SCALAR) {
      // no device-detected errors in this mode: the end of the request is all that is left to wait for
      if (!r.done || !seen_in_time(r.done, r.done_seq)) PSKV_HIP(hipStreamSynchronize(t->stream));
    } else {
      // (also waits for the copies above, where there were any; what the staging ring has carried is here)
      rc = read_state(t, !copying);
      if (rc) return rc;
      rc = report_device_errors(t);
      if (rc) {
        t->cache_valid = false;
        return rc;
      }
    }
    small_idle(t);
    if (out_pinned) std::memcpy(out, r.out, r.out_nvals * 4);
    if (pull && varlen && out_lens && n && lens_pinned) std::memcpy(out_lens, r.out_lens, n * 4);
  }
  return PSKV_OK;
}

// Tables that one launch can serve together: one device, one mode, one stream.
int check_group(pskv_table* const* tables, size_t S) {
  if (!tables && S) return set_error(PSKV_EINVAL, "null table list");
  for (size_t s = 0; s < S; ++s) {
    if (!tables[s]) return set_error(PSKV_EINVAL, "tables[%zu] is null", s);
    if (tables[s]->device != tables[0]->device || tables[s]->mode != tables[0]->mode)
      return set_error(PSKV_EINVAL, "tables[%zu] differs from tables[0] in device or mode", s);
    if (tables[s]->stream != tables[0]->stream)
      return set_error(PSKV_EINVAL,
                       "tables[%zu] runs on a stream of its own: create the tables of a group with "
                       "pskv_opts.stream = pskv_table_stream(first table)", s);
    for (size_t q = 0; q < s; ++q)
      if (tables[q] == tables[s]) return set_error(PSKV_EINVAL, "tables[%zu] is tables[%zu]", s, q);
  }
  return PSKV_OK;
}

// pskv_push_multi / pskv_pull_multi: slice s of the request, keys [pos[s], pos[s+1]), goes to
// tables[s]; slices without keys are skipped as KVWorker::Send skips them (kv_app.h:590-595).
int request_multi(pskv_table* const* tables, size_t S, bool push, bool pull, const uint64_t* keys,
                  const uint64_t* pos, const float* vals, const uint64_t* val_pos, const int32_t* lens,
                  float* out, const uint64_t* out_pos, int32_t* out_lens, uint64_t* out_nvals,
                  int memkind, int replay = 0) {
  clear_error();
  if (memkind != PSKV_MEM_DEVICE)
    return set_error(PSKV_EINVAL, "the multi-table entry points take device-resident buffers "
                                  "(PSKV_MEM_DEVICE); host-resident requests go table by table");
  if (out_nvals)
    for (size_t s = 0; s < S; ++s) out_nvals[s] = 0;
  if (S == 0) return PSKV_OK;
  int rc = check_group(tables, S);
  if (rc) return rc;
  if (!pos) return set_error(PSKV_EINVAL, "null pos");
  const int mode = tables[0]->mode;
  const bool varlen = mode == PSKV_MODE_VARLEN;
  if (pos[S] != pos[0] && !keys) return set_error(PSKV_EINVAL, "null keys");
  if (push && !val_pos) return set_error(PSKV_EINVAL, "null val_pos");
  if (pull && varlen && !out_pos) return set_error(PSKV_EINVAL, "a var-len pull needs out_pos");
  // everything the host can check, for every slice, before anything is enqueued
  std::vector<Request> reqs(S);
  for (size_t s = 0; s < S; ++s) {
    if (pos[s + 1] < pos[s]) return set_error(PSKV_EINVAL, "pos[%zu] > pos[%zu]", s, s + 1);
    Request& r = reqs[s];
    r = Request{};
    r.push = push;
    r.pull = pull;
    r.replay = replay;
    r.n = pos[s + 1] - pos[s];
    r.keys = keys + pos[s];
    if (push) {
      if (val_pos[s + 1] < val_pos[s]) return set_error(PSKV_EINVAL, "val_pos[%zu] > val_pos[%zu]", s, s + 1);
      r.nvals = val_pos[s + 1] - val_pos[s];
      r.vals = vals + val_pos[s];
      r.lens = (varlen && lens) ? lens + pos[s] : nullptr;
      if (r.nvals && !vals) return set_error(PSKV_EINVAL, "null vals");
    }
    if (!r.n) {
      if (r.nvals) return set_error(PSKV_ESIZE_MISMATCH, "slice %zu has values but no keys", s);
      continue;
    }
    rc = validate(tables[s], push, pull, r.n, r.nvals, r.lens, varlen && push ? r.n : 0, memkind);
    if (rc) return rc;
    if (pull) {
      const uint64_t k = mode == PSKV_MODE_SCALAR ? 1 : tables[s]->row_len;
      const uint64_t at = out_pos ? out_pos[s] : pos[s] * k;
      if (out_pos && out_pos[s + 1] < out_pos[s])
        return set_error(PSKV_EINVAL, "out_pos[%zu] > out_pos[%zu]", s, s + 1);
      r.out_cap = out_pos ? out_pos[s + 1] - out_pos[s] : r.n * k;
      r.out = out ? out + at : nullptr;
      if (!varlen) {
        if (r.out_cap < r.n * k)
          return set_error(PSKV_ESIZE_MISMATCH, "slice %zu answers %llu floats, out_pos leaves room for %llu",
                           s, (unsigned long long)(r.n * k), (unsigned long long)r.out_cap);
        if (!r.out) return set_error(PSKV_EINVAL, "null out");
      } else {
        r.out_lens = out_lens ? out_lens + pos[s] : nullptr;
        r.need_total = out_nvals != nullptr;
      }
    }
  }
  DeviceGuard guard(tables[0]->device);
  if (!guard.ok()) return set_error(PSKV_EHIP, "cannot select device %d", tables[0]->device);
  Batch bt;
  std::vector<size_t> who;
  auto flush = [&]() -> int {
    if (bt.empty()) return PSKV_OK;
    const int r = run_batch(bt, push, pull);
    for (size_t i = 0; i < bt.size(); ++i) {
      if (out_nvals) out_nvals[who[i]] = bt[i].r.out_nvals;
      if (r) bt[i].t->cache_valid = false;
    }
    bt.clear();
    who.clear();
    return r;
  };
  for (size_t s = 0; s < S; ++s) {
    if (!reqs[s].n) continue;
    Item it;
    it.t = tables[s];
    it.r = reqs[s];
    bt.push_back(it);
    who.push_back(s);
    if (bt.size() == (size_t)kMaxBatch) {
      rc = flush();
      if (rc) return rc;
    }
  }
  return flush();
}

}  // namespace

extern "C" {

int pskv_table_create(pskv_table** out, const pskv_opts* opts) {
  clear_error();
  if (!out || !opts) return set_error(PSKV_EINVAL, "null argument");
  *out = nullptr;
  if (opts->mode < PSKV_MODE_SCALAR || opts->mode > PSKV_MODE_VARLEN)
    return set_error(PSKV_EINVAL, "bad mode %d", opts->mode);
  if (opts->max_load < 0.f || opts->max_load > 0.9f)
    return set_error(PSKV_EINVAL, "max_load must lie in (0, 0.9]");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0)
    return set_error(PSKV_EHIP, "no HIP device available");
  if (opts->device < 0 || opts->device >= ndev)
    return set_error(PSKV_EINVAL, "device %d out of range (%d present)", opts->device, ndev);
  DeviceGuard guard(opts->device);
  if (!guard.ok()) return set_error(PSKV_EHIP, "cannot select device %d", opts->device);

  pskv_table* t = new (std::nothrow) pskv_table();
  if (!t) return set_error(PSKV_ENOMEM, "out of host memory");
  t->device = opts->device;
  t->mode = opts->mode;
  t->max_load = opts->max_load > 0.f ? opts->max_load : 0.5f;
  t->row_len = opts->mode == PSKV_MODE_FIXED ? opts->row_len : 0;
  device_tables(t->device, 1, give_back);
  // (the environment variable is for tests of workgroups that do not see the verdict)
  t->push_looks = kOwnLooks;
  if (const char* e = std::getenv("PSKV_PUSH_LOOKS")) t->push_looks = (unsigned)std::strtoul(e, nullptr, 10);
  if (const char* e = std::getenv("PSKV_STREAM"))
    t->streams = std::atoi(e) ? pskv_table::Streams::kWhereItFits : pskv_table::Streams::kNever;
  t->sc_min_keys = kScalarCacheMinKeys;
  if (const char* e = std::getenv("PSKV_SCALAR_CACHE_MIN_KEYS")) t->sc_min_keys = std::strtoull(e, nullptr, 10);
  t->pack_min_keys = kPackKeys;
  if (const char* e = std::getenv("PSKV_PACK_MIN_KEYS")) t->pack_min_keys = std::strtoull(e, nullptr, 10);
  auto fail = [&](int rc) {
    pskv_table_destroy(t);
    return rc;
  };
  t->shell = shell_take(t->device);
  if (!t->shell) return fail(set_error(PSKV_ENOMEM, "cannot allocate table state"));
  if (opts->stream) {
    t->stream = static_cast<hipStream_t>(opts->stream);
  } else {
    t->own_stream = stream_take(t->device);
    if (!t->own_stream) return fail(set_error(PSKV_EHIP, "hipStreamCreateWithFlags failed"));
    t->stream = t->own_stream;
  }
  t->st = t->shell->st;
  t->st_host = reinterpret_cast<StateView*>(t->shell->pinned);
  t->snap = reinterpret_cast<Snapshot*>(t->shell->pinned + 256);
  t->outcome = reinterpret_cast<unsigned long long*>(t->shell->pinned + 512);
  t->done = reinterpret_cast<unsigned long long*>(t->shell->pinned + 768);
  *t->done = 0ull;
  t->small_in = t->shell->pinned + 1024;
  t->small_out = t->small_in + kSmallBytes;
  for (int q = 0; q < kSmallParts; ++q) t->small_done[q] = t->shell->done[q];
  std::memset(t->st_host, 0, sizeof(StateView));
  std::memset(t->snap, 0xFF, sizeof(Snapshot));  // names no request
  t->outcome[0] = t->outcome[1] = t->outcome[2] = 0ull;
  const uint64_t keys = opts->initial_capacity ? opts->initial_capacity : kDefaultCapacity;
  t->cap = std::max(kMinSlots, next_pow2((uint64_t)((double)keys / t->max_load) + 1));
  int rc = alloc_slots(t->cap, &t->slots, t->stream);
  if (rc) return fail(rc);
  k_init_table<<<dim3(grid_for(t->cap, kBlock, 1u << 16)), dim3(kBlock), 0, t->stream>>>(t->st, t->slots, t->cap);
  if (hipGetLastError() != hipSuccess) return fail(set_error(PSKV_EHIP, "table initialisation failed"));
  if (t->mode != PSKV_MODE_SCALAR && opts->arena_floats) {
    t->arena_cap = (opts->arena_floats + 1023) & ~(uint64_t)1023;
    if (array_alloc(reinterpret_cast<void**>(&t->arena), t->arena_cap * sizeof(float) + kArenaEnd, t->stream) != PSKV_OK)
      return fail(set_error(PSKV_ENOMEM, "cannot allocate %llu floats of row storage",
                            (unsigned long long)t->arena_cap));
  }
  *out = t;
  return PSKV_OK;
}

int pskv_table_destroy(pskv_table* t) {
  if (!t) return PSKV_OK;
  DeviceGuard guard(t->device);
  if (std::getenv("PSKV_STATS"))
    fprintf(stderr, "[pskv] table %p mode %d: %llu requests, %llu slots at the end, %llu growths (%llu without asking "
            "the device, %llu into an array allocated ahead), %llu waits for exact counters, %llu for the newest record (%.0f us), %llu counter records; host time "
            "allocating %.0f us (%.0f us on the allocating thread), releasing %.0f us\n",
            (void*)t, t->mode, (unsigned long long)t->stats.requests, (unsigned long long)t->cap,
            (unsigned long long)t->stats.growths, (unsigned long long)t->stats.growths_unasked,
            (unsigned long long)t->stats.spare_used, (unsigned long long)t->stats.waits,
            (unsigned long long)t->stats.catch_ups, t->stats.catch_up_us, (unsigned long long)t->stats.records,
            t->stats.alloc_us, t->stats.ahead_us, t->stats.release_us);
  collect_spare(t, true);  // (the stream may have been made to wait for what used that array before)
  const unsigned long long mark = array_mark(t->device);
  const bool idle = !t->stream || hipStreamSynchronize(t->stream) == hipSuccess;
  for (int k = 0; k < PSKV_KERNEL_COUNT; ++k)
    for (const EventPair& ev : t->pending[k]) t->free_events.push_back(ev);
  for (const EventPair& ev : t->free_events) {
    (void)hipEventDestroy(ev.a);
    (void)hipEventDestroy(ev.b);
  }
  // this table's work is done: its arrays are free to go to any other table at once, as are those that were given up
  // before the wait. (Others may use the stream: what they have given up since waits for its own event.)
  if (t->stream && idle) array_settle(t->device, t->stream, mark);
  for (void* ptr : {static_cast<void*>(t->slots), static_cast<void*>(t->arena), static_cast<void*>(t->spare)})
    (void)array_release(ptr, t->stream, idle);
  for (const GrowBuf* b : {&t->ws, &t->tiles, &t->tiles_aff, &t->stage, &t->stage_out, &t->cache_keys, &t->cache_lens,
                           &t->sc_vals, &t->sc_slots})
    (void)array_release(b->ptr, t->stream, idle);
  shell_give(t->device, t->shell);
  if (t->own_stream) stream_give(t->device, t->own_stream);
  device_tables(t->device, -1, give_back);
  delete t;
  return PSKV_OK;
}

int pskv_push(pskv_table* t, const uint64_t* keys, size_t n, const float* vals, size_t nvals,
              const int32_t* lens, size_t nlens, int memkind) {
  return request(t, true, false, keys, n, vals, nvals, lens, nlens, nullptr, 0, nullptr, nullptr,
                 memkind);
}

int pskv_pull(pskv_table* t, const uint64_t* keys, size_t n, float* out, size_t out_cap,
              int32_t* out_lens, size_t* out_nvals, int memkind) {
  return request(t, false, true, keys, n, nullptr, 0, nullptr, 0, out, out_cap, out_lens,
                 out_nvals, memkind);
}

int pskv_pushpull(pskv_table* t, const uint64_t* keys, size_t n, const float* vals, size_t nvals,
                  const int32_t* lens, size_t nlens, float* out, size_t out_cap,
                  int32_t* out_lens, size_t* out_nvals, int memkind) {
  return request(t, true, true, keys, n, vals, nvals, lens, nlens, out, out_cap, out_lens,
                 out_nvals, memkind);
}

void* pskv_table_stream(pskv_table* t) { return t ? static_cast<void*>(t->stream) : nullptr; }

int pskv_push_multi(pskv_table* const* tables, size_t S, const uint64_t* keys, const uint64_t* pos,
                    const float* vals, const uint64_t* val_pos, const int32_t* lens, int memkind) {
  return request_multi(tables, S, true, false, keys, pos, vals, val_pos, lens, nullptr, nullptr, nullptr,
                       nullptr, memkind);
}

int pskv_pushpull_multi(pskv_table* const* tables, size_t S, const uint64_t* keys, const uint64_t* pos,
                        const float* vals, const uint64_t* val_pos, const int32_t* lens, float* out,
                        const uint64_t* out_pos, int32_t* out_lens, uint64_t* out_nvals, int memkind) {
  return request_multi(tables, S, true, true, keys, pos, vals, val_pos, lens, out, out_pos, out_lens, out_nvals,
                       memkind);
}

int pskv_pull_multi(pskv_table* const* tables, size_t S, const uint64_t* keys, const uint64_t* pos,
                    float* out, const uint64_t* out_pos, int32_t* out_lens, uint64_t* out_nvals,
                    int memkind) {
  return request_multi(tables, S, false, true, keys, pos, nullptr, nullptr, nullptr, out, out_pos, out_lens,
                       out_nvals, memkind);
}

// Up to so many launches are made again one by one whatever the caller asked for: they take the calling thread
// 2.7 us each, a graph of one or two kernels 16 us.
constexpr size_t kGraphLaunches = 5;

struct pskv_replay {
  std::vector<pskv_table*> tables;
  std::vector<uint64_t> gen;  // pskv_table::gen of each when the recording was made
  std::vector<SavedLaunch> launches;  // made again one by one: PSKV_REPLAY_LAUNCHES, or few of them
  hipGraphExec_t exec = nullptr;
  hipStream_t stream = nullptr;
  int device = 0;
};

int pskv_replay_record(pskv_replay** out, pskv_table* const* tables, size_t S, int what, const uint64_t* keys,
                       const uint64_t* pos, const float* vals, const uint64_t* val_pos, const int32_t* lens,
                       float* out_vals, const uint64_t* out_pos, int32_t* out_lens) {
  clear_error();
  if (!out) return set_error(PSKV_EINVAL, "null argument");
  *out = nullptr;
  const bool push = (what & PSKV_REPLAY_PUSH) != 0, pull = (what & PSKV_REPLAY_PULL) != 0;
  if ((!push && !pull) || (what & ~(PSKV_REPLAY_PUSH | PSKV_REPLAY_PULL | PSKV_REPLAY_LAUNCHES)))
    return set_error(PSKV_EINVAL, "what = %d names neither a push nor a pull", what);
  if (S == 0) return set_error(PSKV_EINVAL, "no tables");
  int rc = check_group(tables, S);
  if (rc) return rc;
  if (!pos || pos[S] == pos[0]) return set_error(PSKV_EINVAL, "a request without keys cannot be recorded");
  auto both = [&](int replay) -> int {
    // SCALAR: a pull of the keys just pushed is the push's own read-back, so the two go as ONE request
    // with both halves (per key the push first, kv_app.h:451-459): one comparison and one pass
    if (push && pull && tables[0]->mode == PSKV_MODE_SCALAR)
      return request_multi(tables, S, true, true, keys, pos, vals, val_pos, lens, out_vals, out_pos, out_lens,
                           nullptr, PSKV_MEM_DEVICE, replay);
    int r = PSKV_OK;
    if (push)
      r = request_multi(tables, S, true, false, keys, pos, vals, val_pos, lens, nullptr, nullptr, nullptr,
                        nullptr, PSKV_MEM_DEVICE, replay);
    if (!r && pull)
      r = request_multi(tables, S, false, true, keys, pos, nullptr, nullptr, nullptr, out_vals, out_pos, out_lens,
                        nullptr, PSKV_MEM_DEVICE, replay);
    return r;
  };
  // The request itself, the ordinary way: tables grow, buffers get their sizes, the key cache is
  // filled. What the device finds wrong with it ends the recording.
  rc = both(kReplayPrime);
  if (rc) return rc;
  rc = pskv_sync_multi(tables, S);
  if (rc) return rc;
  DeviceGuard guard(tables[0]->device);
  if (!guard.ok()) return set_error(PSKV_EHIP, "cannot select device %d", tables[0]->device);
  // (an allocation that the library's own thread is making on this stream must not land in the graph)
  for (size_t s = 0; s < S; ++s) collect_spare(tables[s], true);
  hipStream_t stream = tables[0]->stream;
  // The launches of a repeat, recorded instead of run. Relaxed: other threads of the process may
  // be allocating or waiting meanwhile, which is none of this capture's business.
  PSKV_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeRelaxed));
  std::vector<SavedLaunch> saved;
  for (size_t s = 0; s < S; ++s) tables[s]->capturing = true;
  g_recording = &saved;
  rc = both(kReplayCapture);
  g_recording = nullptr;
  for (size_t s = 0; s < S; ++s) tables[s]->capturing = false;
  hipGraph_t graph = nullptr;
  const hipError_t e = hipStreamEndCapture(stream, &graph);
  if (rc || e != hipSuccess || !graph) {
    const std::string text = rc ? std::string(pskv_last_error()) : std::string();
    if (graph) (void)hipGraphDestroy(graph);
    (void)hipGetLastError();
    for (size_t s = 0; s < S; ++s) tables[s]->cache_valid = false;
    if (rc) return set_error(rc, "%s", text.c_str());
    return set_error(PSKV_EHIP, "the stream of the tables could not be captured: %s", hipGetErrorString(e));
  }
  pskv_replay* r = new (std::nothrow) pskv_replay();
  if (!r) {
    (void)hipGraphDestroy(graph);
    return set_error(PSKV_ENOMEM, "out of host memory");
  }
  const bool as_graph = (what & PSKV_REPLAY_LAUNCHES) == 0 && saved.size() > kGraphLaunches;
  const hipError_t ei = as_graph ? hipGraphInstantiate(&r->exec, graph, nullptr, nullptr, 0) : hipSuccess;
  (void)hipGraphDestroy(graph);
  if (ei != hipSuccess) {
    delete r;
    (void)hipGetLastError();
    return set_error(PSKV_EHIP, "hipGraphInstantiate: %s", hipGetErrorString(ei));
  }
  if (!as_graph) r->launches.swap(saved);
  r->stream = stream;
  r->device = tables[0]->device;
  r->tables.assign(tables, tables + S);
  for (size_t s = 0; s < S; ++s) r->gen.push_back(tables[s]->gen);
  *out = r;
  return PSKV_OK;
}

int pskv_replay_run(pskv_replay* r) {
  clear_error();
  if (!r || (!r->exec && r->launches.empty())) return set_error(PSKV_EINVAL, "null recording");
  for (size_t s = 0; s < r->tables.size(); ++s)
    if (r->tables[s]->gen != r->gen[s])
      return set_error(PSKV_ESTALE, "tables[%zu] has served other requests since the recording was made", s);
  DeviceGuard guard(r->device);
  if (!guard.ok()) return set_error(PSKV_EHIP, "cannot select device %d", r->device);
  if (r->exec) {
    PSKV_HIP(hipGraphLaunch(r->exec, r->stream));
    return PSKV_OK;
  }
  for (SavedLaunch& l : r->launches) {
    void* args[] = {&l.rb};
    PSKV_HIP(hipLaunchKernel(l.kernel, l.grid, l.block, args, 0, r->stream));
  }
  return PSKV_OK;
}

int pskv_replay_destroy(pskv_replay* r) {
  if (!r) return PSKV_OK;
  DeviceGuard guard(r->device);
  (void)hipStreamSynchronize(r->stream);
  if (r->exec) (void)hipGraphExecDestroy(r->exec);
  delete r;
  return PSKV_OK;
}

int pskv_sync_multi(pskv_table* const* tables, size_t S) {
  clear_error();
  if (S == 0) return PSKV_OK;
  int rc = check_group(tables, S);
  if (rc) return rc;
  DeviceGuard guard(tables[0]->device);
  int first = PSKV_OK;
  std::string first_text;
  for (size_t at = 0; at < S; at += kMaxBatch) {
    Batch bt(std::min<size_t>(S - at, kMaxBatch));
    for (size_t i = 0; i < bt.size(); ++i) bt[i].t = tables[at + i];
    rc = read_state_batch(bt, false);
    if (rc) return rc;
    for (Item& it : bt) {
      rc = report_device_errors(it.t);  // every table's error bits are cleared; the first is reported
      if (rc && !first) {
        first = rc;
        first_text = pskv_last_error();
      }
    }
  }
  if (first) return set_error(first, "%s", first_text.c_str());
  return PSKV_OK;
}

int pskv_sync(pskv_table* t) {
  clear_error();
  if (!t) return set_error(PSKV_EINVAL, "null table");
  DeviceGuard guard(t->device);
  int rc = read_state(t);
  if (rc) return rc;
  prepare_growth(t);  // (the counters are exact now)
  return report_device_errors(t);
}

// The keys and floats that a table holds, its state having just been read.
static int size_of(pskv_table* t, uint64_t* n_keys, uint64_t* n_vals) {
  const uint64_t nk = t->count;  // includes key 2^64-1 when present
  if (n_keys) *n_keys = nk;
  if (!n_vals) return PSKV_OK;
  if (t->mode == PSKV_MODE_SCALAR) {
    *n_vals = nk;
  } else if (t->mode == PSKV_MODE_FIXED) {
    *n_vals = nk * t->row_len;
  } else {
    unsigned long long* d_total = nullptr;
    PSKV_HIP(hipMalloc(reinterpret_cast<void**>(&d_total), sizeof(unsigned long long)));
    PSKV_HIP(hipMemsetAsync(d_total, 0, sizeof(unsigned long long), t->stream));
    k_sum_lens<<<dim3(grid_for(t->cap, kBlock, 4096)), dim3(kBlock), 0, t->stream>>>(
        t->slots, t->cap, t->st, d_total);
    unsigned long long total = 0;
    hipError_t e = hipMemcpyAsync(&total, d_total, sizeof(total), hipMemcpyDeviceToHost, t->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(t->stream);
    (void)hipFree(d_total);
    PSKV_HIP(e);
    *n_vals = total;
  }
  return PSKV_OK;
}

int pskv_size(pskv_table* t, uint64_t* n_keys, uint64_t* n_vals) {
  clear_error();
  if (!t) return set_error(PSKV_EINVAL, "null table");
  DeviceGuard guard(t->device);
  int rc = read_state(t, true);
  if (rc) return rc;
  return size_of(t, n_keys, n_vals);
}

int pskv_size_multi(pskv_table* const* tables, size_t S, uint64_t* n_keys, uint64_t* n_vals) {
  clear_error();
  if (S == 0) return PSKV_OK;
  int rc = check_group(tables, S);
  if (rc) return rc;
  DeviceGuard guard(tables[0]->device);
  for (size_t at = 0; at < S; at += kMaxBatch) {
    rc = read_states(tables + at, std::min<size_t>(S - at, kMaxBatch), true);
    if (rc) return rc;
  }
  for (size_t s = 0; s < S; ++s) {
    rc = size_of(tables[s], n_keys ? n_keys + s : nullptr, n_vals ? n_vals + s : nullptr);
    if (rc) return rc;
  }
  return PSKV_OK;
}

int pskv_dump(pskv_table* t, uint64_t* keys, int32_t* lens, size_t cap_keys, float* vals,
              size_t cap_vals, size_t* n_keys, size_t* n_vals) {
  clear_error();
  if (!t) return set_error(PSKV_EINVAL, "null table");
  uint64_t nk = 0, nv = 0;
  int rc = pskv_size(t, &nk, &nv);
  if (rc) return rc;
  if (n_keys) *n_keys = nk;
  if (n_vals) *n_vals = nv;
  if (nk > cap_keys || nv > cap_vals)
    return set_error(PSKV_ESIZE_MISMATCH, "dump needs room for %llu keys and %llu values",
                     (unsigned long long)nk, (unsigned long long)nv);
  if (nk == 0) return PSKV_OK;
  DeviceGuard guard(t->device);
  const uint64_t in_slots = t->count - (t->st_host->special_present ? 1 : 0);
  if (in_slots) {
    uint64_t* d_keys = nullptr;
    unsigned long long* d_counter = nullptr;
    PSKV_HIP(hipMalloc(reinterpret_cast<void**>(&d_keys), in_slots * sizeof(uint64_t)));
    hipError_t e = hipMalloc(reinterpret_cast<void**>(&d_counter), sizeof(unsigned long long));
    if (e == hipSuccess) e = hipMemsetAsync(d_counter, 0, sizeof(unsigned long long), t->stream);
    if (e == hipSuccess) {
      k_collect_keys<<<dim3(grid_for(t->cap, kBlock, kMaxGrid)), dim3(kBlock), 0, t->stream>>>(
          t->slots, t->cap, d_keys, in_slots, d_counter);
      e = hipMemcpyAsync(keys, d_keys, in_slots * sizeof(uint64_t), hipMemcpyDeviceToHost, t->stream);
    }
    if (e == hipSuccess) e = hipStreamSynchronize(t->stream);
    (void)hipFree(d_keys);
    if (d_counter) (void)hipFree(d_counter);
    PSKV_HIP(e);
  }
  if (t->st_host->special_present) keys[in_slots] = kEmptyKey;
  std::sort(keys, keys + nk);
  // every key is present, so this pull changes nothing in the store
  size_t got = 0;
  std::vector<int32_t> tmp_lens;
  int32_t* lens_out = lens;
  if (t->mode == PSKV_MODE_VARLEN && !lens_out) {
    tmp_lens.resize(nk);
    lens_out = tmp_lens.data();
  }
  t->no_growth = true;
  rc = pskv_pull(t, keys, nk, vals, cap_vals, t->mode == PSKV_MODE_VARLEN ? lens_out : nullptr, &got,
                 PSKV_MEM_HOST);
  t->no_growth = false;
  if (rc) return rc;
  if (lens && t->mode != PSKV_MODE_VARLEN) {
    const int32_t l = t->mode == PSKV_MODE_SCALAR ? 1 : (int32_t)t->row_len;
    for (uint64_t i = 0; i < nk; ++i) lens[i] = l;
  }
  return PSKV_OK;
}

int pskv_prof_enable(pskv_table* t, int on) {
  if (!t) return set_error(PSKV_EINVAL, "null table");
  t->prof = on != 0;
  return PSKV_OK;
}

int pskv_prof_reset(pskv_table* t) {
  if (!t) return set_error(PSKV_EINVAL, "null table");
  DeviceGuard guard(t->device);
  int rc = prof_collect(t);
  for (int k = 0; k < PSKV_KERNEL_COUNT; ++k) {
    t->launches[k] = 0;
    t->total_ms[k] = 0.0;
    t->samples[k].clear();
  }
  return rc;
}

int pskv_prof_read(pskv_table* t, int kernel, uint64_t* launches, double* total_ms) {
  if (!t) return set_error(PSKV_EINVAL, "null table");
  if (kernel < 0 || kernel >= PSKV_KERNEL_COUNT) return set_error(PSKV_EINVAL, "bad kernel id");
  DeviceGuard guard(t->device);
  int rc = prof_collect(t);
  if (launches) *launches = t->launches[kernel];
  if (total_ms) *total_ms = t->total_ms[kernel];
  return rc;
}

int pskv_prof_samples(pskv_table* t, int kernel, float* out_ms, size_t cap, size_t* n) {
  if (!t || !n) return set_error(PSKV_EINVAL, "null argument");
  if (kernel < 0 || kernel >= PSKV_KERNEL_COUNT) return set_error(PSKV_EINVAL, "bad kernel id");
  DeviceGuard guard(t->device);
  int rc = prof_collect(t);
  const std::vector<float>& v = t->samples[kernel];
  *n = v.size();
  if (out_ms)
    for (size_t i = 0; i < v.size() && i < cap; ++i) out_ms[i] = v[i];
  return rc;
}

int pskv_copy_probe(pskv_table* t, void* dst, const void* src, size_t bytes) {
  if (!t) return set_error(PSKV_EINVAL, "null table");
  if ((bytes & 15) || (reinterpret_cast<uintptr_t>(dst) & 15) || (reinterpret_cast<uintptr_t>(src) & 15))
    return set_error(PSKV_EINVAL, "copy probe needs 16-byte aligned buffers and size");
  if (!bytes) return PSKV_OK;
  DeviceGuard guard(t->device);
  const uint64_t n16 = bytes / 16;
  if ((n16 + kBlock - 1) / kBlock > 0x7fffffffull) return set_error(PSKV_EINVAL, "copy too large");
  return launch(t, PSKV_KERNEL_COPY, k_copy, dim3((unsigned)((n16 + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                static_cast<f32x4*>(dst), static_cast<const f32x4*>(src), n16);
}

int pskv_table_counters(pskv_table* t, uint64_t* out, size_t cap) {
  clear_error();
  if (!t || (!out && cap)) return set_error(PSKV_EINVAL, "null argument");
  const uint64_t v[PSKV_COUNTER_COUNT] = {t->stats.requests, t->stats.growths, t->stats.growths_unasked,
                                          t->stats.spare_used, t->stats.waits, t->stats.catch_ups,
                                          t->stats.records, t->cap};
  for (size_t i = 0; i < cap && i < (size_t)PSKV_COUNTER_COUNT; ++i) out[i] = v[i];
  return PSKV_OK;
}

int pskv_device_trim(int device) {
  clear_error();
  if (device < 0 || device >= 64) return set_error(PSKV_EINVAL, "device %d out of range", device);
  DeviceGuard guard(device);
  if (!guard.ok()) return set_error(PSKV_EHIP, "cannot select device %d", device);
  array_trim(device);
  shell_trim(device);
  stream_trim(device);
  return match_trim(device);
}

const char* pskv_last_error(void) { return g_last_error.c_str(); }
const char* pskv_version(void) { return "pskv 0.1 gfx950"; }

}  // extern "C"

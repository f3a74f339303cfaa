// The lists of device arrays behind devpool.h and the threads that allocate ahead, free behind and give back.
#include "devpool.h"

#include <algorithm>
#include <chrono>
#include <condition_variable>
#include <cstdlib>
#include <deque>
#include <list>
#include <mutex>
#include <thread>
#include <unordered_map>
#include <vector>

#include "host_common.h"

namespace pskv {
namespace {

constexpr int kMaxDevices = 64;
// What a device's list may hold: 3 % of the GPU's memory (a store that starts at its default size leaves
// 1.9 GiB of smaller slot arrays behind on its way to 60M keys, and has the next one allocated).
// The oldest arrays beyond it are freed, by the thread below (hipFree waits for the device).
constexpr size_t kKeptBytes = (size_t)8 << 30;

struct Idle {
  void* ptr;
  size_t bytes;
  hipStream_t stream;  // whose work may still use it ...
  hipEvent_t done;     // ... until this event; null: nothing does
  unsigned long long number;  // of its release
};

struct Pool {
  std::mutex mu;
  std::list<Idle> idle;  // oldest first
  size_t kept = 0;
  unsigned long long releases = 0;  // so far
  std::unordered_map<void*, size_t> size_of;  // every array handed out
  std::vector<hipEvent_t> events;             // for reuse
};
Pool* pool_of(int device) {
  static Pool* pools = new Pool[kMaxDevices];  // never destroyed: tables may go during process exit
  return device >= 0 && device < kMaxDevices ? &pools[device] : nullptr;
}

// Steps of an eighth of the next power of two, so that an array one request size left fits another.
size_t rounded(size_t bytes) {
  const size_t step = std::max<size_t>(4096, (size_t)next_pow2(bytes) / 8);
  return (bytes + step - 1) / step * step;
}

// The threads below must not be inside the runtime when the process takes that down: once it is ending they free and
// give back nothing any more, and what they are at is waited for. (An array that somebody still asks for is still
// allocated: whoever asks waits for it.)
class Gate {
 public:
  static Gate& get() {
    static Gate* g = new Gate();  // never destroyed, like the threads
    return *g;
  }
  bool enter() {
    std::lock_guard<std::mutex> lk(mu_);
    if (ending_) return false;
    ++inside_;
    return true;
  }
  void leave() {
    std::lock_guard<std::mutex> lk(mu_);
    if (--inside_ == 0) cv_.notify_all();
  }

 private:
  Gate() {
    std::atexit([] {
      Gate& g = get();
      std::unique_lock<std::mutex> lk(g.mu_);
      g.ending_ = true;
      g.cv_.wait(lk, [&] { return g.inside_ == 0; });
    });
  }
  std::mutex mu_;
  std::condition_variable cv_;
  int inside_ = 0;
  bool ending_ = false;
};

// (other threads of the process may be capturing a stream: what the threads here allocate and free is no part of that)
void relaxed_capture() {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  (void)hipThreadExchangeStreamCaptureMode(&mode);
}

// One thread per process, started with the first job, kept until the process ends.
class Worker {
 public:
  static Worker& get() {
    static Worker* w = new Worker();  // never destroyed: its thread may outlive static destructors
    return *w;
  }
  void submit(const std::shared_ptr<AllocJob>& job) {
    {
      std::lock_guard<std::mutex> lk(mu_);
      start();
      jobs_.push_back(job);
    }
    cv_job_.notify_one();
  }
  void free_later(int device, std::vector<Idle>&& what) {
    {
      std::lock_guard<std::mutex> lk(mu_);
      start();
      for (const Idle& i : what) frees_.push_back({device, i});
    }
    cv_job_.notify_one();
  }
  void wait(const std::shared_ptr<AllocJob>& job) {
    std::unique_lock<std::mutex> lk(mu_);
    cv_done_.wait(lk, [&] { return job->done; });
  }
  bool finished(const std::shared_ptr<AllocJob>& job) {
    std::lock_guard<std::mutex> lk(mu_);
    return job->done;
  }

 private:
  void start() {
    if (started_) return;
    (void)Gate::get();
    std::thread(&Worker::run, this).detach();
    started_ = true;
  }
  void run();
  std::mutex mu_;
  std::condition_variable cv_job_, cv_done_;
  std::deque<std::shared_ptr<AllocJob>> jobs_;
  std::deque<std::pair<int, Idle>> frees_;
  bool started_ = false;
};

// Counts the tables of every device and gives back what they have left some time after the last one has gone, by a
// thread of its own (one that waits with a timer costs the arrays that the other one allocates 2 us each).
class Keeper {
 public:
  static Keeper& get() {
    static Keeper* k = new Keeper();  // never destroyed
    return *k;
  }
  void tables(int device, int change, void (*give_back)(int)) {
    {
      std::lock_guard<std::mutex> lk(mu_);
      Device& d = devices_[device];
      d.tables += change;
      d.due = change < 0 && d.tables == 0;
      if (!d.due) return;
      d.when = Clock::now() + std::chrono::milliseconds(kLingerMs);
      d.give_back = give_back;
      if (!started_) {
        (void)Gate::get();
        std::thread(&Keeper::run, this).detach();
        started_ = true;
      }
      // (waking the thread costs a program that makes and drops one table after the other 5 us each time: one that is
      // going to look in time anyway is left alone)
      if (wakes_ <= d.when) return;
    }
    cv_.notify_one();
  }

 private:
  typedef std::chrono::steady_clock Clock;
  struct Device {
    long tables = 0;
    bool due = false;  // what is kept goes back at `when`
    Clock::time_point when;
    void (*give_back)(int) = nullptr;
  };
  void run() {
    relaxed_capture();
    std::unique_lock<std::mutex> lk(mu_);
    for (;;) {
      Clock::time_point next = Clock::time_point::max();
      int device = -1;
      const Clock::time_point now = Clock::now();
      for (int d = 0; d < kMaxDevices; ++d) {
        if (!devices_[d].due) continue;
        if (devices_[d].when <= now) device = d; else next = std::min(next, devices_[d].when);
      }
      if (device < 0) {
        wakes_ = next;
        if (next == Clock::time_point::max()) cv_.wait(lk); else cv_.wait_until(lk, next);
        wakes_ = Clock::time_point::min();
        continue;
      }
      devices_[device].due = false;
      void (*give_back)(int) = devices_[device].give_back;
      lk.unlock();
      if (Gate::get().enter()) {
        if (hipSetDevice(device) == hipSuccess) give_back(device);
        Gate::get().leave();
      }
      lk.lock();
    }
  }
  std::mutex mu_;
  std::condition_variable cv_;
  Device devices_[kMaxDevices];
  Clock::time_point wakes_ = Clock::time_point::min();  // when the thread is going to look by itself
  bool started_ = false;
};

void free_now(Pool* p, const Idle& i) {
  if (i.done) {
    // (an event of a stream that is gone by now is an error; hipFree waits for the device anyway)
    if (hipEventSynchronize(i.done) != hipSuccess) (void)hipGetLastError();
    std::lock_guard<std::mutex> lk(p->mu);
    p->events.push_back(i.done);
  }
  (void)hipFree(i.ptr);
}

void Worker::run() {
  relaxed_capture();
  for (;;) {
    std::shared_ptr<AllocJob> job;
    std::pair<int, Idle> gone;
    {
      std::unique_lock<std::mutex> lk(mu_);
      cv_job_.wait(lk, [&] { return !jobs_.empty() || !frees_.empty(); });
      if (!jobs_.empty()) {
        job = jobs_.front();
        jobs_.pop_front();
      } else {
        gone = frees_.front();
        frees_.pop_front();
      }
    }
    const bool inside = Gate::get().enter();
    if (!job) {
      if (inside && hipSetDevice(gone.first) == hipSuccess) free_now(pool_of(gone.first), gone.second);
      if (inside) Gate::get().leave();
      continue;
    }
    const auto a0 = std::chrono::steady_clock::now();
    if (hipSetDevice(job->device) != hipSuccess) {
      (void)hipGetLastError();
      job->rc = PSKV_EHIP;
    } else {
      job->rc = array_alloc(&job->ptr, job->bytes, job->stream);
    }
    job->took_us = std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - a0).count();
    {
      std::lock_guard<std::mutex> lk(mu_);
      job->done = true;
    }
    cv_done_.notify_all();
    if (inside) Gate::get().leave();
  }
}

}  // namespace

int array_alloc(void** out, size_t bytes, hipStream_t stream) {
  int dev = 0;
  PSKV_HIP(hipGetDevice(&dev));
  Pool* p = pool_of(dev);
  if (!p) return set_error(PSKV_EINVAL, "device %d out of range", dev);
  bytes = rounded(bytes ? bytes : 1);
  if (!arrays_are_kept()) {
    PSKV_HIP(hipMalloc(out, bytes));
    return PSKV_OK;
  }
  Idle got = {nullptr, 0, nullptr, nullptr, 0};
  {
    std::lock_guard<std::mutex> lk(p->mu);
    // the smallest that fits without wasting more than a quarter; among equals one that nothing waits for
    auto best = p->idle.end();
    auto ready = [&](const Idle& i) { return !i.done || i.stream == stream; };
    for (auto i = p->idle.begin(); i != p->idle.end(); ++i) {
      if (i->bytes < bytes || i->bytes > bytes + bytes / 4) continue;
      if (best == p->idle.end() || i->bytes < best->bytes || (i->bytes == best->bytes && !ready(*best) && ready(*i)))
        best = i;
    }
    if (best != p->idle.end()) {
      got = *best;
      p->kept -= got.bytes;
      p->size_of[got.ptr] = got.bytes;
      p->idle.erase(best);
      if (got.done && got.stream == stream) {  // the order of the stream is all it takes
        p->events.push_back(got.done);
        got.done = nullptr;
      }
    }
  }
  if (got.ptr) {
    if (got.done) {
      const hipError_t e = hipStreamWaitEvent(stream, got.done, 0);
      {
        std::lock_guard<std::mutex> lk(p->mu);
        p->events.push_back(got.done);
      }
      if (e != hipSuccess) {
        (void)array_release(got.ptr, stream);
        PSKV_HIP(e);
      }
    }
    *out = got.ptr;
    return PSKV_OK;
  }
  hipError_t e = hipMalloc(out, bytes);
  if (e == hipErrorOutOfMemory) {  // (what the list holds may be what is missing)
    (void)hipGetLastError();
    array_trim(dev);
    e = hipMalloc(out, bytes);
  }
  PSKV_HIP(e);
  std::lock_guard<std::mutex> lk(p->mu);
  p->size_of[*out] = bytes;
  return PSKV_OK;
}

bool arrays_are_kept() {
  static const bool kept = std::getenv("PSKV_NO_ASYNC_ALLOC") == nullptr;
  return kept;
}

int array_release(void* ptr, hipStream_t stream, bool idle) {
  if (!ptr) return PSKV_OK;
  if (!arrays_are_kept()) {
    if (!idle) PSKV_HIP(hipStreamSynchronize(stream));
    PSKV_HIP(hipFree(ptr));
    return PSKV_OK;
  }
  int dev = 0;
  PSKV_HIP(hipGetDevice(&dev));
  Pool* p = pool_of(dev);
  Idle i = {ptr, 0, stream, nullptr, 0};
  std::vector<Idle> over;
  {
    std::lock_guard<std::mutex> lk(p->mu);
    auto it = p->size_of.find(ptr);
    if (it == p->size_of.end()) return set_error(PSKV_EINVAL, "an array that is not this device's");
    if (!idle) {
      hipError_t e = hipSuccess;
      if (p->events.empty()) {
        e = hipEventCreateWithFlags(&i.done, hipEventDisableTiming);
      } else {
        i.done = p->events.back();
        p->events.pop_back();
      }
      if (e == hipSuccess) e = hipEventRecord(i.done, stream);
      if (e != hipSuccess) {  // (no event to go by: wait here)
        (void)hipGetLastError();
        PSKV_HIP(hipStreamSynchronize(stream));
        if (i.done) p->events.push_back(i.done);
        i.done = nullptr;
      }
    }
    i.bytes = it->second;
    i.number = ++p->releases;
    p->size_of.erase(it);
    p->idle.push_back(i);
    p->kept += i.bytes;
    while (p->kept > kKeptBytes) {
      over.push_back(p->idle.front());
      p->kept -= p->idle.front().bytes;
      p->idle.pop_front();
    }
  }
  if (!over.empty()) Worker::get().free_later(dev, std::move(over));
  return PSKV_OK;
}

unsigned long long array_mark(int device) {
  Pool* p = pool_of(device);
  if (!p) return 0;
  std::lock_guard<std::mutex> lk(p->mu);
  return p->releases;
}

void array_settle(int device, hipStream_t stream, unsigned long long mark) {
  Pool* p = pool_of(device);
  if (!p) return;
  std::lock_guard<std::mutex> lk(p->mu);
  for (Idle& i : p->idle) {
    if (!i.done || i.stream != stream || i.number > mark) continue;
    p->events.push_back(i.done);
    i.done = nullptr;
  }
}

void array_trim(int device) {
  Pool* p = pool_of(device);
  if (!p) return;
  std::list<Idle> all;
  {
    std::lock_guard<std::mutex> lk(p->mu);
    all.swap(p->idle);
    p->kept = 0;
  }
  for (const Idle& i : all) free_now(p, i);
}

void device_tables(int device, int tables, void (*give_back)(int device)) {
  if (device >= 0 && device < kMaxDevices) Keeper::get().tables(device, tables, give_back);
}

void alloc_submit(const std::shared_ptr<AllocJob>& job) { Worker::get().submit(job); }
void alloc_wait(const std::shared_ptr<AllocJob>& job) { Worker::get().wait(job); }
bool alloc_finished(const std::shared_ptr<AllocJob>& job) { return Worker::get().finished(job); }

}  // namespace pskv

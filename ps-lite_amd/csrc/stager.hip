// The ring of pinned pieces and the worker threads behind Stager (stager.h).
#include "stager.h"

#include <emmintrin.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <deque>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "host_common.h"

namespace pskv {

// memcpy whose stores go past the caches: what it writes is read by the copy engine, or by the caller a while
// later, and stores through the caches read every line from memory before they write it.
static void copy_past_caches(void* dst, const void* src, size_t len) {
  char* d = static_cast<char*>(dst);
  const char* s = static_cast<const char*>(src);
  const size_t head = std::min(len, (size_t)(-reinterpret_cast<uintptr_t>(d) & 63));
  std::memcpy(d, s, head);
  d += head, s += head, len -= head;
  for (; len >= 64; d += 64, s += 64, len -= 64) {
    const __m128i a = _mm_loadu_si128(reinterpret_cast<const __m128i*>(s));
    const __m128i b = _mm_loadu_si128(reinterpret_cast<const __m128i*>(s + 16));
    const __m128i c = _mm_loadu_si128(reinterpret_cast<const __m128i*>(s + 32));
    const __m128i e = _mm_loadu_si128(reinterpret_cast<const __m128i*>(s + 48));
    _mm_stream_si128(reinterpret_cast<__m128i*>(d), a);
    _mm_stream_si128(reinterpret_cast<__m128i*>(d + 16), b);
    _mm_stream_si128(reinterpret_cast<__m128i*>(d + 32), c);
    _mm_stream_si128(reinterpret_cast<__m128i*>(d + 48), e);
  }
  std::memcpy(d, s, len);
  _mm_sfence();
}

struct Stager::Impl {
  int device = 0;
  // The streams of the copy commands (default priority), which take turns: one stream leaves the link idle for
  // about 15 us between two commands, a tenth of a piece's time.
  hipStream_t copy[kStreams] = {nullptr};
  char* ring = nullptr;        // kSlots pieces of pinned memory
  hipEvent_t dma_done[kSlots];   // the copy command that last used the slot has finished
  hipEvent_t prod_done[2];       // device -> host: the producer has written the first piece, and everything

  std::mutex op_mu;  // one transfer at a time: the host link is what they would share anyway

  // worker threads: plain memcpy between caller memory and the ring
  struct Job {
    void* dst;
    const void* src;
    size_t len;
    int slot;
  };
  std::mutex mu;
  std::condition_variable cv_job, cv_done;
  std::deque<Job> jobs;
  std::atomic<int> queued{0};                 // jobs.size()
  std::atomic<int> pending[kSlots] = {};      // parts of the slot's piece that workers still owe
  std::atomic<int> sleepers{0}, waiters{0};   // threads in cv_job and cv_done

  char* slot_ptr(int s) const { return ring + (size_t)s * kPiece; }

  // Looks for `ready` for about 100 us before a thread goes to sleep: the next piece, or the next transfer, is
  // mostly nearer than that, and waking a thread costs the start and the end of a transfer 30 to 50 us each.
  template <typename F>
  static bool look_for(F ready) {
    const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(100);
    do {
      for (int spin = 0; spin < 64; ++spin) {
        if (ready()) return true;
        __builtin_ia32_pause();
      }
    } while (std::chrono::steady_clock::now() < until);
    return ready();
  }

  void work() {
    for (;;) {
      (void)look_for([&] { return queued.load() > 0; });
      Job j;
      {
        std::unique_lock<std::mutex> lk(mu);
        if (jobs.empty()) {
          ++sleepers;
          cv_job.wait(lk, [&] { return !jobs.empty(); });
          --sleepers;
        }
        j = jobs.front();
        jobs.pop_front();
        --queued;
      }
      copy_past_caches(j.dst, j.src, j.len);
      // (a waiter counts itself in before it looks at `pending` for the last time)
      if (--pending[j.slot] == 0 && waiters.load() > 0) {
        std::lock_guard<std::mutex> lk(mu);
        cv_done.notify_all();
      }
    }
  }
  // A piece is copied in kParts parts by as many workers: it is ready (or gone) in an eighth of
  // the time, which is what a transfer of a few dozen pieces waits for at its start and its end.
  void submit(void* dst, const void* src, size_t len, int slot) {
    const size_t part = ((len + kParts - 1) / kParts + 4095) & ~(size_t)4095;
    if (len == 0) return;
    bool wake;
    {
      std::lock_guard<std::mutex> lk(mu);
      int n = 0;
      for (size_t at = 0; at < len; at += part, ++n)
        jobs.push_back(Job{static_cast<char*>(dst) + at, static_cast<const char*>(src) + at,
                           std::min(part, len - at), slot});
      pending[slot] = n;
      queued += n;
      wake = sleepers.load() > 0;
    }
    if (wake) cv_job.notify_all();
  }
  void wait_slot(int slot) {
    if (look_for([&] { return pending[slot].load() == 0; })) return;
    std::unique_lock<std::mutex> lk(mu);
    ++waiters;
    cv_done.wait(lk, [&] { return pending[slot].load() == 0; });
    --waiters;
  }
  bool slot_free(int slot) { return pending[slot].load() == 0; }
};

Stager* Stager::get(int device) {
  constexpr int kMaxDevices = 64;
  static std::mutex* mu = new std::mutex();
  static Stager* table[kMaxDevices] = {nullptr};
  static bool failed[kMaxDevices] = {false};
  if (device < 0 || device >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lk(*mu);
  if (table[device] || failed[device]) return table[device];
  // never destroyed: worker threads and pinned memory live until the process ends
  Impl* im = new (std::nothrow) Impl();
  if (!im) return nullptr;
  im->device = device;
  bool ok = true;
  for (int q = 0; ok && q < kStreams; ++q) ok = hipStreamCreateWithFlags(&im->copy[q], hipStreamNonBlocking) == hipSuccess;
  ok = ok && hipHostMalloc(reinterpret_cast<void**>(&im->ring), (size_t)kSlots * kPiece, hipHostMallocDefault) ==
                 hipSuccess;
  for (int s = 0; ok && s < kSlots; ++s) {
    ok = hipEventCreateWithFlags(&im->dma_done[s], hipEventDisableTiming) == hipSuccess;
  }
  for (hipEvent_t& e : im->prod_done) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
  if (!ok) {
    (void)hipGetLastError();
    failed[device] = true;  // (what was created stays; this happens once)
    return nullptr;
  }
  for (int w = 0; w < kWorkers; ++w) std::thread([im] { im->work(); }).detach();
  table[device] = new Stager(im);
  return table[device];
}

namespace {

// Where the pieces of a transfer begin (and, last, where it ends). Whatever the workers copy before the first
// command can go out, or after the last one has come in, is time in which the link stands still: on the way to
// the device the first pieces are short and double up to kPiece, on the way back the last ones halve.
std::vector<size_t> cut(size_t bytes, bool to_device) {
  constexpr size_t kLeast = 512u << 10, kUnit = 64u << 10;
  std::vector<size_t> at(1, 0);
  for (size_t len = kLeast; at.back() < bytes;) {
    const size_t left = bytes - at.back();
    if (!to_device) len = std::max(kLeast, (left / 2 + kUnit - 1) / kUnit * kUnit);
    at.push_back(at.back() + std::min(left, std::min(len, Stager::kPiece)));
    if (to_device) len = std::min(2 * len, Stager::kPiece);
  }
  return at;
}

}  // namespace

int Stager::to_device(void* dst, const void* src, size_t bytes, hipStream_t consumer,
                      const std::function<int(size_t, size_t)>& consume) {
  static_assert(kStreams == 2, "the last two commands are the last of each stream");
  Impl* im = impl_;
  std::lock_guard<std::mutex> op(im->op_mu);
  const std::vector<size_t> at = cut(bytes, true);
  const size_t npieces = at.size() - 1;
  auto len_of = [&](size_t c) { return at[c + 1] - at[c]; };
  size_t issued = 0, sent = 0, consumed = 0;
  int status = PSKV_OK;
  auto check = [&](hipError_t e) {
    if (e != hipSuccess && !status)
      status = set_error(PSKV_EHIP, "staging a request failed: %s", hipGetErrorString(e));
    return e == hipSuccess;
  };
  while (sent < npieces && status == PSKV_OK) {
    // keep the workers busy: the free slots of the ring get the next pieces. kSlack slots stay
    // behind the piece being sent, so that the wait below is for a copy command two or three
    // back and the copy engine always has the next command queued.
    while (issued < npieces && issued + kSlack < sent + kSlots) {
      const int slot = (int)(issued % kSlots);
      // the copy command that last read this slot (this transfer's or an earlier one's) is done
      if (!check(hipEventSynchronize(im->dma_done[slot]))) break;
      im->submit(im->slot_ptr(slot), static_cast<const char*>(src) + at[issued], len_of(issued), slot);
      ++issued;
    }
    if (status) break;
    const int slot = (int)(sent % kSlots);
    const size_t off = at[sent], len = len_of(sent);
    hipStream_t copy = im->copy[sent % kStreams];
    im->wait_slot(slot);
    if (!check(hipMemcpyAsync(static_cast<char*>(dst) + off, im->slot_ptr(slot), len, hipMemcpyHostToDevice, copy)) ||
        !check(hipEventRecord(im->dma_done[slot], copy)))
      break;
    // The consumer works through what has arrived in stretches of kStretch pieces, and at the end on the last
    // piece alone: it needs a fortieth of the transfer's time, and a stream that waits for every piece holds
    // up the copy commands where it shares a hardware queue with one of theirs.
    if ((sent + 1) % kStretch == 0 || sent + 2 >= npieces) {
      bool ok = check(hipStreamWaitEvent(consumer, im->dma_done[slot], 0));
      if (ok && sent > 0) ok = check(hipStreamWaitEvent(consumer, im->dma_done[(sent - 1) % kSlots], 0));
      if (!ok) break;
      if (consume) status = consume(at[consumed], off + len - at[consumed]);
      consumed = sent + 1;
    }
    ++sent;
  }
  if (status) {
    // the workers still read the caller's memory: it is the caller's again only when they are done
    for (int s = 0; s < kSlots; ++s) im->wait_slot(s);
  }
  return status;
}

int Stager::to_host(void* dst, const void* src, size_t bytes, hipStream_t producer,
                    const std::function<int(size_t, size_t)>& produce) {
  // A slot that this transfer fills may still be read by a copy command of the transfer before it: no wait is made
  // for that, both are on the same stream (piece c lies in slot c % kSlots and goes over stream c % kStreams).
  static_assert(kSlots % kStreams == 0, "a slot always meets the same stream");
  Impl* im = impl_;
  std::lock_guard<std::mutex> op(im->op_mu);
  const std::vector<size_t> at = cut(bytes, false);
  const size_t npieces = at.size() - 1;
  auto len_of = [&](size_t c) { return at[c + 1] - at[c]; };
  size_t launched = 0, drained = 0;
  int status = PSKV_OK;
  while (drained < npieces && status == PSKV_OK) {
    // Produce and send off every piece whose slot is free (the worker that emptied it for an
    // earlier piece is done); never wait for a worker while pieces that have arrived could be
    // handed to the others.
    while (launched < npieces && launched < drained + kSlots) {
      const int slot = (int)(launched % kSlots);
      if (!im->slot_free(slot)) {
        if (drained < launched) break;  // hand out what has arrived first
        im->wait_slot(slot);
      }
      const size_t off = at[launched], len = len_of(launched);
      hipStream_t copy = im->copy[launched % kStreams];
      // The producer's work is done for the first piece, then for all the others at once: it takes a fortieth of
      // the transfer's time, and a producer that takes turns with the copy commands holds them up (9 to 20 us a
      // piece).
      hipError_t e = hipSuccess;
      if (launched < 2) {
        if (produce) {
          status = produce(off, launched == 0 ? len : bytes - off);
          if (status) break;
        }
        e = hipEventRecord(im->prod_done[launched], producer);
        if (e == hipSuccess) e = hipStreamWaitEvent(copy, im->prod_done[launched], 0);
      } else if (launched < 1 + kStreams) {
        e = hipStreamWaitEvent(copy, im->prod_done[1], 0);
      }
      if (e == hipSuccess)
        e = hipMemcpyAsync(im->slot_ptr(slot), static_cast<const char*>(src) + off, len, hipMemcpyDeviceToHost,
                           copy);
      if (e == hipSuccess) e = hipEventRecord(im->dma_done[slot], copy);
      if (e != hipSuccess) {
        status = set_error(PSKV_EHIP, "staging a response failed: %s", hipGetErrorString(e));
        break;
      }
      ++launched;
    }
    if (status) break;
    const int slot = (int)(drained % kSlots);
    const hipError_t e = hipEventSynchronize(im->dma_done[slot]);
    if (e != hipSuccess) {
      status = set_error(PSKV_EHIP, "staging a response failed: %s", hipGetErrorString(e));
      break;
    }
    im->submit(static_cast<char*>(dst) + at[drained], im->slot_ptr(slot), len_of(drained), slot);
    ++drained;
  }
  // nothing of this transfer may be left in the ring or in flight when the caller gets its buffer
  for (int s = 0; s < kSlots; ++s) im->wait_slot(s);
  if (status)
    for (hipStream_t copy : im->copy) (void)hipStreamSynchronize(copy);
  return status;
}

}  // namespace pskv

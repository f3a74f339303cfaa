// A stand-in for the few calls that csrc/devpool.hip makes, for tests of its bookkeeping on the CPU: memory is host
// memory, a stream is a counter of work queued and done, an event the count that it was recorded at. Every call is
// written down where a test can look.
#ifndef PSKV_TEST_HOST_HIP_H_
#define PSKV_TEST_HOST_HIP_H_
#include <stddef.h>
#include <stdlib.h>

#include <map>
#include <mutex>
#include <utility>
#include <vector>

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorInvalidValue = 1 };
enum hipStreamCaptureMode { hipStreamCaptureModeRelaxed = 2 };
struct HostStream {
  unsigned long queued = 0, done = 0;
};
struct HostEvent {
  HostStream* stream = nullptr;
  unsigned long at = 0;
  bool complete() const { return !stream || stream->done >= at; }
};
typedef HostStream* hipStream_t;
typedef HostEvent* hipEvent_t;
constexpr unsigned hipEventDisableTiming = 2;

struct HostHip {
  std::mutex mu;
  std::map<void*, size_t> live;                               // memory that is allocated
  size_t live_bytes = 0, room = (size_t)1 << 40;              // `room`: more than that fails
  std::vector<std::pair<hipStream_t, HostEvent>> waits;       // what streams were made to wait for
};
inline HostHip& host_hip() {
  static HostHip* h = new HostHip();
  return *h;
}

inline const char* hipGetErrorString(hipError_t) { return "error"; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*) { return hipSuccess; }
inline hipError_t hipMalloc(void** p, size_t bytes) {
  std::lock_guard<std::mutex> lk(host_hip().mu);
  if (host_hip().live_bytes + bytes > host_hip().room) return hipErrorOutOfMemory;
  *p = malloc(1);  // (nobody looks inside)
  host_hip().live[*p] = bytes;
  host_hip().live_bytes += bytes;
  return hipSuccess;
}
inline hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> lk(host_hip().mu);
  auto it = host_hip().live.find(p);
  if (it == host_hip().live.end()) return hipErrorInvalidValue;
  host_hip().live_bytes -= it->second;
  host_hip().live.erase(it);
  free(p);
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = new HostEvent(), hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { return delete e, hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { return e->stream = s, e->at = s->queued, hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  if (e->stream && e->stream->done < e->at) e->stream->done = e->at;
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) { return s->done = s->queued, hipSuccess; }
inline hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  std::lock_guard<std::mutex> lk(host_hip().mu);
  host_hip().waits.push_back({s, *e});
  return hipSuccess;
}
#endif  // PSKV_TEST_HOST_HIP_H_

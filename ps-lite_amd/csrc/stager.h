// Staging of large host-resident requests and responses.
//
// A ps-lite server receives requests in ordinary host memory (the transport's receive buffers,
// src/zmq_van.h:179-227; KVServer::Process hands them over as they are, include/ps/kv_app.h:468-494)
// and answers into host memory. The copy engines of the GPU only reach pinned memory at full
// speed, so a large transfer goes through a ring of pinned pieces, and the three stages of
// every piece overlap with those of its neighbours:
//   host -> device:  worker threads copy piece c+1 into the ring while piece c is in flight to
//                    the GPU and the kernel that consumes earlier pieces runs;
//   device -> host:  piece c+1 is in flight to the ring while worker threads copy piece c to the
//                    caller's buffer; the kernel that produces what follows the first piece runs
//                    while that piece is in flight.
#ifndef PSKV_STAGER_H_
#define PSKV_STAGER_H_
#include <hip/hip_runtime.h>
#include <stddef.h>

#include <functional>

namespace pskv {

class Stager {
 public:
  static constexpr size_t kPiece = 8u << 20;  // most bytes per piece of the ring
  static constexpr int kSlots = 16;           // pieces in the ring (128 MiB of pinned memory)
  static constexpr int kSlack = 3;            // slots kept between the piece being sent and the next refill
  static constexpr int kStreams = 2;          // streams that the copy commands alternate between
  static constexpr int kStretch = 8;          // pieces that the consumer of a transfer takes at a time
  static constexpr int kWorkers = 8;          // threads that copy between caller memory and the ring
  static constexpr int kParts = 8;            // a piece is copied in this many parts, by as many workers

  // The stager of `device`, created on first use and kept until the process ends; nullptr when
  // its pinned memory cannot be had (the caller then falls back to plain copy commands).
  static Stager* get(int device);

  // Copies `bytes` from ordinary host memory `src` to device memory `dst`, piece by piece, in
  // order. Every few pieces, `consumer` is made to wait for all that is on its way and
  // `consume(offset, len)` is called on the calling thread for what is new of it (it may enqueue the work
  // that consumes those bytes on `consumer`; it may be empty). Returns a PSKV_* status.
  int to_device(void* dst, const void* src, size_t bytes, hipStream_t consumer,
                const std::function<int(size_t, size_t)>& consume);

  // Copies `bytes` from device memory `src` to ordinary host memory `dst`, piece by piece, in
  // order. `produce(offset, len)` is called on the calling thread, for the first piece and for all
  // that follows it (it may enqueue the work that produces those bytes on `producer`; it may be empty);
  // a piece is copied once `producer` has got that far. Returns when everything has arrived in `dst`.
  int to_host(void* dst, const void* src, size_t bytes, hipStream_t producer,
              const std::function<int(size_t, size_t)>& produce);

 private:
  struct Impl;
  explicit Stager(Impl* impl) : impl_(impl) {}
  Impl* impl_;
};

}  // namespace pskv
#endif  // PSKV_STAGER_H_

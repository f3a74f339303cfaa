// Device arrays that outlive the table they were made for.
//
// A slot array, a row arena or a request buffer that a table gives up (a growth has replaced it, or the
// table is gone) goes on a list of its device and serves the next table or growth that asks for about
// that size. Releasing it instead, and allocating again, sends the memory through the driver: unmapped,
// cleared, mapped, 0.15 to 0.4 ms per array on a quiet process and up to 300 ms where GBs have changed
// hands shortly before. (The runtime's own stream-ordered pool was measured in this place first: it
// hands back what an idle stream frees, whatever its release threshold, and cost a store that is
// filled, dropped and filled again 25 to 160 ms per round.)
#ifndef PSKV_DEVPOOL_H_
#define PSKV_DEVPOOL_H_
#include <hip/hip_runtime.h>
#include <stddef.h>

#include <memory>

namespace pskv {

// An array of at least `bytes` bytes on the current device, to be used in the order of `stream`. (The
// memory may still be in use by earlier work of that stream, or of one that `stream` is made to wait for.)
int array_alloc(void** out, size_t bytes, hipStream_t stream);
// Gives an array back (null: nothing). Work already enqueued on `stream` may still use it; `idle`: nothing does.
int array_release(void* ptr, hipStream_t stream, bool idle = false);
// For a stream of `device` that is waited for and may be destroyed: array_mark() before the wait, and
// behind it array_settle() with what it said: nothing that had been released by then depends on the stream any
// more. (What another thread releases on the same stream meanwhile does.)
unsigned long long array_mark(int device);
void array_settle(int device, hipStream_t stream, unsigned long long mark);
// Frees every array on the list of `device` (current). Waits for those that are still in use.
void array_trim(int device);
// False with PSKV_NO_ASYNC_ALLOC in the environment: arrays come from hipMalloc and go to hipFree, nothing is kept.
bool arrays_are_kept();

// A table of `device` has come (`tables` = 1) or gone (-1). What tables leave is there for the next ones, so it goes
// back when there are none: kLingerMs after the last table of the device has gone, unless another has come by then,
// a thread of the library's own calls `give_back` (with the device current). A program that drops its tables and makes others, the
// case the lists are for, does so within that time; giving back at once is what cost it 25 to 160 ms.
constexpr int kLingerMs = 2000;
void device_tables(int device, int tables, void (*give_back)(int device));

// Allocations made by a thread of the library's own: allocating a few hundred MB costs the calling
// thread 50 us on a good day and 800 on a bad one, so the array of a coming growth is asked for
// while the caller goes on enqueuing requests; the growth picks the result up (and waits for it in the
// unlikely case that it is not there yet).
struct AllocJob {
  int device = 0;
  size_t bytes = 0;
  hipStream_t stream = nullptr;
  void* ptr = nullptr;
  int rc = 0;
  double took_us = 0;  // what the allocation cost the allocating thread
  bool done = false;   // guarded by the worker's lock
};
void alloc_submit(const std::shared_ptr<AllocJob>& job);
void alloc_wait(const std::shared_ptr<AllocJob>& job);
bool alloc_finished(const std::shared_ptr<AllocJob>& job);

}  // namespace pskv
#endif  // PSKV_DEVPOOL_H_

// Runs a kernel of csrc/ on the CPU, one workgroup after the other, for tests of what its wavefronts do to each
// other: every thread is a context of its own, the 64 threads of a wavefront meet in their shuffles and all of a
// workgroup at its barriers, and between two barriers the wavefronts run one after the other in an order that the
// test chooses. (One that runs ahead as far as the barriers let it is an order the GPU may take as well.)
// Compile with clang (vector types) and -fno-strict-aliasing.
#ifndef PSKV_TEST_HOST_WAVE_H_
#define PSKV_TEST_HOST_WAVE_H_
#include <stddef.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>
#include <ucontext.h>

#include <vector>

#define __device__
#define __global__
#define __host__
#define __forceinline__ inline
#define __shared__ thread_local  // (one thread runs them all; `extern` may stand in front of it)
#define __launch_bounds__(...)
#define __align__(n) alignas(n)
#define __HIP_MEMORY_SCOPE_AGENT 0
#define __HIP_MEMORY_SCOPE_SYSTEM 0
#define __hip_atomic_store(p, v, order, scope) (*(p) = (v))
#define __hip_atomic_load(p, order, scope) (*(p))
#define __builtin_amdgcn_fence(...) ((void)0)
#define __builtin_amdgcn_s_waitcnt(x) ((void)0)
#define __builtin_amdgcn_s_sleep(x) ((void)0)
#define __builtin_amdgcn_wave_barrier() ((void)0)

struct ulonglong2 {
  unsigned long long x, y;
};
struct dim3 {
  unsigned x = 1, y = 1, z = 1;
};

struct HostWaves {
  enum At { kRuns, kShuffle, kBarrier, kDone };
  std::vector<ucontext_t> ctx;
  std::vector<std::vector<char>> stack;
  std::vector<At> at;
  std::vector<unsigned long long> given, got;
  std::vector<int> from;  // whose word a lane asks for
  std::vector<int> any;   // __syncthreads_or
  int any_of_all = 0;
  ucontext_t back;
  unsigned now = 0;
  dim3 thread, block, grid, block_dim;
  void (*body)(void*) = nullptr;
  void* arg = nullptr;
};
inline HostWaves& host_waves() {
  static HostWaves* w = new HostWaves();
  return *w;
}
#define threadIdx (host_waves().thread)
#define blockIdx (host_waves().block)
#define gridDim (host_waves().grid)
#define blockDim (host_waves().block_dim)

inline void host_yield(HostWaves::At why) {
  HostWaves& w = host_waves();
  const unsigned me = w.now;
  w.at[me] = why;
  swapcontext(&w.ctx[me], &w.back);
}
inline void host_thread() {
  HostWaves& w = host_waves();
  w.body(w.arg);
  host_yield(HostWaves::kDone);
}

inline void __syncthreads() { host_yield(HostWaves::kBarrier); }
inline int __syncthreads_or(int x) {
  HostWaves& w = host_waves();
  w.any[w.now] = x;
  host_yield(HostWaves::kBarrier);
  return w.any_of_all;
}
template <typename T>
T host_shuffle(T x, int from) {
  static_assert(sizeof(T) <= 8, "one word");
  HostWaves& w = host_waves();
  const unsigned me = w.now;
  w.given[me] = 0;
  memcpy(&w.given[me], &x, sizeof(T));
  w.from[me] = from;
  host_yield(HostWaves::kShuffle);
  memcpy(&x, &w.got[me], sizeof(T));
  return x;
}
inline unsigned __lane_id() { return host_waves().now & 63u; }
template <typename T> T __shfl_xor(T x, int o) { return host_shuffle(x, (int)__lane_id() ^ o); }
template <typename T> T __shfl_up(T x, int o) { return host_shuffle(x, (int)__lane_id() >= o ? (int)__lane_id() - o : (int)__lane_id()); }
template <typename T> T __shfl_down(T x, int o) { return host_shuffle(x, (int)__lane_id() + o < 64 ? (int)__lane_id() + o : (int)__lane_id()); }
template <typename T> T __shfl(T x, int from) { return host_shuffle(x, from & 63); }

inline unsigned long long __ballot(int) { abort(); }  // (no kernel that a test runs here has one)
inline int __any(int) { abort(); }

inline void __threadfence() {}
inline void __threadfence_system() {}
template <typename T, typename U> T atomicAdd(T* p, U x) { const T old = *p; *p = old + (T)x; return old; }
template <typename T, typename U> T atomicOr(T* p, U x) { const T old = *p; *p = old | (T)x; return old; }
template <typename T, typename U> T atomicExch(T* p, U x) { const T old = *p; *p = (T)x; return old; }
template <typename T> T atomicCAS(T* p, T from, T to) { const T old = *p; if (old == from) *p = to; return old; }
inline float __uint_as_float(unsigned x) { float f; memcpy(&f, &x, 4); return f; }
inline unsigned __float_as_uint(float f) { unsigned x; memcpy(&x, &f, 4); return x; }

// One workgroup of `threads` threads: between barriers wavefront order[0] runs first, then order[1], ...
inline void host_workgroup(unsigned threads, const std::vector<unsigned>& order, void (*body)(void*), void* arg) {
  HostWaves& w = host_waves();
  w.ctx.resize(threads), w.stack.resize(threads);
  w.at.assign(threads, HostWaves::kRuns);
  w.given.assign(threads, 0), w.got.assign(threads, 0), w.from.assign(threads, 0), w.any.assign(threads, 0);
  w.body = body, w.arg = arg;
  w.block_dim.x = threads;
  for (unsigned i = 0; i < threads; ++i) {
    w.stack[i].resize(64 << 10);
    getcontext(&w.ctx[i]);
    w.ctx[i].uc_stack.ss_sp = w.stack[i].data();
    w.ctx[i].uc_stack.ss_size = w.stack[i].size();
    w.ctx[i].uc_link = &w.back;
    makecontext(&w.ctx[i], host_thread, 0);
  }
  for (;;) {
    bool over = true;
    for (unsigned wave : order) {
      const unsigned lo = wave * 64, hi = lo + 64 < threads ? lo + 64 : threads;
      for (bool more = true; more;) {  // until every thread of the wavefront is at a barrier or done
        more = false;
        for (unsigned i = lo; i < hi; ++i) {
          if (w.at[i] != HostWaves::kRuns) continue;
          w.now = i, w.thread.x = i;
          swapcontext(&w.back, &w.ctx[i]);
        }
        for (unsigned i = lo; i < hi; ++i)
          if (w.at[i] == HostWaves::kShuffle) w.got[i] = w.given[lo + (unsigned)w.from[i]];
        for (unsigned i = lo; i < hi; ++i)
          if (w.at[i] == HostWaves::kShuffle) w.at[i] = HostWaves::kRuns, more = true;
      }
    }
    // (threads that have ended do not count at a barrier)
    w.any_of_all = 0;
    for (unsigned i = 0; i < threads; ++i)
      if (w.at[i] == HostWaves::kBarrier) over = false, w.any_of_all |= w.any[i];
    for (unsigned i = 0; i < threads; ++i) w.any[i] = 0;
    if (over) return;
    for (unsigned i = 0; i < threads; ++i)
      if (w.at[i] == HostWaves::kBarrier) w.at[i] = HostWaves::kRuns;
  }
}
#endif  // PSKV_TEST_HOST_WAVE_H_

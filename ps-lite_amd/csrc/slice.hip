// Worker-side kernels: the key-range slicer that replaces KVWorker::DefaultSlicer
// (include/ps/kv_app.h:517-572) and the device-side reassembly of pulled slices
// that mirrors the callback of KVWorker::AddPullCB (kv_app.h:663-714).
#include <algorithm>
#include <cstring>
#include <limits>
#include <mutex>
#include <numeric>
#include <vector>

#include "device_common.h"
#include "host_common.h"
#include "parts.h"
#include "search.h"
#include "stream_choice.h"

namespace pskv {
namespace {

// One wavefront per search target.
__global__ __launch_bounds__(kBlock) void k_bounds(const uint64_t* __restrict__ keys, uint64_t n,
                                                  const uint64_t* __restrict__ targets,
                                                  uint64_t ntargets, uint64_t* __restrict__ lb) {
  const uint64_t w = ((uint64_t)blockIdx.x * kBlock + threadIdx.x) >> 6;
  const unsigned lane = threadIdx.x & 63;
  if (w >= ntargets) return;  // whole wavefronts leave together
  const uint64_t lo = wave_lower_bound(keys, n, targets[w], lane);
  if (lane == 0) lb[w] = lo;
}

// (a marked word of parts.h)
__device__ __forceinline__ void tell(uint64_t* to, uint64_t x) {
  __hip_atomic_store(to, x | kHere, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The largest of this lane's and all lower lanes' values.
__device__ __forceinline__ uint64_t wave_running_max(uint64_t x, unsigned lane) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint64_t y = __shfl_up(x, o);
    if (lane >= (unsigned)o && y > x) x = y;
  }
  return x;
}

// kv_app.h:528-541: pos[0] = lower_bound(keys, ranges[0].begin); every further
// boundary is searched in the suffix that starts at the previous one, which for
// sorted keys is max(previous, lower_bound over the whole array).
// One wavefront. `pos` is device memory (read by the lens sums), `pos_host` pinned host
// memory the caller reads after the stream wait (may be null); `sums` (may be null) is
// cleared for the kernel that follows.
__global__ void k_bounds_chain(const uint64_t* __restrict__ lb, uint64_t S,
                               uint64_t* __restrict__ pos, uint64_t* __restrict__ pos_host,
                               unsigned long long* __restrict__ sums) {
  if (blockIdx.x != 0) return;
  if (sums)
    for (uint64_t i = threadIdx.x; i < S; i += blockDim.x) sums[i] = 0ull;
  if (threadIdx.x != 0) return;
  uint64_t p = lb[0];
  pos[0] = p;
  if (pos_host) tell(&pos_host[0], p);
  for (uint64_t i = 0; i < S; ++i) {
    const uint64_t e = lb[i + 1];
    p = e > p ? e : p;
    pos[i + 1] = p;
    if (pos_host) tell(&pos_host[i + 1], p);
  }
}

// Both of the above in one launch when the boundaries are few and the positions are for a kernel behind it: one
// workgroup of up to 16 wavefronts, each searching one or two boundaries, then the chain.
// The boundaries travel with the launch: no read across the host link before the search.
constexpr unsigned kFusedWaves = 16;
struct FusedTargets {
  uint64_t v[kFusedTargets];
};
__global__ __launch_bounds__(kFusedWaves * 64) void k_bounds_fused(
    const uint64_t* __restrict__ keys, uint64_t n, uint64_t* __restrict__ pos, uint64_t* __restrict__ pos_host,
    unsigned long long* __restrict__ sums, unsigned S, unsigned waves, FusedTargets targets) {
  __shared__ uint64_t s_lb[kFusedTargets];
  const unsigned lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  static_assert(kFusedTargets == 2 * kFusedWaves, "two boundaries for a wavefront at most");
  const unsigned second = wave + waves < kFusedTargets ? wave + waves : 0u;
  const uint64_t target[2] = {targets.v[wave], targets.v[second]};
  PSKV_ASK_ARGS("s"(keys), "s"(n), "s"(pos), "s"(pos_host), "s"(sums), "s"(S), "s"(target[0]), "s"(target[1]));
#pragma unroll
  for (unsigned q = 0; q < 2; ++q) {
    const unsigned w = wave + q * waves;
    if (w > S) continue;
    const uint64_t lo = wave_lower_bound(keys, n, target[q], lane);
    if (lane == 0) s_lb[w] = lo;
  }
  __syncthreads();
  if (threadIdx.x >= 64) return;
  if (sums && lane < S) sums[lane] = 0ull;
  static_assert(kFusedTargets <= 64, "a lane per position");
  uint64_t p = 0;  // (the reads of LDS do not wait for each other, the steps of a scan over the lanes would)
  for (unsigned i = 0; i <= S; ++i) p = i <= lane && s_lb[i] > p ? s_lb[i] : p;
  if (lane <= S) {
    pos[lane] = p;
    if (pos_host) tell(&pos_host[lane], p);
  }
}

// The searches of a request without lens, or whose lens nobody adds up here: a wavefront and compute unit for each boundary,
// which tells the host what it has found; the host takes the larger of each and the one before. (A round of a search is 64
// lines, and one compute unit asks for a line a clock: 17 searches in one workgroup took 2 us longer than two. us per call,
// one workgroup -> this: 1,000 keys over 4 ranges 9.6 -> 8.4, 20,000 over 1 9.5 -> 8.7, over 16 11.6 -> 9.2, 1M over 4 9.9 ->
// 9.0, 16M over 16 11.8 -> 9.4. More probes a round, to save rounds: slower, a round that follows is 0.3 us.)
__global__ __launch_bounds__(64) void k_bounds_tell(const uint64_t* __restrict__ keys, uint64_t n,
                                                   uint64_t* __restrict__ lb_host, FusedTargets targets) {
  const uint64_t target = targets.v[blockIdx.x];
  PSKV_ASK_ARGS("s"(keys), "s"(n), "s"(lb_host), "s"(target));
  const uint64_t lo = wave_lower_bound(keys, n, target, threadIdx.x);
  if (threadIdx.x == 0) tell(&lb_host[blockIdx.x], lo);
}

// Boundaries and the lens sums of the slices between them in one launch (few boundaries, in ascending
// order). A workgroup takes one stretch of the request: two keys tell it which boundaries fall inside,
// it searches those there, adds up the lens between them, and hands positions and sums over past the
// L2; the workgroup that finishes last writes everything to pinned memory. The lens of a request are
// read once and nothing else is: 2M keys over 16 ranges took three launches (6.8 + 10.1 us, and the sums'
// way to the host) and a stream wait, 38 us per call; this is one launch and the watched word.
constexpr unsigned kSumsMaxBlocks = 256;  // (every workgroup takes a ticket of one counter, about 10 ns each)
struct SumsState {                         // device memory of one slicer context, all zero between calls
  unsigned long long pos[kFusedTargets];
  unsigned long long sums[kFusedTargets];
  unsigned ticket;
};
// What the workgroup that finishes last hands to the host. One wavefront.
__device__ __forceinline__ void hand_over(SumsState* state, unsigned S, unsigned lane, uint64_t* pos_host,
                                          unsigned long long* sums_host) {
  uint64_t p = 0;
  if (lane <= S) p = __hip_atomic_load(&state->pos[lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (lane < S)
    tell(reinterpret_cast<uint64_t*>(&sums_host[lane]),
         __hip_atomic_load(&state->sums[lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  p = wave_running_max(p, lane);
  if (lane <= S) tell(&pos_host[lane], p);
  // (the next call's kernel is behind this one on the stream)
  if (lane < S) state->sums[lane] = 0ull;
  if (lane <= S) state->pos[lane] = 0ull;  // (keys that are not sorted may leave a boundary without an owner)
  if (lane == 0) state->ticket = 0;
}

// A request of up to kFewSumsKeys keys: everything that a workgroup needs is asked for at once, eight keys and lens a
// thread, the lens are added up by one scan, and the key that a boundary falls in front of says where that is and what lies
// below. The workgroups do not meet: each tells the host what its part's lens add up to, which boundaries are its own and,
// for each of those, where in the part it is and what lies below it there, and the host puts the parts together (a word a
// part, told of in the order they arrive). (The searches of the kernel below are trips to memory that follow from each other,
// every slice is added up for itself, and a sum passes through the L2, a ticket and the workgroup that finishes last.
// us per call: 1,000 keys over 3 ranges 10.6 (12.2 when the workgroups met over a ticket and the last handed everything
// over), 5,000 over 16 11.9 (13.6; the searches of the kernel below 19.2), 15,826 over 3 11.1 (12.6; 15.1), 262,144 over 4
// 12.0 (13.6). The searches against this: 400,000 over 8 15.5 and 12.8, 1M over 16 16.9 and 14.9, but with a thousand words
// for the host to read 2M over 16 17.0 and 17.3: up to 512 parts.)
__global__ __launch_bounds__(kFewSumsBlock) void k_bounds_sums_few(const uint64_t* __restrict__ keys,
                                                                   const int32_t* __restrict__ lens, uint64_t n,
                                                                   uint64_t* __restrict__ bounds_host,
                                                                   uint64_t* __restrict__ parts_host, unsigned S,
                                                                   FusedTargets targets) {
  PSKV_ASK_ARGS("s"(keys), "s"(lens), "s"(n), "s"(bounds_host), "s"(parts_host), "s"(S));
  constexpr unsigned kWaves = kFewSumsBlock / 64;
  typedef int32_t i32x4u __attribute__((ext_vector_type(4), aligned(4)));
  typedef unsigned long long u64x2u __attribute__((ext_vector_type(2), aligned(8)));
  __shared__ unsigned long long s_wave[kWaves];
  __shared__ uint64_t s_at[kFusedTargets], s_target[kFusedTargets];
  __shared__ unsigned long long s_below[kFusedTargets];
  __shared__ uint64_t s_before, s_end;
  const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t c0 = (uint64_t)blockIdx.x * kFewSumsPart;
  const uint64_t c1 = n - c0 < kFewSumsPart ? n : c0 + kFewSumsPart;
  const uint64_t i0 = c0 + (uint64_t)threadIdx.x * kFewSumsItems;
  const unsigned mine = i0 >= c1 ? 0u : c1 - i0 < kFewSumsItems ? (unsigned)(c1 - i0) : kFewSumsItems;
  uint64_t key[kFewSumsItems], prev = 0;
  unsigned long long len[kFewSumsItems];
  if (mine == kFewSumsItems) {
#pragma unroll
    for (unsigned j = 0; j < kFewSumsItems; j += 4) {
      const u64x2u a = *reinterpret_cast<const u64x2u*>(keys + i0 + j), b = *reinterpret_cast<const u64x2u*>(keys + i0 + j + 2);
      const i32x4u l = *reinterpret_cast<const i32x4u*>(lens + i0 + j);
      key[j] = a.x, key[j + 1] = a.y, key[j + 2] = b.x, key[j + 3] = b.y;
#pragma unroll
      for (unsigned r = 0; r < 4; ++r) len[j + r] = (unsigned long long)(long long)l[r];
    }
  } else {
#pragma unroll
    for (unsigned j = 0; j < kFewSumsItems; ++j) {
      key[j] = j < mine ? keys[i0 + j] : 0;
      len[j] = j < mine ? (unsigned long long)(long long)lens[i0 + j] : 0ull;
    }
  }
  if (mine && i0) prev = keys[i0 - 1];
  if (threadIdx.x < kFusedTargets) s_target[threadIdx.x] = targets.v[threadIdx.x];
  if (threadIdx.x == 0) s_before = prev;
  uint64_t top = key[0];  // the thread's last key
#pragma unroll
  for (unsigned j = 1; j < kFewSumsItems; ++j) top = j < mine ? key[j] : top;
  if (mine && i0 + mine == c1) s_end = top;
  unsigned long long sum = 0;
#pragma unroll
  for (unsigned j = 0; j < kFewSumsItems; ++j) sum += len[j];
  const unsigned long long upto = wave_incl_scan_u64(sum);
  if (lane == 63) s_wave[wave] = upto;
  __syncthreads();
  unsigned long long below = upto - sum, all = 0;
#pragma unroll
  for (unsigned w = 0; w < kWaves; ++w) {
    if (w < wave) below += s_wave[w];
    all += s_wave[w];
  }
  uint64_t near = s_target[0];
  for (unsigned i = 0; i <= S; ++i) {  // (few threads hold a boundary, most boundaries lie elsewhere)
    const uint64_t target = near;
    near = s_target[i < S ? i + 1 : S];  // (the next one is on its way)
    if (!mine || top < target || (i0 && prev >= target)) continue;
    unsigned long long x = below;
    uint64_t at = i0;
#pragma unroll
    for (unsigned j = 0; j + 1 < kFewSumsItems; ++j)
      if (j < mine && key[j] < target) x += len[j], ++at;
    s_at[i] = at;
    s_below[i] = x;
  }
  __syncthreads();
  if (threadIdx.x >= 64) return;
  const uint64_t before = s_before, end = s_end;
  bool own = false;
  if (lane <= S) {
    const uint64_t target = s_target[lane];
    const bool after_start = c0 == 0 || before < target, inside = after_start && end >= target;
    // the boundary is this part's if it does not lie before it, nor behind it unless it is the last one
    own = after_start && (c1 == n || inside);
    if (own) tell(&bounds_host[lane], part_word(inside ? s_below[lane] : all, (inside ? s_at[lane] : c1) - c0));
  }
  const unsigned long long owned = __ballot(own);  // (the boundaries ascend: these follow each other)
  if (lane == 0)
    tell(&parts_host[blockIdx.x],
         part_word(all, owned ? (unsigned long long)__builtin_ctzll(owned) | (unsigned long long)__popcll(owned) << 6 : 0ull));
}

__global__ __launch_bounds__(kBlock) void k_bounds_sums(const uint64_t* __restrict__ keys,
                                                       const int32_t* __restrict__ lens, uint64_t n, uint64_t chunk,
                                                       FusedTargets targets, unsigned S, SumsState* state,
                                                       uint64_t* __restrict__ pos_host,
                                                       unsigned long long* __restrict__ sums_host) {
  __shared__ uint64_t s_b[kFusedTargets];
  __shared__ unsigned long long s_red[kBlock / 64];
  __shared__ unsigned s_last;
  const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t c0 = (uint64_t)blockIdx.x * chunk;
  const uint64_t c1 = n - c0 < chunk ? n : c0 + chunk;
  const uint64_t before = c0 ? keys[c0 - 1] : 0, last = keys[c1 - 1];
  for (unsigned i = wave; i <= S; i += kBlock / 64) {  // whole wavefronts
    const uint64_t target = targets.v[i];
    const bool after_start = c0 == 0 || before < target;  // the boundary does not lie before this stretch
    const bool mine = after_start && (c1 == n || last >= target);
    uint64_t at = after_start ? c1 : c0;
    if (mine) at = c0 + wave_lower_bound(keys + c0, c1 - c0, target, lane);
    if (lane == 0) {
      s_b[i] = at;
      if (mine) __hip_atomic_store(&state->pos[i], (unsigned long long)at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  __syncthreads();
  for (unsigned i = 0; i < S; ++i) {
    const uint64_t b = s_b[i], e = s_b[i + 1];
    if (e <= b) continue;  // (the same for the whole workgroup)
    unsigned long long sum = 0;
    uint64_t j = b + threadIdx.x;
    for (; j + 7 * kBlock < e; j += 8 * kBlock) {  // loads of a round before its adds
      int32_t l[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) l[u] = lens[j + (uint64_t)u * kBlock];
#pragma unroll
      for (int u = 0; u < 8; ++u) sum += (unsigned long long)(long long)l[u];
    }
    for (; j < e; j += kBlock) sum += (unsigned long long)(long long)lens[j];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    if (lane == 0) s_red[wave] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
      unsigned long long t = 0;
      for (unsigned w = 0; w < kBlock / 64; ++w) t += s_red[w];
      if (t) atomicAdd(&state->sums[i], t);
    }
    __syncthreads();
  }
  __builtin_amdgcn_s_waitcnt(0);  // what this lane has handed over is there before the ticket is taken
  __syncthreads();
  if (threadIdx.x == 0) {
    s_last = atomicAdd(&state->ticket, 1u) == gridDim.x - 1 ? 1u : 0u;
    if (s_last) __threadfence();
  }
  __syncthreads();
  if (!s_last) return;
  if (threadIdx.x >= 64) return;
  hand_over(state, S, lane, pos_host, sums_host);
}

// ---- the slicer for callers that cannot allocate ------------------------------------------
// Working memory of pskv_slice_noalloc: the lower bounds of the boundary searches followed by
// the per-slice sums of lens. It lives in the code object, so every GPU that loads the library
// holds its own copy until the process ends; host code reaches it through the address that
// hipGetSymbolAddress returns on that GPU, never through this name.
constexpr size_t kNoAllocMaxRanges = PSKV_SLICE_NOALLOC_MAX_RANGES;
constexpr size_t kNoAllocLb = kNoAllocMaxRanges + 1;            // words [0, kNoAllocLb): lower bounds
constexpr size_t kNoAllocWords = kNoAllocLb + kNoAllocMaxRanges;  // then kNoAllocMaxRanges sums
static __device__ __align__(256) unsigned long long scratch[kNoAllocWords];

// Up to kFusedTargets searches whose targets travel with the launch; the answers go to lb[].
__global__ __launch_bounds__(kFusedWaves * 64) void k_bounds_args(const uint64_t* __restrict__ keys,
                                                                 uint64_t n, FusedTargets targets,
                                                                 unsigned count,
                                                                 unsigned long long* __restrict__ lb) {
  const unsigned lane = threadIdx.x & 63, waves = blockDim.x >> 6;
  for (unsigned w = threadIdx.x >> 6; w < count; w += waves) {  // whole wavefronts
    const uint64_t lo = wave_lower_bound(keys, n, targets.v[w], lane);
    if (lane == 0) lb[w] = lo;
  }
}

// What pskv_slice does on the host once the positions and the per-slice sums are known
// (kv_app.h:540-571), by one thread, with the outputs in device memory: the `first` flags,
// the coverage check, the value offsets and their checks. `late_error` is a status the host
// already knows but which the reference raises only after the coverage check.
__global__ void k_noalloc_finish(const uint64_t* __restrict__ pos,
                                 const unsigned long long* __restrict__ sums, uint64_t S, uint64_t n,
                                 uint64_t nvals, uint64_t k, int has_lens, int late_error,
                                 uint64_t* __restrict__ val_pos, uint8_t* __restrict__ used,
                                 int32_t* __restrict__ status) {
  for (uint64_t i = threadIdx.x; i <= S; i += blockDim.x) val_pos[i] = 0;
  for (uint64_t i = threadIdx.x; i < S; i += blockDim.x) used[i] = pos[i + 1] != pos[i];  // kv_app.h:540
  __syncthreads();
  if (threadIdx.x != 0) return;
  if (pos[S] != n) {  // kv_app.h:542
    *status = PSKV_EUNCOVERED_KEY;
    return;
  }
  *status = PSKV_OK;
  if (n == 0) return;  // kv_app.h:543
  if (late_error) {    // kv_app.h:549,551
    *status = late_error;
    return;
  }
  if (!has_lens) {
    for (uint64_t i = 0; i <= S; ++i) val_pos[i] = pos[i] * k;  // kv_app.h:569
    return;
  }
  uint64_t val_begin = 0, val_end = 0;  // kv_app.h:563-567 with the CHECKs of sarray.h:249
  for (uint64_t i = 0; i < S; ++i) {
    val_pos[i] = val_begin;
    if (pos[i + 1] != pos[i]) {
      val_end += sums[i];
      if (val_end < val_begin || val_end > nvals) {
        val_pos[i + 1] = val_end;
        *status = PSKV_ESIZE_MISMATCH;
        return;
      }
      val_begin = val_end;
    }
    val_pos[i + 1] = val_end;
  }
}

// Hands the per-slice sums to the host (pinned memory).
__global__ void k_export_sums(const unsigned long long* __restrict__ sums, uint64_t S,
                              unsigned long long* __restrict__ sums_host) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < S;
       i += (uint64_t)gridDim.x * blockDim.x)
    sums_host[i] = sums[i];
}

// kv_app.h:565 `for (int l : kv.lens) val_end += l;` for every slice at once:
// blockIdx.y is the slice, the workgroups of a slice stride over its lens.
// Sums are taken modulo 2^64 over sign-extended lens, like size_t += int.
__global__ __launch_bounds__(kBlock) void k_segment_sums(const int32_t* __restrict__ lens,
                                                        const uint64_t* __restrict__ pos,
                                                        unsigned long long* __restrict__ sums) {
  __shared__ unsigned long long red[kBlock / 64];
  const uint64_t begin = pos[blockIdx.y], end = pos[blockIdx.y + 1];
  unsigned long long s = 0;
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t i = begin + (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < end; i += stride)
    s += (unsigned long long)(long long)lens[i];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long t = 0;
    for (int w = 0; w < kBlock / 64; ++w) t += red[w];
    if (t) atomicAdd(&sums[blockIdx.y], t);
  }
}

// First key and last key + 1 of every response (FindRange arguments, kv_app.h:671).
__global__ void k_response_ends(const uint64_t* const* __restrict__ resp_keys,
                                const uint64_t* __restrict__ resp_nkeys, uint64_t R,
                                uint64_t* __restrict__ targets) {
  const uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= R) return;
  targets[2 * r] = resp_keys[r][0];
  targets[2 * r + 1] = resp_keys[r][resp_nkeys[r] - 1] + 1;  // wraps to 0 for kMaxKey, as Key does
}

// One piece of a concatenation: `bytes` bytes (a multiple of 4, 4-byte aligned) from src to dst.
struct Segment {
  const char* src;
  char* dst;
  uint64_t bytes;
};

struct __attribute__((packed, aligned(4))) Words4 {
  uint32_t w[4];
};

// Copies all segments of a table (blockIdx.y = segment; the workgroups of a row stride over
// it). The destination is written with aligned 128-bit stores whatever its start: the first
// lanes move single words up to the next 16-byte boundary, and the loads that feed the
// stores may then sit on any 4-byte boundary, which global memory allows.
__global__ __launch_bounds__(kBlock) void k_concat(const Segment* __restrict__ segs) {
  const Segment sg = segs[blockIdx.y];
  if (sg.bytes == 0) return;
  uint64_t head = (16 - (reinterpret_cast<uintptr_t>(sg.dst) & 15)) & 15;  // bytes to the boundary
  if (head > sg.bytes) head = sg.bytes;
  const uint64_t body = (sg.bytes - head) / 16;  // 128-bit pieces
  const uint64_t tail_at = head + body * 16;
  const uint64_t t0 = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  if (t0 < head / 4)
    reinterpret_cast<uint32_t*>(sg.dst)[t0] = reinterpret_cast<const uint32_t*>(sg.src)[t0];
  if (t0 < (sg.bytes - tail_at) / 4)
    reinterpret_cast<uint32_t*>(sg.dst + tail_at)[t0] =
        reinterpret_cast<const uint32_t*>(sg.src + tail_at)[t0];
  const Words4* src = reinterpret_cast<const Words4*>(sg.src + head);
  f32x4* dst = reinterpret_cast<f32x4*>(sg.dst + head);
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t i = t0; i < body; i += stride) {
    const Words4 x = src[i];
    f32x4 y;
    y.x = __uint_as_float(x.w[0]);
    y.y = __uint_as_float(x.w[1]);
    y.z = __uint_as_float(x.w[2]);
    y.w = __uint_as_float(x.w[3]);
    __builtin_nontemporal_store(y, dst + i);
  }
}

// Per-call state of the slicer. Calls may come from any thread at once
// (KVWorker::Push is thread-safe, kv_app.h:101-104), so each call takes a context
// of its own from a pool and returns it afterwards.
struct SliceCtx {
  int device = -1;
  hipStream_t stream = nullptr;  // the one in use, of
  hipStream_t streams[kSliceStreams] = {nullptr};
  StreamChoice choice;
  SumsState* sums_state = nullptr;
  void* dev = nullptr;      // device scratch: targets, lower bounds, positions, sums
  size_t dev_bytes = 0;
  void* pinned = nullptr;   // pinned host memory the kernels read targets from and answer into
  size_t pinned_bytes = 0;
};

std::mutex g_pool_mu;
std::vector<SliceCtx*> g_pool;

SliceCtx* take_ctx(int device) {
  {
    std::lock_guard<std::mutex> lk(g_pool_mu);
    for (size_t i = 0; i < g_pool.size(); ++i) {
      if (g_pool[i]->device == device) {
        SliceCtx* c = g_pool[i];
        g_pool.erase(g_pool.begin() + i);
        return c;
      }
    }
  }
  SliceCtx* c = new (std::nothrow) SliceCtx();
  if (!c) return nullptr;
  c->device = device;
  // (all of them at once: a stream gets the queue that the fewest are on, so they end up on one each and leave the tables'
  // streams spread as they were)
  bool streams = true;
  for (hipStream_t& s : c->streams) streams = streams && hipStreamCreateWithFlags(&s, hipStreamNonBlocking) == hipSuccess;
  if (!streams ||
      hipMalloc(reinterpret_cast<void**>(&c->sums_state), sizeof(SumsState)) != hipSuccess ||
      hipMemset(c->sums_state, 0, sizeof(SumsState)) != hipSuccess) {
    if (c->sums_state) (void)hipFree(c->sums_state);
    for (hipStream_t s : c->streams)
      if (s) (void)hipStreamDestroy(s);
    delete c;
    return nullptr;
  }
  c->stream = c->streams[0];
  return c;
}

// A call on the context's stream has taken `us`, `own` by itself, and nothing of it is left: the stream of the next one.
void note_call(SliceCtx* c, float us, float own) {
  const int next = c->choice.note(us, own);
  if (next == c->choice.at) return;
  if (hipStreamSynchronize(c->stream) != hipSuccess) return;  // (the kernel may still be clearing its state)
  c->choice.at = next;
  c->stream = c->streams[next];
}

void give_ctx(SliceCtx* c) {
  std::lock_guard<std::mutex> lk(g_pool_mu);
  g_pool.push_back(c);
}

// A context goes back to the pool only when nothing enqueued on its stream can still touch its
// buffers: a call that leaves early (after a failed runtime call) waits for the stream first.
struct CtxLease {
  SliceCtx* c;
  bool idle = true;  // nothing has been enqueued since the stream was last waited for
  explicit CtxLease(int device) : c(take_ctx(device)) {}
  ~CtxLease() {
    if (!c) return;
    if (!idle) (void)hipStreamSynchronize(c->stream);
    give_ctx(c);
  }
};

int ctx_reserve(SliceCtx* c, size_t dev_bytes, size_t pinned_bytes) {
  if (dev_bytes > c->dev_bytes) {
    if (c->dev) PSKV_HIP(hipFree(c->dev));
    c->dev = nullptr;
    c->dev_bytes = 0;
    PSKV_HIP(hipMalloc(&c->dev, dev_bytes));
    c->dev_bytes = dev_bytes;
  }
  if (pinned_bytes > c->pinned_bytes) {
    if (c->pinned) PSKV_HIP(hipHostFree(c->pinned));
    c->pinned = nullptr;
    c->pinned_bytes = 0;
    // coherent: never cached by the GPU, so every call sees what the host wrote for it
    PSKV_HIP(hipHostMalloc(&c->pinned, pinned_bytes, hipHostMallocCoherent));
    c->pinned_bytes = pinned_bytes;
  }
  return PSKV_OK;
}

inline size_t pad256(size_t b) { return (b + 255) & ~(size_t)255; }

int launch_bounds_search(const uint64_t* keys, uint64_t n, const uint64_t* targets, uint64_t nt,
                         uint64_t* lb, hipStream_t stream) {
  const unsigned blocks = (unsigned)((nt * 64 + kBlock - 1) / kBlock);
  k_bounds<<<dim3(blocks), dim3(kBlock), 0, stream>>>(keys, n, targets, nt, lb);
  PSKV_HIP(hipGetLastError());
  return PSKV_OK;
}

}  // namespace
}  // namespace pskv

using namespace pskv;

extern "C" {

int pskv_server_ranges(uint64_t num_servers, uint64_t* range_begin, uint64_t* range_end) {
  clear_error();
  if (num_servers == 0 || !range_begin || !range_end)
    return set_error(PSKV_EINVAL, "need at least one server and two output arrays");
  const uint64_t max_key = std::numeric_limits<uint64_t>::max();  // ps::kMaxKey, base.h:18
  for (uint64_t i = 0; i < num_servers; ++i) {
    range_begin[i] = max_key / num_servers * i;        // postoffice.cc:174
    range_end[i] = max_key / num_servers * (i + 1);    // postoffice.cc:175
  }
  return PSKV_OK;
}

int pskv_slice(int device, const uint64_t* keys, size_t n, const int32_t* lens, size_t nlens,
               size_t nvals, const uint64_t* range_begin, const uint64_t* range_end, size_t S,
               uint64_t* pos, uint64_t* val_pos, uint8_t* used, int memkind) {
  clear_error();
  if (memkind != PSKV_MEM_HOST && memkind != PSKV_MEM_DEVICE)
    return set_error(PSKV_EINVAL, "bad memkind %d", memkind);
  if (!pos || !val_pos || (S && (!used || !range_begin || !range_end)))
    return set_error(PSKV_EINVAL, "null argument");
  if (n && !keys) return set_error(PSKV_EINVAL, "null keys");
  for (size_t i = 0; i <= S; ++i) pos[i] = val_pos[i] = 0;
  for (size_t i = 0; i < S; ++i) used[i] = 0;
  // kv_app.h:533 CHECK_EQ(ranges[i-1].end(), ranges[i].begin()); it fires inside the
  // loop, before the coverage check of :542
  for (size_t i = 1; i < S; ++i) {
    if (range_end[i - 1] != range_begin[i])
      return set_error(PSKV_ERANGE_GAP, "ranges[%zu].end != ranges[%zu].begin", i - 1, i);
  }
  if (S == 0) {
    if (n) return set_error(PSKV_EUNCOVERED_KEY, "no ranges for %zu keys", n);
    return PSKV_OK;
  }
  const bool has_lens = lens != nullptr && nlens != 0;

  const bool do_sums = has_lens && nlens == n;
  if (n && do_sums && S > 65535) return set_error(PSKV_EINVAL, "more than 65535 ranges with lens");
  bool on_device = n != 0;  // (device-resident requests: searches and sums on the GPU)
  if (n && memkind == PSKV_MEM_HOST) {
    // Keys in host memory are searched where they lie: S+1 lower bounds touch (S+1) log2 n keys,
    // and shipping all n keys over the host link for that would cost milliseconds at model size
    // (and a launch and a wait at any size). This is the reference's own loop (kv_app.h:524-541).
    const uint64_t* begin = keys;
    const uint64_t* end = keys + n;
    for (size_t i = 0; i < S; ++i) {
      if (i == 0) {
        pos[0] = (uint64_t)(std::lower_bound(begin, end, range_begin[0]) - begin);
        begin += pos[0];
      }
      const size_t len = (size_t)(std::lower_bound(begin, end, range_end[i]) - begin);
      begin += len;
      pos[i + 1] = pos[i] + len;
    }
    // The lens too: one core adds them up faster (8 MB in 0.2 ms) than pageable memory crosses the
    // host link (0.28 ms for the same 8 MB, before any kernel runs): the walk of kv_app.h:563-565.
    on_device = false;
    if (do_sums) {
      for (size_t i = 0; i < S; ++i) {
        uint64_t sum = 0;
        for (uint64_t j = pos[i]; j < pos[i + 1]; ++j) sum += (uint64_t)(int64_t)lens[j];
        val_pos[i + 1] = sum;  // per-slice sums for now
      }
    }
  }

  if (on_device) {
    DeviceGuard guard(device);
    if (!guard.ok()) return set_error(PSKV_EHIP, "cannot select device %d", device);
    CtxLease lease(device);
    SliceCtx* c = lease.c;
    if (!c) return set_error(PSKV_EHIP, "cannot create a slicer context on device %d", device);
    lease.idle = false;
    // device: lb[S+1] | pos[S+1] | sums[S]      pinned: targets[S+1] | pos[S+1] | sums[S] | parts[kFewSumsParts]
    const size_t arr = pad256((S + 1) * 8);
    constexpr size_t kParts = kFewSumsParts * 8;
    int rc = ctx_reserve(c, 3 * arr, 3 * arr + kParts);
    if (rc) return rc;
    char* d = static_cast<char*>(c->dev);
    uint64_t* d_lb = reinterpret_cast<uint64_t*>(d);
    uint64_t* d_pos = reinterpret_cast<uint64_t*>(d + arr);
    unsigned long long* d_sums = reinterpret_cast<unsigned long long*>(d + 2 * arr);
    char* h = static_cast<char*>(c->pinned);
    uint64_t* h_targets = reinterpret_cast<uint64_t*>(h);
    uint64_t* h_pos = reinterpret_cast<uint64_t*>(h + arr);
    unsigned long long* h_sums = reinterpret_cast<unsigned long long*>(h + 2 * arr);
    uint64_t* h_parts = reinterpret_cast<uint64_t*>(h + 3 * arr);
    h_targets[0] = range_begin[0];
    for (size_t i = 0; i < S; ++i) h_targets[i + 1] = range_end[i];
    // With few boundaries one kernel leaves everything this call waits for in pinned memory, word by word:
    // watching for those costs about 5 us less than a stream wait. (With lens the
    // boundaries must ascend, as those of contiguous ranges do unless a range ends before it begins.)
    const bool few = S + 1 <= kFusedTargets;
    const bool sums_too = do_sums && few && n < (1ull << 31) && std::is_sorted(h_targets, h_targets + S + 1);
    const bool watch = !do_sums || sums_too;
    const auto asked = std::chrono::steady_clock::now();
    std::memset(h_pos, 0, (S + 1) * 8);
    const bool in_parts = sums_too && n <= kFewSumsKeys;
    const uint64_t nparts = in_parts ? (n + kFewSumsPart - 1) / kFewSumsPart : 0;
    if (in_parts) std::memset(h_parts, 0, nparts * 8);
    if (sums_too && !in_parts) std::memset(h_sums, 0, S * 8);
    FusedTargets ft = {};
    if (few)
      for (size_t i = 0; i <= S; ++i) ft.v[i] = h_targets[i];
    if (in_parts) {
      k_bounds_sums_few<<<dim3((unsigned)nparts), dim3(kFewSumsBlock), 0, c->stream>>>(keys, lens, n, h_pos, h_parts,
                                                                                      (unsigned)S, ft);
      PSKV_HIP(hipGetLastError());
    } else if (sums_too) {
      // (a stretch of at least 2,048 keys, a multiple of four)
      const uint64_t chunk = std::max<uint64_t>(2048, ((n + kSumsMaxBlocks - 1) / kSumsMaxBlocks + 3) & ~(uint64_t)3);
      k_bounds_sums<<<dim3((unsigned)((n + chunk - 1) / chunk)), dim3(kBlock), 0, c->stream>>>(
          keys, lens, n, chunk, ft, (unsigned)S, c->sums_state, h_pos, h_sums);
      PSKV_HIP(hipGetLastError());
    } else if (few && !do_sums) {
      k_bounds_tell<<<dim3((unsigned)(S + 1)), dim3(64), 0, c->stream>>>(keys, n, h_pos, ft);
      PSKV_HIP(hipGetLastError());
    } else if (few) {  // one launch for the boundaries
      const unsigned waves = (unsigned)std::min<size_t>(S + 1, kFusedWaves);
      k_bounds_fused<<<dim3(1), dim3(waves * 64), 0, c->stream>>>(keys, n, d_pos, h_pos, d_sums, (unsigned)S, waves, ft);
      PSKV_HIP(hipGetLastError());
    } else {
      rc = launch_bounds_search(keys, n, h_targets, S + 1, d_lb, c->stream);
      if (rc) return rc;
      k_bounds_chain<<<dim3(1), dim3(64), 0, c->stream>>>(d_lb, S, d_pos, h_pos, do_sums ? d_sums : nullptr);
      PSKV_HIP(hipGetLastError());
    }
    if (do_sums && !sums_too) {
      uint64_t per = n / S / (kBlock * 8) + 1;
      if (per > 1024) per = 1024;
      k_segment_sums<<<dim3((unsigned)per, (unsigned)S), dim3(kBlock), 0, c->stream>>>(lens, d_pos, d_sums);
      PSKV_HIP(hipGetLastError());
      k_export_sums<<<dim3((unsigned)((S + 255) / 256)), dim3(256), 0, c->stream>>>(d_sums, S, h_sums);
      PSKV_HIP(hipGetLastError());
    }
    const WatchEnd end = watch_end(std::chrono::steady_clock::now());
    if (in_parts) {
      if (!join_parts(h_parts, h_pos, n, S, pos, val_pos + 1, end)) {
        PSKV_HIP(hipStreamSynchronize(c->stream));
        (void)join_parts(h_parts, h_pos, n, S, pos, val_pos + 1, end);
      }
    } else if (!watch || !all_here(h_pos, S + 1, end) ||
               (sums_too && !all_here(reinterpret_cast<uint64_t*>(h_sums), S, end))) {
      PSKV_HIP(hipStreamSynchronize(c->stream));
    }
    lease.idle = true;  // (what the kernel still does is clear its state for the next one on the stream)
    if (watch)
      note_call(c, std::chrono::duration<float, std::micro>(std::chrono::steady_clock::now() - asked).count(),
                own_slice_us(n, S, do_sums));
    for (size_t i = 0; i <= S && !in_parts; ++i) pos[i] = std::max(told(h_pos[i]), i ? pos[i - 1] : 0);
    if (do_sums && !in_parts)
      for (size_t i = 0; i < S; ++i) val_pos[i + 1] = sums_too ? told(h_sums[i]) : h_sums[i];  // per-slice sums for now
  }

  for (size_t i = 0; i < S; ++i) used[i] = pos[i + 1] != pos[i];  // kv_app.h:540
  if (pos[S] != n)  // kv_app.h:542
    return set_error(PSKV_EUNCOVERED_KEY,
                     "Check failed: (pos[n]) == (send.keys.size()): %llu keys fall in the ranges, "
                     "%zu were given", (unsigned long long)pos[S], n);
  if (n == 0) return PSKV_OK;  // kv_app.h:543

  if (!has_lens) {
    const size_t k = nvals / n;  // kv_app.h:548
    if (k * n != nvals)          // kv_app.h:549
      return set_error(PSKV_ESIZE_MISMATCH, "%zu values do not divide over %zu keys", nvals, n);
    for (size_t i = 0; i <= S; ++i) val_pos[i] = pos[i] * k;  // kv_app.h:569
    return PSKV_OK;
  }
  if (nlens != n)  // kv_app.h:551
    return set_error(PSKV_ESIZE_MISMATCH, "%zu keys but %zu lens", n, nlens);
  // kv_app.h:563-567 with the CHECKs of SArray::segment (sarray.h:249)
  uint64_t val_begin = 0, val_end = 0;
  for (size_t i = 0; i < S; ++i) {
    const uint64_t sum = val_pos[i + 1];
    val_pos[i] = val_begin;
    if (pos[i + 1] != pos[i]) {
      val_end += sum;
      if (val_end < val_begin || val_end > nvals) {
        val_pos[i + 1] = val_end;
        return set_error(PSKV_ESIZE_MISMATCH, "lens of slice %zu reach past the %zu values", i, nvals);
      }
      val_begin = val_end;
    }
    val_pos[i + 1] = val_end;
  }
  return PSKV_OK;
}

namespace {
// Device address of `scratch` on every GPU this process has used the entry point on.
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
unsigned long long* g_scratch_ptr[kMaxDevices] = {nullptr};

// Called with `device` current. The first call on a device asks the runtime where that
// device's copy of the array lives; later calls read the table.
int noalloc_scratch(int device, unsigned long long** out) {
  if (device < 0 || device >= kMaxDevices) return set_error(PSKV_EINVAL, "device %d out of range", device);
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[device]) {
    void* p = nullptr;
    PSKV_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) return set_error(PSKV_EHIP, "no device address for the slicer's working memory");
    g_scratch_ptr[device] = static_cast<unsigned long long*>(p);
  }
  *out = g_scratch_ptr[device];
  return PSKV_OK;
}
}  // namespace

int pskv_slice_noalloc(int device, void* stream, const uint64_t* keys, size_t n, const int32_t* lens,
                       size_t nlens, size_t nvals, const uint64_t* range_begin,
                       const uint64_t* range_end, size_t S, uint64_t* pos, uint64_t* val_pos,
                       uint8_t* used, int32_t* status) {
  clear_error();
  if (!pos || !val_pos || !status || (S && (!used || !range_begin || !range_end)))
    return set_error(PSKV_EINVAL, "null argument");
  if (n && !keys) return set_error(PSKV_EINVAL, "null keys");
  if (S == 0) return set_error(PSKV_EINVAL, "pskv_slice_noalloc needs at least one range");
  if (S > kNoAllocMaxRanges)
    return set_error(PSKV_EINVAL, "pskv_slice_noalloc serves at most %zu ranges, %zu were given",
                     kNoAllocMaxRanges, S);
  for (size_t i = 1; i < S; ++i) {  // kv_app.h:533
    if (range_end[i - 1] != range_begin[i])
      return set_error(PSKV_ERANGE_GAP, "ranges[%zu].end != ranges[%zu].begin", i - 1, i);
  }
  DeviceGuard guard(device);
  if (!guard.ok()) return set_error(PSKV_EHIP, "cannot select device %d", device);
  unsigned long long* ws = nullptr;
  int rc = noalloc_scratch(device, &ws);
  if (rc) return rc;
  hipStream_t st = static_cast<hipStream_t>(stream);
  unsigned long long* d_lb = ws;
  unsigned long long* d_sums = ws + kNoAllocLb;

  const bool has_lens = lens != nullptr && nlens != 0;
  const bool do_sums = has_lens && nlens == n && n != 0;
  int late_error = PSKV_OK;
  uint64_t k = 0;
  if (n) {
    if (!has_lens) {
      k = nvals / n;  // kv_app.h:548-549
      if (k * n != nvals) late_error = PSKV_ESIZE_MISMATCH;
    } else if (nlens != n) {  // kv_app.h:551
      late_error = PSKV_ESIZE_MISMATCH;
    }
  }
  if (S + 1 <= kFusedTargets) {  // searches, chain and the clearing of the sums in one launch
    FusedTargets ft = {};
    ft.v[0] = range_begin[0];
    for (size_t i = 0; i < S; ++i) ft.v[i + 1] = range_end[i];
    const unsigned waves = (unsigned)std::min<size_t>(S + 1, kFusedWaves);
    k_bounds_fused<<<dim3(1), dim3(waves * 64), 0, st>>>(keys, n, pos, (uint64_t*)nullptr, d_sums, (unsigned)S, waves, ft);
    PSKV_HIP(hipGetLastError());
  } else {
    for (size_t first = 0; first <= S; first += kFusedTargets) {
      const size_t count = std::min<size_t>(S + 1 - first, kFusedTargets);
      FusedTargets ft = {};
      for (size_t j = 0; j < count; ++j) {
        const size_t i = first + j;
        ft.v[j] = i == 0 ? range_begin[0] : range_end[i - 1];
      }
      const unsigned waves = (unsigned)std::min<size_t>(count, kFusedWaves);
      k_bounds_args<<<dim3(1), dim3(waves * 64), 0, st>>>(keys, n, ft, (unsigned)count, d_lb + first);
      PSKV_HIP(hipGetLastError());
    }
    k_bounds_chain<<<dim3(1), dim3(64), 0, st>>>(reinterpret_cast<const uint64_t*>(d_lb), S, pos,
                                                (uint64_t*)nullptr, d_sums);
    PSKV_HIP(hipGetLastError());
  }
  if (do_sums) {
    uint64_t per = n / S / (kBlock * 8) + 1;
    if (per > 1024) per = 1024;
    k_segment_sums<<<dim3((unsigned)per, (unsigned)S), dim3(kBlock), 0, st>>>(lens, pos, d_sums);
    PSKV_HIP(hipGetLastError());
  }
  k_noalloc_finish<<<dim3(1), dim3(256), 0, st>>>(pos, d_sums, S, n, nvals, k, has_lens ? 1 : 0,
                                                   late_error, val_pos, used, status);
  PSKV_HIP(hipGetLastError());
  return PSKV_OK;
}

int pskv_assemble_pull(int device, const uint64_t* req_keys, size_t n, size_t R,
                       const uint64_t* const* resp_keys, const size_t* resp_nkeys,
                       const float* const* resp_vals, const size_t* resp_nvals,
                       const int32_t* const* resp_lens, float* out, size_t out_cap,
                       int32_t* out_lens, size_t* out_nvals, int memkind) {
  clear_error();
  if (memkind != PSKV_MEM_DEVICE)
    return set_error(PSKV_EINVAL,
                     "pskv_assemble_pull concatenates device-resident slices; host-resident "
                     "slices are reassembled by KVWorker itself");
  if (out_nvals) *out_nvals = 0;
  if (R && (!resp_keys || !resp_nkeys || !resp_vals || !resp_nvals))
    return set_error(PSKV_EINVAL, "null argument");
  size_t total_key = 0, total_val = 0;
  for (size_t r = 0; r < R; ++r) {
    if (resp_nkeys[r] == 0)  // front()/back() CHECK(!empty()), sarray.h:221-222
      return set_error(PSKV_EINVAL, "response %zu has no keys", r);
    total_key += resp_nkeys[r];
    total_val += resp_nvals[r];
  }
  std::vector<uint64_t> ends(2 * R);
  if (R) {
    DeviceGuard guard(device);
    if (!guard.ok()) return set_error(PSKV_EHIP, "cannot select device %d", device);
    CtxLease lease(device);
    SliceCtx* c = lease.c;
    if (!c) return set_error(PSKV_EHIP, "cannot create a context on device %d", device);
    lease.idle = false;
    // pinned, read and written by the kernels in place:
    //   key pointers[R] | nkeys[R] | targets[2R] | lower bounds[2R] | segments[2R]
    const size_t a = pad256(R * 8), b = pad256(2 * R * 8), sg = pad256(2 * R * sizeof(Segment));
    int rc = ctx_reserve(c, 0, 2 * a + 2 * b + sg);
    if (rc) return rc;
    char* h = static_cast<char*>(c->pinned);
    const uint64_t** h_ptrs = reinterpret_cast<const uint64_t**>(h);
    uint64_t* h_nk = reinterpret_cast<uint64_t*>(h + a);
    uint64_t* h_targets = reinterpret_cast<uint64_t*>(h + 2 * a);
    uint64_t* h_lb = reinterpret_cast<uint64_t*>(h + 2 * a + b);
    Segment* h_segs = reinterpret_cast<Segment*>(h + 2 * a + 2 * b);
    for (size_t r = 0; r < R; ++r) {
      h_ptrs[r] = resp_keys[r];
      h_nk[r] = resp_nkeys[r];
    }
    k_response_ends<<<dim3((unsigned)((R + 63) / 64)), dim3(64), 0, c->stream>>>(h_ptrs, h_nk, R,
                                                                                 h_targets);
    PSKV_HIP(hipGetLastError());
    rc = launch_bounds_search(req_keys, n, h_targets, 2 * R, h_lb, c->stream);
    if (rc) return rc;
    PSKV_HIP(hipStreamSynchronize(c->stream));
    lease.idle = true;
    for (size_t r = 0; r < R; ++r) {  // kv_app.h:670-677
      const uint64_t lower = h_targets[2 * r], upper = h_targets[2 * r + 1];
      const uint64_t size = upper <= lower ? 0 : h_lb[2 * r + 1] - h_lb[2 * r];  // sarray.h:283
      if (size != resp_nkeys[r])
        return set_error(PSKV_ESIZE_MISMATCH, "unmatched keys size from one server (response %zu)", r);
      ends[2 * r] = lower;
    }
    if (total_key != n)  // kv_app.h:678
      return set_error(PSKV_ESIZE_MISMATCH, "lost some servers? %zu of %zu keys answered", total_key, n);
    if (out_nvals) *out_nvals = total_val;
    if (total_val > out_cap)  // kv_app.h:686-690
      return set_error(PSKV_ESIZE_MISMATCH, "response needs %zu floats, buffer holds %zu", total_val,
                       out_cap);
    std::vector<size_t> order(R);
    std::iota(order.begin(), order.end(), (size_t)0);
    std::sort(order.begin(), order.end(),  // kv_app.h:681-684
              [&](size_t x, size_t y) { return ends[2 * x] < ends[2 * y]; });
    // kv_app.h:701-708: one launch copies every slice to its place
    size_t voff = 0, koff = 0, nseg = 0;
    uint64_t longest = 0;
    for (size_t i = 0; i < R; ++i) {
      const size_t r = order[i];
      if (resp_nvals[r]) {
        h_segs[nseg++] = Segment{reinterpret_cast<const char*>(resp_vals[r]),
                                 reinterpret_cast<char*>(out + voff), resp_nvals[r] * sizeof(float)};
        longest = std::max<uint64_t>(longest, resp_nvals[r] * sizeof(float));
      }
      voff += resp_nvals[r];
      if (out_lens && resp_lens) {
        h_segs[nseg++] = Segment{reinterpret_cast<const char*>(resp_lens[r]),
                                 reinterpret_cast<char*>(out_lens + koff), resp_nkeys[r] * sizeof(int32_t)};
        longest = std::max<uint64_t>(longest, resp_nkeys[r] * sizeof(int32_t));
      }
      koff += resp_nkeys[r];
    }
    lease.idle = false;
    for (size_t first = 0; first < nseg; first += 65535) {  // gridDim.y holds 65535 segments
      const size_t now = std::min<size_t>(nseg - first, 65535);
      const uint64_t per = std::min<uint64_t>(longest / (16 * kBlock) + 1, 4096);
      k_concat<<<dim3((unsigned)per, (unsigned)now), dim3(kBlock), 0, c->stream>>>(h_segs + first);
      PSKV_HIP(hipGetLastError());
    }
    PSKV_HIP(hipStreamSynchronize(c->stream));
    lease.idle = true;
    return PSKV_OK;
  }
  if (total_key != n)
    return set_error(PSKV_ESIZE_MISMATCH, "lost some servers? %zu of %zu keys answered", total_key, n);
  return PSKV_OK;
}

}  // extern "C"

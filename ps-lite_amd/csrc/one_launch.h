// Requests of the row modes that are ONE launch: what a lookup kernel and a row kernel of table_kernels.h do one after the
// other. A small request is bound by its launches (2.2 us of the calling thread for each, and 3 to 5 us of the GPU's
// between dependent ones), not by what they do.
#ifndef PSKV_ONE_LAUNCH_H_
#define PSKV_ONE_LAUNCH_H_
#include "table_kernels.h"

namespace pskv {

// FIXED rows of up to kOwnQuads quads: a workgroup looks up as many consecutive keys as kOwnQuads quads hold (at most one
// a thread) and moves their rows; what it finds stays in LDS. A lane moves four quads: with one the lookups in front of
// a few rows are most of a workgroup's time (1M rows of 64 floats: 750 us for the three pulls and two pushes of a step
// against 645), with eight too few wavefronts fit (910).
// Pulls need nothing from each other, so there may be any number of workgroups.
// A push changes nothing before it is known that the request repeats no key: the workgroups hand in what they have
// found once their keys are looked up, ask for their rows, and the verdict is there by the time those are. They have
// to be on the GPU together for that: kOwnPushGroups of them are a third of what it holds. Who does not see the verdict
// in time all the same (d.cache_mode looks: something else may keep a part of the workgroups off the GPU) reads all
// keys of the request itself, so nobody depends on the others but for time.
// Measured (us per step of three pulls and two pushes, three tables in turn; lookup and rows as two launches -> one):
// 9,639 rows of 7 floats 37.2 -> 23.2, 59,871 of 16 36.4 -> 26.2, 30,000 of 64 43.3 -> 33.4; pulls alone as one launch:
// 193,521 rows of 30 126 -> 120, 1M of 64 663 -> 645.
constexpr unsigned kOwnTurns = 4;
constexpr unsigned kOwnQuads = kBlock * kOwnTurns;
constexpr uint64_t kOwnPushGroups = 512;
constexpr unsigned kOwnLooks = 1u << 10;  // (about half a millisecond)
// Keys per workgroup.
__host__ __device__ constexpr unsigned own_keys(uint64_t k) {
  const uint64_t keys = kOwnQuads / ((k + 3) / 4);
  return (unsigned)(keys < kBlock ? keys : kBlock);
}

__device__ __forceinline__ unsigned long long ask_verdict(const DevState* st) {
  return __hip_atomic_load(&st->push_verdict, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <bool PUSH, bool PULL, bool STREAM, int TABLES>
__global__ __launch_bounds__(kBlock) void k_fixed_own(ReqBatch<TABLES> b) {
  const TableReq& d = b.t[blockIdx.y];
  PSKV_ASK_ARGS("s"(d.slots), "s"(d.mask), "s"(d.st), "s"(d.keys), "s"(d.n), "s"(d.ref), "s"(d.cache_keys), "s"(d.vals),
                "s"(d.out), "s"(d.arena), "s"(d.k), "s"(d.snap), "s"(d.tag.epoch), "s"(d.cached), "s"(d.nblk));
  const unsigned nblk = d.nblk;
  if (blockIdx.x >= nblk) return;
  DevState* st = d.st;
  const uint64_t n = d.n, k = d.k;
  const ReqTag tag = d.tag;
  __shared__ unsigned long long red[kBlock / 64 + 1];
  __shared__ unsigned long long s_first;
  __shared__ uint64_t s_ref[kBlock];
  __shared__ unsigned s_verdict;
  unsigned long long before = 0;
  if (threadIdx.x == 0) {
    if (PUSH) before = ask_verdict(st);
    if (blockIdx.x == 0) st->cache_epoch = tag.epoch;
  }
  const unsigned quads = (unsigned)((k + 3) >> 2), rest = (unsigned)k & 3u;
  const unsigned share = own_keys(k);
  const uint64_t first = (uint64_t)blockIdx.x * share;
  const unsigned mine = n - first < share ? (unsigned)(n - first) : share;  // keys of this workgroup
  const bool live = threadIdx.x < mine;
  const uint64_t i = first + threadIdx.x;
  uint64_t key = 0, left = 0, cached_key = 0, was = kRefAbsent;
  if (live) {
    key = d.keys[i];
    left = d.keys[i ? i - 1 : 0];
    cached_key = d.cache_keys[i];
    was = d.ref[i];
  }
  // the values of the workgroup's quads, which lie one behind the other in the request
  const unsigned all = mine * quads;
  f32x4 x[kOwnTurns];
  unsigned row[kOwnTurns], col[kOwnTurns], count[kOwnTurns];
#pragma unroll
  for (unsigned q = 0; q < kOwnTurns; ++q) {
    const unsigned quad = q * kBlock + threadIdx.x;
    row[q] = quad / quads;
    const unsigned c = quad - row[q] * quads;
    col[q] = c * 4;
    count[q] = quad >= all ? 0u : rest && c + 1 == quads ? rest : 4u;
    x[q] = (f32x4)(0.f);
    if (PUSH && count[q]) {
      const float* side = d.vals + (first + row[q]) * k + col[q];
      // (a shorter quad is read whole where the next row follows it)
      x[q] = count[q] == 4 || first + row[q] + 1 < n ? load_quad<STREAM>(side) : load_part<STREAM>(side, count[q]);
    }
  }
  uint64_t* p = nullptr;
  uint64_t seen = 0;
  bool is_new = false, repeated = false, known = false;
  if (live) {
    // (as in k_lookup_fixed)
    if (i > 0 && left == key) {
      repeated = true;
      d.cache_keys[i] = key;
    } else if (i < d.cached && cached_key == key && was != kRefAbsent) {
      known = true;
    } else {
      d.cache_keys[i] = key;
      p = find_or_insert(d.slots, d.mask, st, key, is_new, seen);
      if (p && !is_new && seen == kPayloadUnset) {
        repeated = true;  // (unsorted request) another lane of this request is creating the very same key
        p = nullptr;
      }
    }
    if (repeated) refuse_fixed(st, tag);
  }
  if (!p) is_new = false;
  const bool any_repeated = __syncthreads_or(repeated ? 1 : 0) != 0;
  uint64_t r = known ? was & ~kRefNew : p ? seen : kRefAbsent;
  if (__syncthreads_or(is_new ? 1 : 0)) {
    unsigned long long total;
    const unsigned long long at = block_excl_scan_u64(is_new ? 1ull : 0ull, red, total);
    if (threadIdx.x == 0) {
      s_first = atomicAdd(&st->arena_top, total);
      atomicAdd(&st->count_shard[(blockIdx.x % kCountShards) * kShardStride], total);
    }
    __syncthreads();
    if (is_new) {
      *p = s_first + at;
      r = (s_first + at) | kRefNew;
    }
  }
  if (live) {
    s_ref[threadIdx.x] = r;
    if (r != was) d.ref[i] = r;
  }
  __syncthreads();
  // the rows
  f32x4 y[kOwnTurns];
  uint64_t ref[kOwnTurns];
#pragma unroll
  for (unsigned q = 0; q < kOwnTurns; ++q) {
    ref[q] = count[q] ? s_ref[row[q]] : kRefAbsent;
    y[q] = (f32x4)(0.f);
    // (a key that was refused has no row; a created row is zero)
    if (ref[q] != kRefAbsent && !(ref[q] & kRefNew)) y[q] = load_quad<STREAM>(d.arena + ref[q] * k + col[q]);
  }
  // (before anything is stored: the counter record goes past the caches and would wait for the rows)
  unsigned verdict = 2;  // not known yet
  if ((PUSH || d.snap) && threadIdx.x < 64) {
    unsigned last = 0;
    if (threadIdx.x == 0) {
      if (PUSH && any_repeated) report_facts(st, kReqDuplicate, nblk);
      asm volatile("" : "+v"(before) : : "memory");  // (the old verdict has to be here before the ticket goes out)
      last = ticket_last(st, nblk) ? 1u : 0u;
    }
    if (__shfl(last, 0)) {
      if (PUSH) {
        verdict = take_facts(st, nblk) & kReqDuplicate ? 1u : 0u;
        if (threadIdx.x == 0)
          __hip_atomic_store(&st->push_verdict, ((before >> 1) + 1) << 1 | verdict, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
      }
      if (d.snap) publish_snapshot(st, d.snap, d.snap_seq);
    } else if (PUSH && threadIdx.x == 0) {
      for (unsigned looks = d.cache_mode; looks && verdict == 2; --looks) {
        const unsigned long long now = ask_verdict(st);
        if (now != before) verdict = (unsigned)now & 1u; else __builtin_amdgcn_s_sleep(1);
      }
    }
    if (threadIdx.x == 0) s_verdict = verdict;
  }
  bool rejected = false;
  if (PUSH) {
    __syncthreads();
    verdict = s_verdict;
    if (verdict == 2) {
      bool any = false;
      for (uint64_t at = 1 + threadIdx.x; at < n; at += kBlock) any |= d.keys[at] == d.keys[at - 1];
      verdict = __syncthreads_or(any ? 1 : 0) ? 1u : 0u;
    }
    rejected = verdict != 0;
  }
#pragma unroll
  for (unsigned q = 0; q < kOwnTurns; ++q) {
    if (ref[q] == kRefAbsent) continue;
    const bool fresh = (ref[q] & kRefNew) != 0;
    // a refused push changes no stored value; rows it created stay, as zero rows
    if (PUSH && !rejected) y[q] = y[q] + x[q];  // a created row is a zero row first (0.0f + v), kv_app.h:454
    if (fresh || (PUSH && !rejected)) store_part<STREAM>(y[q], d.arena + (ref[q] & ~kRefNew) * k + col[q], count[q]);
    if (PULL) store_part<STREAM>(y[q], d.out + (first + row[q]) * k + col[q], count[q]);
  }
}

}  // namespace pskv
#endif  // PSKV_ONE_LAUNCH_H_

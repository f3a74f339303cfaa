// Requests of the row modes in fewer launches: what kernels of table_kernels.h do one after the other in one. A small
// request is bound by its launches (2.2 us of the calling thread for each, and 3 to 5 us of the GPU's between dependent
// ones), not by what they do.
#ifndef PSKV_ONE_LAUNCH_H_
#define PSKV_ONE_LAUNCH_H_
#include "handover.h"
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
// in time all the same (d.cache_mode looks: something else may keep a part of the workgroups off the GPU) leaves its rows to
// the workgroup that reaches the verdict (handover.h), so nobody depends on the others but for time, and there is one
// verdict for the whole request, whatever it rests on: that a new key comes twice in a request that is not sorted only those
// notice who claim its slot. (Shares that are left take some 10 us each.)
// Measured (us per two steps of pull and push and a pull, lookup and rows as two launches -> one): 49,881 rows of 15 floats
// one table 49-53 -> 40, three in turn 28-39 -> 20.4; 30,000 of 64 53-59 -> 41, 37-45 -> 30.6; 1M of 64, whose pushes are two
// launches, 668 -> 633, 643 -> 633. Of that the loads of a lane's rows side by side, the ticket in front of them and its
// fence without a write-back are 45.6 -> 40, 24 -> 20.4 and 48.8 -> 41, 33.2 -> 30.6.
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

// The memory of leave_share.
struct ShareMem {
  DevState* st;
  __device__ unsigned long long* word() { return &st->shares_left[blockIdx.x / 64]; }
  __device__ unsigned long long bit() { return 1ull << (blockIdx.x % 64); }
  __device__ void mark() {
    unsigned long long was = atomicOr(word(), bit());
    asm volatile("" : "+v"(was) : : "memory");  // (it is there before anything that follows)
  }
  __device__ bool unmark() { return (atomicAnd(word(), ~bit()) & bit()) != 0; }
  __device__ unsigned long long swap(unsigned long long from, unsigned long long to) {
    unsigned long long was = atomicCAS(&st->push_verdict, from, to);
    asm volatile("" : "+v"(was) : : "memory");
    return was;
  }
};
static_assert(kOwnPushGroups == 64 * (sizeof(DevState::shares_left) / 8), "a bit for every workgroup of a push");

// The rows of the workgroups that have left theirs to this one. Every thread calls it.
template <bool PULL, bool STREAM>
__device__ __forceinline__ void serve_shares_left(const TableReq& d, bool rejected) {
  __shared__ unsigned long long s_left;
  const unsigned quads = (unsigned)((d.k + 3) >> 2), rest = (unsigned)d.k & 3u, share = own_keys(d.k);
  for (unsigned w = 0; w * 64 < d.nblk; ++w) {
    __syncthreads();
    if (threadIdx.x == 0) s_left = atomicExch(&d.st->shares_left[w], 0ull);
    __syncthreads();
    __threadfence();  // nothing stale is left of what those workgroups have written in front of their marks
    for (unsigned long long left = s_left; left; left &= left - 1) {
      const uint64_t first = ((uint64_t)w * 64 + __builtin_ctzll(left)) * share;
      const unsigned mine = d.n - first < share ? (unsigned)(d.n - first) : share;
      for (unsigned quad = threadIdx.x; quad < mine * quads; quad += kBlock) {
        const unsigned row = quad / quads, c = quad - row * quads, col = c * 4, count = rest && c + 1 == quads ? rest : 4u;
        const uint64_t ref = d.ref[first + row];
        if (ref == kRefAbsent) continue;
        const bool fresh = (ref & kRefNew) != 0;
        float* const at = d.arena + (ref & ~kRefNew) * d.k + col;
        f32x4 y = (f32x4)(0.f);
        if (!fresh) y = load_part<STREAM>(at, count);
        if (!rejected) y = y + load_part<STREAM>(d.vals + (first + row) * d.k + col, count);
        if (fresh || !rejected) store_part<STREAM>(y, at, count);
        if (PULL) store_part<STREAM>(y, d.out + (first + row) * d.k + col, count);
      }
    }
  }
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
  // (a lane behind the end takes the last one and does not store it: a load under a condition is waited for before the next
  // is asked for)
  f32x4 x[kOwnTurns];
  unsigned row[kOwnTurns], col[kOwnTurns], count[kOwnTurns];
#pragma unroll
  for (unsigned q = 0; q < kOwnTurns; ++q) {
    const unsigned quad = q * kBlock + threadIdx.x, there = quad < all ? quad : all - 1;
    row[q] = there / quads;
    const unsigned c = there - row[q] * quads;
    col[q] = c * 4;
    count[q] = quad >= all ? 0u : rest && c + 1 == quads ? rest : 4u;
    x[q] = (f32x4)(0.f);
  }
  if (PUSH && whole_quads(first + mine, k, n)) {  // a shorter quad is read whole where rows enough follow it
#pragma unroll
    for (unsigned q = 0; q < kOwnTurns; ++q) x[q] = load_quad<STREAM>(d.vals + (first + row[q]) * k + col[q]);
  } else if (PUSH) {
#pragma unroll
    for (unsigned q = 0; q < kOwnTurns; ++q)
      if (count[q]) x[q] = load_part<STREAM>(d.vals + (first + row[q]) * k + col[q], count[q]);
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
    if (threadIdx.x == 0) my_atomics_are_there();
  }
  if (live) {
    s_ref[threadIdx.x] = r;
    if (r != was) d.ref[i] = r;
  }
  __syncthreads();
  // The ticket goes out in front of the loads of the rows: behind them it would wait for them.
  unsigned ticket = 0;
  if ((PUSH || d.snap) && threadIdx.x == 0) {
    if (PUSH && any_repeated) {
      report_facts(st, kReqDuplicate, nblk);
      my_atomics_are_there();
    }
    asm volatile("" : "+v"(before) : : "memory");  // (the old verdict has to be here before the ticket goes out)
    ticket = ticket_take(st, nblk);
  }
  // the rows
  f32x4 y[kOwnTurns];
  uint64_t ref[kOwnTurns];
#pragma unroll
  for (unsigned q = 0; q < kOwnTurns; ++q) {
    ref[q] = count[q] ? s_ref[row[q]] : kRefAbsent;
    // (a key that was refused has no row, a created row is zero: read is the table's first one then)
    y[q] = load_quad<STREAM>(d.arena + (ref[q] & kRefNew ? 0 : ref[q]) * k + col[q]);
  }
#pragma unroll
  for (unsigned q = 0; q < kOwnTurns; ++q)
    if (ref[q] & kRefNew) y[q] = (f32x4)(0.f);
  // (before anything is stored: the counter record goes past the caches and would wait for the rows)
  constexpr unsigned kUnknown = 2, kIsLast = 4;
  unsigned verdict = kUnknown;
  // The last workgroup: what the word of the verdict was in front of its own. (Nobody waits for it in front of the rows: it
  // has no other value, and it is looked at behind them. With a wait small pushes took 0.35 us of 11 longer.)
  unsigned long long exchanged;
  asm volatile("" : "=v"(exchanged));
  if ((PUSH || d.snap) && threadIdx.x < 64) {
    unsigned last = 0;
    if (threadIdx.x == 0) last = ticket_is_last(st, nblk, ticket) ? 1u : 0u;
    if (__shfl(last, 0)) {
      if (PUSH) {
        verdict = (take_facts(st, nblk) & kReqDuplicate ? 1u : 0u) | kIsLast;
        if (threadIdx.x == 0) exchanged = atomicExch(&st->push_verdict, next_verdict(before, verdict & 1u));
      }
      if (d.snap) publish_snapshot(st, d.snap, d.snap_seq);
    } else if (PUSH && threadIdx.x == 0) {
      for (unsigned looks = d.cache_mode; looks && verdict == kUnknown; --looks) {
        const unsigned long long now = ask_verdict(st);
        if (has_verdict(now, before)) verdict = (unsigned)(now & kVerdictYes); else __builtin_amdgcn_s_sleep(1);
      }
    }
    if (threadIdx.x == 0) s_verdict = verdict;
  }
  bool rejected = false;
  if (PUSH) {
    __syncthreads();
    verdict = s_verdict;
    if (verdict == kUnknown) {
      __threadfence();  // the rows of its keys are there for whoever moves them
      __syncthreads();
      if (threadIdx.x == 0) {
        ShareMem m{st};
        const int late = leave_share(m, before);
        s_verdict = late < 0 ? kUnknown : (unsigned)late;
      }
      __syncthreads();
      verdict = s_verdict;
      if (verdict == kUnknown) return;
    }
    rejected = (verdict & 1u) != 0;
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
  if (PUSH && (verdict & kIsLast)) {
    __syncthreads();
    asm volatile("" : "+v"(exchanged));
    if (threadIdx.x == 0) s_verdict = exchanged & kSharesLeft ? 1u : 0u;
    __syncthreads();
    if (s_verdict) serve_shares_left<PULL, STREAM>(d, rejected);
  }
}

// FIXED rows of more than kOwnQuads quads: a workgroup moves an even part of one row, up to kOwnQuads quads, and every
// workgroup of a row looks up the row's key, so nobody waits for the others' lookups. Whoever claims the slot of a new key
// gives it its row; the others find the key and wait for its payload, which follows from nothing but the claim. That the
// row is new they can see from DevState::fresh_from: before the first creator of a request counts the rows up it notes
// there, under the number of the request, how many there were, so every row from there on is new to this request. (Number
// and rows are one word: 2^26 rows of 4,100 floats are four times what the GPU holds, 2^38 requests years.)
// Whether a request repeats a key every workgroup sees for itself: there are at most as many keys as threads.
// Bound by the chain from a key to its slot, from there to the row, and back. Up to kLongFloats floats that is better than
// the two launches of lookup and rows (us per push + pull, one table; three in turn, of which the launches are most:
// 5,000 floats 19.6 -> 18.7; 12.7-15 -> 8.1-9.5, 43 rows of 36,505 27 -> 22; 12.4-15.9 -> 9.3, 200 of 10,000 28 -> 23;
// 12.4-15.5 -> 11.1, and per four pushes + pull 40 of 100,000 92 -> 71; 71 -> 61). Beyond it other requests' rows fill the
// gap in front of theirs, and workgroups that ask for less before their rows stream faster (three pushes + pull of 8 rows
// of 960,704 100 -> 82; 73 -> 81). Quads a lane: 4, with 2 30 rows of 262,144 38 -> 41, with 1 47; past the caches 42.
constexpr uint64_t kLongFloats = 1u << 22;
constexpr uint64_t kLongKeys = kBlock;
constexpr unsigned kFreshBits = 26;
constexpr unsigned kLongLooks = 1u << 16;  // (nobody gets that far: a claimed slot has its row some 2 us later)
__host__ __device__ constexpr unsigned long_groups(uint64_t k) { return (unsigned)(((k + 3) / 4 + kOwnQuads - 1) / kOwnQuads); }

// The row of `key`, with kRefNew if this call has created it. One thread.
__device__ __forceinline__ uint64_t find_or_make_row(const TableReq& d, uint64_t key) {
  DevState* st = d.st;
  bool is_new;
  uint64_t seen;
  uint64_t* p = find_or_insert(d.slots, d.mask, st, key, is_new, seen);
  if (!p) return kRefAbsent;
  if (!is_new) {
    for (unsigned looks = kLongLooks; seen == kPayloadUnset && looks; --looks)
      seen = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (seen != kPayloadUnset) return seen;
    refuse_fixed(st, d.tag);
    return kRefAbsent;
  }
  const unsigned long long word = __hip_atomic_load(&st->fresh_from, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (word >> kFreshBits != d.tag.epoch) {
    // (as long as the word can be exchanged, nobody has counted up)
    const unsigned long long rows = __hip_atomic_load(&st->arena_top, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    unsigned long long was = atomicCAS(&st->fresh_from, word, (unsigned long long)d.tag.epoch << kFreshBits | rows);
    asm volatile("" : "+v"(was) : : "memory");  // (it is there before the count changes)
  }
  const unsigned long long row = atomicAdd(&st->arena_top, 1ull);
  atomicAdd(&st->count_shard[(blockIdx.x % kCountShards) * kShardStride], 1ull);
  __hip_atomic_store(p, row, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  my_atomics_are_there();
  return row | kRefNew;
}

template <bool PUSH, bool PULL, int TABLES>
__global__ __launch_bounds__(kBlock) void k_fixed_long(ReqBatch<TABLES> b) {
  const TableReq& d = b.t[blockIdx.y];
  PSKV_ASK_ARGS("s"(d.slots), "s"(d.mask), "s"(d.st), "s"(d.keys), "s"(d.n), "s"(d.ref), "s"(d.cache_keys), "s"(d.vals),
                "s"(d.out), "s"(d.arena), "s"(d.k), "s"(d.snap), "s"(d.tag.epoch), "s"(d.nblk));
  const unsigned nblk = d.nblk;
  if (blockIdx.x >= nblk) return;
  DevState* st = d.st;
  const uint64_t k = d.k;
  const unsigned n = (unsigned)d.n;
  __shared__ uint64_t s_ref;
  const unsigned quads = (unsigned)((k + 3) >> 2), rest = (unsigned)k & 3u;
  const unsigned per = long_groups(k), i = blockIdx.x / per, part = blockIdx.x - i * per;
  const uint64_t key = d.keys[i], left = d.keys[i ? i - 1 : 0];
  // whole quads, four a lane, and the rest of the row, which is one lane's (a case of its own: with the rest as a case of
  // every quad the code was half as long again, and a small request reads all of it for the first time)
  const unsigned wholes = quads - (rest ? 1u : 0u), share = (quads + per - 1) / per, c0 = part * share + threadIdx.x;
  const unsigned end = (part + 1) * share < wholes ? (part + 1) * share : wholes;
  const bool tail = rest && part + 1 == per && threadIdx.x == kBlock - 1;
  // (a lane behind the end moves the last whole quad, and does not store it: a load under a condition is waited for)
  unsigned at[kOwnTurns];
#pragma unroll
  for (unsigned q = 0; q < kOwnTurns; ++q) at[q] = (c0 + q * kBlock < end ? c0 + q * kBlock : end - 1) * 4;
  const float* side = d.vals + i * k;
  f32x4 x[kOwnTurns], x_tail = (f32x4)(0.f);
  if (PUSH) {
#pragma unroll
    for (unsigned q = 0; q < kOwnTurns; ++q) x[q] = load_quad<false>(side + at[q]);
    if (tail) x_tail = load_part<false>(side + wholes * 4, rest);
  }
  bool repeated = false, twice = false, unsorted = false;
  uint64_t r = kRefAbsent;
  if (threadIdx.x == 0) {
    if (blockIdx.x == 0) st->cache_epoch = d.tag.epoch;
    repeated = i > 0 && left == key;
    if (!repeated) r = find_or_make_row(d, key);
    s_ref = r;
  }
  if (threadIdx.x && threadIdx.x < n) {
    const uint64_t a = d.keys[threadIdx.x - 1], c = d.keys[threadIdx.x];
    twice = a == c;
    unsorted = a > c;
  }
  bool rejected = __syncthreads_or(twice ? 1 : 0) != 0;  // (s_ref is there)
  bool again = false;
  if (__syncthreads_or(unsorted ? 1 : 0)) {  // (then a key may be anywhere again)
    const unsigned j = threadIdx.x;
    again = j < n && j != i && d.keys[j] == key;
    for (unsigned l = 0; PUSH && j < n && l < j; ++l) twice |= d.keys[l] == d.keys[j];
    again = __syncthreads_or(again ? 1 : 0) != 0;
    rejected = __syncthreads_or(twice ? 1 : 0) != 0;
  }
  unsigned ticket = 0;  // (in front of the loads of the row, see k_fixed_own)
  if (d.snap && threadIdx.x == 0) ticket = ticket_take(st, nblk);
  r = s_ref;
  const uint64_t row = r & ~kRefNew;
  float* const base = d.arena + (r != kRefAbsent ? row : 0) * k;  // (a refused key reads the table's first row)
  f32x4 y[kOwnTurns], y_tail = (f32x4)(0.f);
#pragma unroll
  for (unsigned q = 0; q < kOwnTurns; ++q) y[q] = load_quad<false>(base + at[q]);
  if (tail) y_tail = load_part<false>(base + wholes * 4, rest);
  // (behind the row's number, which its creator leaves behind this word; the row is on its way meanwhile)
  const unsigned long long word = __hip_atomic_load(&st->fresh_from, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const bool fresh = r != kRefAbsent && word >> kFreshBits == d.tag.epoch && row >= (word & ((1ull << kFreshBits) - 1));
  if (threadIdx.x == 0 && part == 0) {
    // (a pull is served from the rows that are there however often a key comes; none is created twice)
    if (repeated || (PUSH ? rejected && again : fresh && again)) refuse_fixed(st, d.tag);
    d.cache_keys[i] = key;
    d.ref[i] = fresh ? row | kRefNew : r;
  }
  if (d.snap && threadIdx.x < 64) {
    unsigned last = 0;
    if (threadIdx.x == 0) last = ticket_is_last(st, nblk, ticket) ? 1u : 0u;
    if (__shfl(last, 0)) publish_snapshot(st, d.snap, d.snap_seq);
  }
  if (r == kRefAbsent) return;
  // a refused push changes no stored value; rows it created stay, as zero rows
  const bool add = PUSH && !rejected, keep = fresh || add;
  float* const out = PULL ? d.out + i * k : nullptr;
#pragma unroll
  for (unsigned q = 0; q < kOwnTurns; ++q) {
    if (c0 + q * kBlock >= end) continue;
    if (fresh) y[q] = (f32x4)(0.f);
    if (add) y[q] = y[q] + x[q];  // a created row is a zero row first (0.0f + v), kv_app.h:454
    if (keep) store_quad<false>(y[q], base + at[q]);
    if (PULL) store_quad<false>(y[q], out + at[q]);
  }
  if (!tail) return;
  if (fresh) y_tail = (f32x4)(0.f);
  if (add) y_tail = y_tail + x_tail;
  if (keep) store_part<false>(y_tail, base + wholes * 4, rest);
  if (PULL) store_part<false>(y_tail, out + wholes * 4, rest);
}

// VARLEN requests of up to kVarParts workgroups: what the first two kernels of a push, or of a pull, do, in one. A
// workgroup takes kStartPart consecutive keys, two a thread, and keeps them in registers. What it has to know of the
// others (where its rows start in the request, what is the matter with any key or length) it reads off one word of
// each, which it watches until all of them are there: no election, no scan by one for all (with those, and the outcome in
// a word for everyone, 15,826 rows over 3 tables took 14.8 us to start a push, now 8.6; begin + lookup 6.7 + 7.2 and the
// launch between them). With four keys a thread it was the walks of a wavefront's keys one after the other, 13.4. The
// workgroups have to be on the GPU together, and kVarParts of them are a fifth of what it holds; who does not see all
// words in time (d.cache_mode looks: something else may keep a part of the workgroups off the GPU) goes through the
// request itself, so nobody depends on the others but for time.
// The row kernel behind it takes the words away again, and leaves the counter record of a push (finish_start).
// Measured (us per step of slice, push and pull, other rows in every step, three tables in turn): 10,562 rows of 8 to 128
// floats over 4 tables 36.3 -> 35.5, 15,826 of 1 to 90 over 3 42.2 -> 38.6, 50,000 of 8 to 64 over 4 43.9 -> 38.6.
constexpr int kStartItems = 2;
constexpr uint64_t kStartPart = (uint64_t)kBlock * kStartItems;
inline uint64_t start_parts(uint64_t n) { return (n + kStartPart - 1) / kStartPart; }
constexpr unsigned long long kPartHere = 1ull << 63;
constexpr unsigned kPartFlagsAt = 40;  // (512 lengths below 2^28 add up to less)
static_assert(kStartPart <= 1u << 10 && PSKV_MAX_VARLEN_ROW < (1u << 28), "a part's total fits below its flags");

struct OfAllParts {
  unsigned long long before, all;  // floats in front of this workgroup's part, and in the request
  unsigned flags;                  // kReq*
  bool known;
};
struct PartRed {
  unsigned long long before[kBlock / 64], all[kBlock / 64];
  unsigned flags[kBlock / 64];
};
__device__ __forceinline__ void reduce_parts(OfAllParts& x, PartRed* red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    x.before += __shfl_xor(x.before, o);
    x.all += __shfl_xor(x.all, o);
    x.flags |= __shfl_xor(x.flags, o);
  }
  const unsigned wave = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red->before[wave] = x.before, red->all[wave] = x.all, red->flags[wave] = x.flags;
  __syncthreads();
  x.before = x.all = 0, x.flags = 0;
#pragma unroll
  for (unsigned w = 0; w < kBlock / 64; ++w) x.before += red->before[w], x.all += red->all[w], x.flags |= red->flags[w];
}
// Every thread of the workgroup calls it with its own floats and flags.
__device__ __forceinline__ OfAllParts meet_parts(DevState* st, unsigned nblk, unsigned long long floats, unsigned flags,
                                                 unsigned looks, PartRed* red) {
  OfAllParts mine{0, floats, flags, true};
  reduce_parts(mine, red);
  if (threadIdx.x == 0)
    publish_u64(&st->parts[blockIdx.x], kPartHere | (unsigned long long)mine.flags << kPartFlagsAt |
                                            (mine.flags & kReqBadLen ? 0ull : mine.all));
  OfAllParts x{0, 0, 0, true};
#pragma unroll
  for (unsigned q = 0; q < kVarParts / kBlock; ++q) {
    const unsigned i = q * kBlock + threadIdx.x;
    if (i >= nblk) continue;
    unsigned long long w = 0;
    for (unsigned look = looks;; --look) {
      w = __hip_atomic_load(&st->parts[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if ((w & kPartHere) || !look) break;
      __builtin_amdgcn_s_sleep(1);
    }
    const unsigned long long sum = w & ((1ull << kPartFlagsAt) - 1);
    x.known = x.known && (w & kPartHere) != 0;
    x.all += sum;
    if (i < blockIdx.x) x.before += sum;
    x.flags |= (unsigned)(w >> kPartFlagsAt) & 63u;
  }
  x.known = __syncthreads_and(x.known ? 1 : 0) != 0;
  if (x.known) reduce_parts(x, red);
  return x;
}
static_assert(kReqLong == 32u && (kReqMisaligned | kReqBadLen | kReqDiffer | kReqDuplicate) == 31u, "six bits of flags");

typedef int32_t i32x2u __attribute__((ext_vector_type(2), aligned(4)));
struct TwoKeys {
  uint64_t k[kStartItems];
  int32_t v[kStartItems];
};
__device__ __forceinline__ void load_two(TwoKeys& f, const uint64_t* keys, const int32_t* lens, uint64_t at, uint64_t n) {
  static_assert(kStartItems == 2, "two keys per thread");
  if (at + 2 <= n) {
    const u64x2u a = *reinterpret_cast<const u64x2u*>(keys + at);
    const i32x2u w = *reinterpret_cast<const i32x2u*>(lens + at);
    f.k[0] = a.x, f.k[1] = a.y, f.v[0] = w.x, f.v[1] = w.y;
  } else {
    f.k[0] = at < n ? keys[at] : 0, f.v[0] = at < n ? lens[at] : 0;
    f.k[1] = 0, f.v[1] = 0;
  }
}

template <int TABLES>
__global__ __launch_bounds__(kBlock) void k_var_push_start(ReqBatch<TABLES> b) {
  const TableReq& d = b.t[blockIdx.y];
  PSKV_ASK_ARGS("s"(d.slots), "s"(d.mask), "s"(d.st), "s"(d.keys), "s"(d.lens), "s"(d.n), "s"(d.nvals), "s"(d.ref),
                "s"(d.off), "s"(d.tile_key), "s"(d.ntiles), "s"(d.cache_keys), "s"(d.cache_lens), "s"(d.tag.epoch),
                "s"(d.nblk), "s"(d.ragged));
  const unsigned nblk = d.nblk;
  if (blockIdx.x >= nblk) return;
  DevState* st = d.st;
  const uint64_t n = d.n;
  constexpr unsigned max_len = PSKV_MAX_VARLEN_ROW;
  const unsigned longest = longest_by_row(d);
  __shared__ PartRed red;
  __shared__ unsigned long long wsum[kBlock / 64 + 1];
  __shared__ unsigned cred[kBlock / 64];
  __shared__ unsigned long long s_start;
  const uint64_t base = ((uint64_t)blockIdx.x * kBlock + threadIdx.x) * kStartItems;
  TwoKeys mine;
  load_two(mine, d.keys, d.lens, base, n);
  const uint64_t left = (base > 0 && base < n) ? d.keys[base - 1] : 0;
  // The keys' home slots are on the way while the workgroups wait (an empty slot that has been taken since shows when it
  // is claimed).
  u64x2 home[kStartItems];
#pragma unroll
  for (int j = 0; j < kStartItems; ++j) home[j] = load_slot(&d.slots[home_slot(mine.k[j], d.mask)]);
  unsigned long long len[kStartItems], s = 0;
  unsigned flags = 0;
#pragma unroll
  for (int j = 0; j < kStartItems; ++j) {  // (as in k_var_push_begin)
    const int32_t l = mine.v[j];
    len[j] = (unsigned long long)(uint32_t)l;
    s += len[j];
    flags |= (unsigned)l & kReqMisaligned;
    flags |= (unsigned)l > longest ? kReqLong : 0u;
    flags |= (l < 0 || (unsigned)l > max_len) ? kReqBadLen : 0u;
    const bool has_left = base + j < n && base + j > 0;
    flags |= (has_left && mine.k[j] == (j ? mine.k[j - 1] : left)) ? kReqDuplicate : 0u;
  }
  OfAllParts of = meet_parts(st, nblk, s, flags, d.cache_mode, &red);
  if (!of.known) {
    of = OfAllParts{0, 0, 0, true};
    for (uint64_t i = threadIdx.x; i < n; i += kBlock) {
      const int32_t l = d.lens[i];
      of.all += (unsigned long long)(uint32_t)l;
      if (i < (uint64_t)blockIdx.x * kStartPart) of.before += (unsigned long long)(uint32_t)l;
      of.flags |= (unsigned)l & kReqMisaligned;
      of.flags |= (unsigned)l > longest ? kReqLong : 0u;
      of.flags |= (l < 0 || (unsigned)l > max_len) ? kReqBadLen : 0u;
      of.flags |= i > 0 && d.keys[i] == d.keys[i - 1] ? kReqDuplicate : 0u;
    }
    reduce_parts(of, &red);
  }
  const unsigned refused = (of.flags & kReqBadLen ? kDevErrBadLen : 0u) | (of.flags & kReqDuplicate ? kDevErrDuplicate : 0u);
  const unsigned bad = refused ? refused : of.all != d.nvals ? kDevErrSizeMismatch : 0u;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    // what k_var_push_begin's last workgroup leaves of a request that does not repeat the cached one
    if (st->req_error) atomicOr(&st->error, st->req_error);
    st->req_error = bad;
    st->scan_total = of.all;
    st->misaligned = of.flags & (kReqMisaligned | kReqLong);
    st->cache_epoch = d.tag.epoch;
    if (bad) st->bad_epoch = d.tag.epoch;
    tell_ragged(st, d.outcome, of.flags);
  }
  if (bad) return;  // nothing is created
  scan_pass2_offsets<kStartItems>(len, base, n, of.before, d.off, d.tile_key, d.ntiles, kTileVar, wsum);
  uint64_t* p[kStartItems];
  uint64_t seen[kStartItems];
  bool is_new[kStartItems], live[kStartItems];
  unsigned long long units = 0;
  unsigned created = 0;
#pragma unroll
  for (int j = 0; j < kStartItems; ++j) live[j] = base + j < n;
  find_or_insert_all<kStartItems>(d.slots, d.mask, st, mine.k, home, live, p, is_new, seen);
#pragma unroll
  for (int j = 0; j < kStartItems; ++j) {
    const uint64_t i = base + j;
    if (live[j]) {
      d.cache_keys[i] = mine.k[j];
      d.cache_lens[i] = mine.v[j];
      if (p[j] && !is_new[j] && seen[j] == kPayloadUnset) {
        atomicOr(&st->error, kDevErrDuplicate);  // the same key twice in this request
        st->bad_epoch = d.tag.epoch;
        p[j] = nullptr;
      }
    }
    if (p[j] && is_new[j]) {
      units += (len[j] + 3) >> 2;
      ++created;
    }
  }
  if (__syncthreads_or(created ? 1 : 0)) {
    unsigned long long total;
    unsigned long long at = block_excl_scan_u64(units, wsum, total);
    if (threadIdx.x == 0) {
      // (the rows of the part start where the request's do, modulo 128 bytes: see k_var_push_lookup)
      const unsigned long long first = atomicAdd(&st->arena_top, total + (kArenaPadUnits - 1));
      const unsigned long long want = (of.before >> 2) & (kArenaPadUnits - 1);
      s_start = first + ((want - first) & (kArenaPadUnits - 1));
    }
    __syncthreads();
    at += s_start;
#pragma unroll
    for (int j = 0; j < kStartItems; ++j) {
      if (!p[j] || !is_new[j]) continue;
      seen[j] = ((uint64_t)at << kLenBits) | len[j];
      at += (len[j] + 3) >> 2;
      *p[j] = seen[j];
    }
    block_count_add(st, created, cred);
  }
#pragma unroll
  for (int j = 0; j < kStartItems; ++j) {
    const uint64_t i = base + j;
    if (i >= n) continue;
    if (!p[j]) {
      d.ref[i] = kRefAbsent;
      continue;
    }
    if (!is_new[j] && (seen[j] & kLenMask) != len[j]) {
      atomicOr(&st->error, kDevErrLenChanged);
      st->bad_epoch = d.tag.epoch;
      st->refused_epoch = d.tag.epoch;  // (req_error is the first workgroup's, which may be behind this one)
    }
    d.ref[i] = seen[j] | (is_new[j] ? kRefNew : 0ull);
  }
}

// VARLEN pull: k_var_pull_lookup and k_var_offsets in one. d.ntiles: room in the tile table.
template <int TABLES>
__global__ __launch_bounds__(kBlock) void k_var_pull_start(ReqBatch<TABLES> b) {
  const TableReq& d = b.t[blockIdx.y];
  PSKV_ASK_ARGS("s"(d.slots), "s"(d.mask), "s"(d.st), "s"(d.keys), "s"(d.n), "s"(d.ref), "s"(d.off), "s"(d.tile_key),
                "s"(d.ntiles), "s"(d.cache_keys), "s"(d.cache_lens), "s"(d.out_lens), "s"(d.tag.epoch), "s"(d.nblk));
  const unsigned nblk = d.nblk;
  if (blockIdx.x >= nblk) return;
  DevState* st = d.st;
  const uint64_t n = d.n;
  const ReqTag tag = d.tag;
  __shared__ PartRed red;
  __shared__ unsigned long long wsum[kBlock / 64];
  const uint64_t base = ((uint64_t)blockIdx.x * kBlock + threadIdx.x) * kStartItems;
  // (the first workgroup alone changes what this reads, after every workgroup has handed in its word; one that has not
  // seen the words may read it late, and looks up its keys)
  const bool usable = cache_usable(st, tag);
  uint64_t key[kStartItems];
  TwoKeys old;
  bool known[kStartItems];
  uint64_t payload[kStartItems];
  int32_t l[kStartItems];
  if (base + kStartItems <= n) {
    const u64x2u a = *reinterpret_cast<const u64x2u*>(d.keys + base);
    key[0] = a.x, key[1] = a.y;
  } else {
#pragma unroll
    for (int j = 0; j < kStartItems; ++j) key[j] = base + j < n ? d.keys[base + j] : 0;
  }
  if (usable) load_two(old, d.cache_keys, d.cache_lens, base, n);
  unsigned flags = 0;
#pragma unroll
  for (int j = 0; j < kStartItems; ++j) {
    known[j] = base + j >= n || (usable && old.k[j] == key[j]);
    l[j] = known[j] && base + j < n ? old.v[j] : 0;
    if (!known[j]) flags = kReqDiffer;
  }
  if (flags) {
    u64x2 home[kStartItems];
#pragma unroll
    for (int j = 0; j < kStartItems; ++j)
      if (!known[j]) home[j] = load_slot(&d.slots[home_slot(key[j], d.mask)]);
#pragma unroll
    for (int j = 0; j < kStartItems; ++j) {
      if (known[j]) continue;
      bool hit = home[j].x == key[j] && key[j] != kEmptyKey;
      payload[j] = home[j].y;
      if (!hit) hit = find_only(d.slots, d.mask, st, key[j], payload[j]);
      l[j] = hit ? (int32_t)(payload[j] & kLenMask) : 0;
      d.ref[base + j] = hit ? payload[j] : kRefAbsent;
    }
  }
  unsigned long long len[kStartItems], s = 0;
#pragma unroll
  for (int j = 0; j < kStartItems; ++j) {
    len[j] = (unsigned long long)(uint32_t)l[j];
    s += len[j];
    flags |= (unsigned)l[j] & kReqMisaligned;
  }
  if (base + kStartItems <= n) {
    i32x2u w;
    w.x = l[0], w.y = l[1];
    *reinterpret_cast<i32x2u*>(d.out_lens + base) = w;
  } else {
#pragma unroll
    for (int j = 0; j < kStartItems; ++j)
      if (base + j < n) d.out_lens[base + j] = l[j];
  }
  OfAllParts of = meet_parts(st, nblk, s, flags, d.cache_mode, &red);
  if (!of.known) {
    of = OfAllParts{0, 0, kReqDiffer, true};
    for (uint64_t i = threadIdx.x; i < n; i += kBlock) {
      uint64_t r = 0;
      const unsigned x = find_only(d.slots, d.mask, st, d.keys[i], r) ? (unsigned)(r & kLenMask) : 0u;
      of.all += x;
      if (i < (uint64_t)blockIdx.x * kStartPart) of.before += x;
      of.flags |= x & kReqMisaligned;
    }
    reduce_parts(of, &red);
  }
  const bool same = !(of.flags & kReqDiffer) && usable;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    // what k_var_pull_lookup's last workgroup leaves
    if (st->req_error) atomicOr(&st->error, st->req_error);
    st->req_error = 0;
    st->misaligned = of.flags & kReqMisaligned;
    if (same) {
      st->same_epoch = tag.epoch;
    } else {
      st->scan_total = of.all;
      // this pull rewrites references and offsets in the workspace: the cached push is gone
      st->bad_epoch = st->cache_epoch;
    }
    if (d.outcome && tag.try_cache) *d.outcome = (tag.epoch << 1) | (same ? 1ull : 0ull);
  }
  if (same) return;  // offsets and tile table of the cached request hold
  uint64_t ntiles = (of.all + kTileVar - 1) / kTileVar;
  if (ntiles > d.ntiles) ntiles = d.ntiles;
  scan_pass2_offsets<kStartItems>(len, base, n, of.before, d.off, d.tile_key, ntiles, kTileVar, wsum);
}

}  // namespace pskv
#endif  // PSKV_ONE_LAUNCH_H_

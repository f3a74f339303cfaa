// Shared device-side definitions of the pskv library (gfx950 only).
#ifndef PSKV_DEVICE_COMMON_H_
#define PSKV_DEVICE_COMMON_H_
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "start_rule.h"

// Asks for all of a kernel's arguments at once (the compiler otherwise fetches them group by group where they are first
// used, one wait each).
#define PSKV_ASK_ARGS(...) asm volatile("" ::__VA_ARGS__)
// The same in front of what `x`, a word that is the same for all lanes, is used for, and in the way of no scalar load behind it.
// (The kernels are also compiled for the CPU, which knows no such registers.)
#ifdef __HIP__
#define PSKV_SCALAR "s"
#define PSKV_ASK_ARGS_FOR(x, ...) asm("" : "+" PSKV_SCALAR(x) : __VA_ARGS__)
#else
#define PSKV_SCALAR "r"
#define PSKV_ASK_ARGS_FOR(x, ...) (void)0
#endif

namespace pskv {

// ps::kMaxKey (include/ps/base.h:18). The stock server ranges never cover it
// (src/postoffice.cc:169-180), so it marks an empty slot; a caller that pushes it
// directly is served from one side slot kept in DevState.
constexpr uint64_t kEmptyKey = ~0ull;

// A launch serves up to kMaxBatch tables at once: blockIdx.y selects the table, blockIdx.x is the
// workgroup's number among those that serve it.
constexpr int kMaxBatch = 16;

// Row reference handed from the lookup kernel to the row kernels.
//   FIXED : low bits = row index
//   VARLEN: bits [28,63) = arena offset in 16-byte units, bits [0,28) = row length in floats
// bit 63 = the key was created by this request; all ones = key absent (var-len pull).
constexpr uint64_t kRefNew = 1ull << 63;
constexpr uint64_t kRefAbsent = ~0ull;
constexpr int kLenBits = 28;
constexpr uint64_t kLenMask = (1ull << kLenBits) - 1;

// Per-tile shortcut of the var-len row kernel. When the rows that overlap a request-side tile
// lie in the arena back to back, in request order and without padding, the whole tile maps to
// the arena with one offset: the arena position (in floats) of the tile's first float.
constexpr uint64_t kTileNotAffine = ~0ull;
// The note a var-len row kernel leaves per tile for requests that repeat its request: where in
// the arena the tile's floats lie when they form one or two unbroken pieces.
//   first  = arena offset (floats) that the tile's float 0 maps to, or kTileNotAffine
//   second = 0 for one piece; else (arena offset that float 0 would map to by the second
//            piece's distance + kTileNoteBias) << kTileSplitBits | index of the first float
//            of the second piece
struct alignas(16) TileNote {
  uint64_t first, second;
};
constexpr int kTileSplitBits = 10;
constexpr int64_t kTileNoteBias = 1 << kTileSplitBits;  // keeps the second distance non-negative

// sticky device-side error bits (DevState::error)
constexpr unsigned kDevErrLenChanged = 1u;  // var-len push: stored length differs
constexpr unsigned kDevErrFull = 2u;        // probe sequence found no free slot (host sizing bug)
constexpr unsigned kDevErrBadLen = 4u;      // negative or too long length
constexpr unsigned kDevErrSizeMismatch = 8u;  // lens do not add up to the number of values
constexpr unsigned kDevErrNoRoom = 16u;       // asynchronous var-len pull: response larger than the buffer
constexpr unsigned kDevErrDuplicate = 32u;    // the same key twice in one request (row modes)
constexpr unsigned kDevErrReplay = 64u;       // a replayed request no longer names the keys it was recorded with

// Payload of a slot that has been claimed but not filled in yet (slots start as all ones).
// No valid payload has bit 63 set.
constexpr uint64_t kPayloadUnset = ~0ull;

constexpr int kBlock = 256;             // threads per workgroup of every kernel here (4 waves)

struct __align__(16) Slot {
  uint64_t key;
  uint64_t payload;  // SCALAR: the complement of a float's bits in the low word; row modes: see above (without bit 63)
};

// An empty slot is all ones, so a SCALAR slot whose key has just been written holds 0.0f: a pull that creates a key (kv_app.h:457)
// has nothing more to write. (It used to write the value as well, a third request to memory next to the line and the
// compare-and-swap: 16M keys pulled, 8.9M of them absent, 715 -> 665 us: the request that it saved had mostly been merged with the swap.)
__device__ __forceinline__ float stored_value(uint64_t payload) { return __uint_as_float(~(unsigned)payload); }
__device__ __forceinline__ void store_value(uint64_t* payload, float v) {
  *reinterpret_cast<unsigned*>(payload) = ~__float_as_uint(v);
}
// The sum of two values, of two NaNs the first. (Which of the operands of a `+` comes first the compiler chooses from kernel to kernel.
// The kernels that take pushes past k_scalar leave what it leaves: the pushed NaN, and of a run the first.)
__device__ __forceinline__ float sum_in_order(float first, float second) {
#ifdef __HIP_DEVICE_COMPILE__
  float sum;
  asm("v_add_f32 %0, %1, %2" : "=v"(sum) : "v"(first), "v"(second));
  return sum;
#else
  return first + second;
#endif
}

// Counters that every workgroup bumps are spread over kCountShards cache lines:
// atomics on one address are served one at a time, and a request can run thousands
// of workgroups.
constexpr int kCountShards = 32;
constexpr int kShardStride = 16;  // in 8-byte words: one shard per 128-byte line
constexpr int kTicketShards = 32;

struct alignas(32) DevState {
  // The first 32 bytes are what a row kernel needs to know about its request (ReqFacts below):
  // every wavefront reads them with one load.
  // "Same keys as the request that last filled the workspace" fast path of the row modes.
  // Every row-mode request has a number (epoch). cache_epoch is the request whose keys, lens,
  // row references, offsets and tile table the workspace and the key cache hold; bad_epoch ==
  // cache_epoch marks them unusable. same_epoch == e is the decision, reached once by the
  // compare kernel before anything else of request e runs, that e may reuse them.
  unsigned long long same_epoch;
  unsigned long long scan_total;       // grand total of the last lens scan
  unsigned int error;                  // sticky error bits of finished requests
  unsigned int req_error;              // error bits of the request in flight (follows `error`)
  unsigned int misaligned;             // OR of (len & 3) over the lens of the current request; a push: kReqLong as well
  unsigned int req_flags;              // kReq* facts the workgroups of the kernel in flight have found
  // 32
  unsigned long long arena_top;        // FIXED: rows handed out; VARLEN: 16-byte units handed out
  unsigned long long special_payload;  // payload of key 2^64-1
  unsigned int special_present;
  unsigned int ticket_top;             // second level of the last-workgroup ticket (ticket_last)
  unsigned long long cache_epoch;
  unsigned long long bad_epoch;
  // The request with this number was refused (FIXED: it repeats a key; k_var_push_start: a length differs from the stored
  // one): its row kernels change no stored value and leave the rows it created as zero rows
  unsigned long long refused_epoch;
  // SCALAR key cache: the last request that changed cached values without touching the slots, and
  // the value of dirty_epoch up to which the slots have been brought up to date since
  unsigned long long dirty_epoch;
  unsigned long long clean_epoch;
  // the newest request that found cached values ahead of the slots and named other keys (k_scalar<BEHIND>)
  unsigned long long behind_epoch;
  // k_scalar_repeat: votes of the launch in flight (vote.h), and launches served so far << 1 | verdict of the newest
  unsigned int repeat_arrived;
  unsigned int told_ragged;  // what the host has been told of the rows of var-len pushes (tell_ragged)
  unsigned long long repeat_verdict;
  // keys held (slot array plus the side slot) = sum of the shards
  unsigned long long count_shard[kCountShards * kShardStride];
  // first level of the last-workgroup ticket: one counter per 128-byte line, and behind it the facts of its
  // workgroups (report_facts)
  unsigned int ticket_sub[kTicketShards * 32];
  // k_fixed_own: the word of the verdict (handover.h); everyone watches it, so the line is its own
  unsigned long long push_verdict;
  // k_fixed_long: the newest of its requests that has created a row, and how many rows there were before it
  unsigned long long fresh_from;
  // k_fixed_own: a bit for every workgroup of a push that has left its rows to the last one, all zero between requests
  unsigned long long shares_left[8];
  // stream_push.h: keys that the pass over the slots leaves to the kernel behind it (requests use the two in turn, the one that
  // is not in use is zero), and the sum of the hashes of the keys of the newest such request (of the one in flight: next to
  // each word of count_shard)
  unsigned left_keys[2];
  unsigned long long keys_sum;
  unsigned long long packed_epoch;  // the cached request whose keys are there packed as well (PackedKeys)
  unsigned long long pad[3];
  // one_launch.h: what the workgroups of a var-len request tell each other, all zero between requests
  unsigned long long parts[kVarParts];
};

// The head of DevState as one load.
struct ReqFacts {
  unsigned long long same_epoch, scan_total;
  unsigned int error, req_error, misaligned, req_flags;
};
static_assert(offsetof(DevState, same_epoch) == 0 && offsetof(DevState, scan_total) == 8 &&
                  offsetof(DevState, error) == 16 && offsetof(DevState, req_error) == 20 &&
                  offsetof(DevState, misaligned) == 24 && offsetof(DevState, req_flags) == 28,
              "ReqFacts mirrors the head of DevState");
typedef unsigned int u32x8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ ReqFacts load_req_facts(const DevState* st) {
  static_assert(sizeof(ReqFacts) == 32, "ReqFacts is the first 32 bytes of DevState");
  const u32x8 w = *reinterpret_cast<const u32x8*>(st);
  ReqFacts f;
  f.same_epoch = ((unsigned long long)w[1] << 32) | w[0];
  f.scan_total = ((unsigned long long)w[3] << 32) | w[2];
  f.error = w[4];
  f.req_error = w[5];
  f.misaligned = w[6];
  f.req_flags = w[7];
  return f;
}

// Facts about the request that workgroups report into DevState::req_flags.
constexpr unsigned kReqMisaligned = 3u;  // OR of (len & 3)
constexpr unsigned kReqBadLen = 4u;      // a length negative or above the maximum
constexpr unsigned kReqDiffer = 8u;      // a key or length differs from the cached request
constexpr unsigned kReqDuplicate = 16u;  // a key equals its left neighbour (requests are sorted)
constexpr unsigned kReqLong = 32u;       // a row is much longer than the others (by_row)
constexpr unsigned kReqWide = 64u;       // two neighbouring keys are too far apart to be packed (PackedKeys)

// Counters of the table as they are after request `seq`, written by the device into pinned host memory so that the host
// can bound the counters without waiting for the stream. Both counters carry the low bits of the request's number above
// them: where those are the number's, the record is whole, whatever the order in which its words have arrived. (With a
// number in front of the counters and one behind, each waited for, it was there two trips over the host link later: four
// pushes and a pull of 4 rows of 33,728 floats, a table that is full, 38.5 -> 35.2 us; of 40 of 100,000 60 -> 57.)
constexpr unsigned kRecordTagAt = 36;  // (2^36 units of 16 bytes are four times what the GPU holds)
struct Snapshot {
  volatile uint64_t seq;
  volatile uint64_t count;
  volatile uint64_t arena_top;
};
__host__ __device__ constexpr uint64_t record_word(uint64_t counter, uint64_t seq) {
  return counter | seq << kRecordTagAt;
}

// What a row-mode kernel needs to know about the request it belongs to.
struct ReqTag {
  unsigned long long epoch;  // number of the request
  unsigned int try_cache;    // not 0: the host found the key cache structurally usable for this request (kTry*)
  // The request is a replay of a recorded one (a node of a HIP graph, launched again and again with
  // the same arguments, this number included): it is only ever served from the cache. When the
  // comparison finds other keys than the cached ones, none of its kernels changes or answers
  // anything and the table's error state says so (kDevErrReplay): the host has not sized anything
  // for keys that it has not seen.
  unsigned int replay;
};

constexpr unsigned kTryKeys = 1u;     // compared key by key
constexpr unsigned kTryPacked = 2u;   // SCALAR: the cached keys have been asked to be packed (PackedKeys)
constexpr unsigned kTryAndPack = 3u;  // SCALAR: and this is who asks

// True when request `tag` carries exactly the keys (and lens) of the cached request, so that
// the row references, offsets and tile table still in the workspace are this request's too.
// The decision is written once, by the compare kernel that runs before the other kernels of
// the request, so every workgroup of every later kernel sees the same answer.
__device__ __forceinline__ bool cache_same(const DevState* st, const ReqTag& tag) {
  return st->same_epoch == tag.epoch;
}

// True in every kernel of a replayed request whose comparison has found other keys: the kernel
// returns at once.
__device__ __forceinline__ bool replay_blocked(const DevState* st, const ReqTag& tag) {
  return tag.replay != 0u && st->same_epoch != tag.epoch;
}

// Records an error of request `epoch`; whatever that request left in the workspace is not
// to be reused.
__device__ __forceinline__ void raise_error(DevState* st, unsigned bit, unsigned long long epoch) {
  atomicOr(&st->req_error, bit);
  st->bad_epoch = epoch;
}

// Finds the workgroup that finishes last among the `nblk` workgroups that serve one table in a
// launch (workgroups blockIdx.x = 0 .. nblk-1 of the table's row of the grid). Thread 0 of EVERY
// one of them calls it once, after the writes the last workgroup is to see; it returns true in
// exactly one of them, and that thread then sees those writes.
// What the callers hand to the last workgroup must have been written with device-scope
// atomics (atomicOr, publish_u64 below): those are performed at the memory side, past the
// per-XCD L2, so all a workgroup has to do before its ticket is wait for its own
// outstanding operations. A full release fence would write the L2 back instead, once per
// workgroup, which for a grid of 2,000 workgroups costs tens of microseconds.
// Two levels of counters, the first spread over kTicketShards cache lines, because atomics
// on one address are served one at a time (about 15 ns each).
// The counters are left at zero; kernels that use it must not overlap on one table.
// In two halves, for a thread that has something to ask for in between: what it has to see to is that its atomics and
// atomic stores are complete before it takes the ticket.
__device__ __forceinline__ unsigned ticket_take(DevState* st, unsigned nblk) {
  // (a small grid goes straight to the second level)
  return atomicAdd(nblk > (unsigned)kTicketShards ? &st->ticket_sub[blockIdx.x % kTicketShards * 32] : &st->ticket_top, 1u);
}
__device__ __forceinline__ bool ticket_is_last(DevState* st, unsigned nblk, unsigned ticket) {
  unsigned shards = nblk;
  if (nblk > (unsigned)kTicketShards) {
    shards = (unsigned)kTicketShards;
    const unsigned sub = blockIdx.x % shards;
    const unsigned members = (nblk - sub + shards - 1) / shards;  // workgroups b with b % shards == sub
    if (ticket != members - 1) return false;
    st->ticket_sub[sub * 32] = 0;
    ticket = atomicAdd(&st->ticket_top, 1u);
  }
  if (ticket != shards - 1) return false;
  st->ticket_top = 0;
  // once per grid: nothing stale is left in this XCD's L2 (__threadfence would also write back what others have left there)
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  return true;
}
__device__ __forceinline__ void my_atomics_are_there() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_waitcnt(0);
}
__device__ __forceinline__ bool ticket_last(DevState* st, unsigned nblk) {
  my_atomics_are_there();
  return ticket_is_last(st, nblk, ticket_take(st, nblk));
}

// Adds a workgroup's facts (one thread calls it, before its ticket) to those of the other workgroups of a launch of
// `nblk`. Every workgroup of a request that differs from the cached one, or has ragged rows, finds the same fact, and
// accesses to one address past the L2 are served one at a time: they go next to the tickets, one word per line (a
// comparison of 4M keys that differ took 46 us with one word for all, of keys that do not 12).
__device__ __forceinline__ void report_facts(DevState* st, unsigned facts, unsigned nblk) {
  atomicOr(nblk > (unsigned)kTicketShards ? &st->ticket_sub[blockIdx.x % kTicketShards * 32 + 1] : &st->req_flags, facts);
}
// All of them, taken away: called by the 64 lanes of one wavefront of the workgroup that finished last.
__device__ __forceinline__ unsigned take_facts(DevState* st, unsigned nblk) {
  const unsigned lane = threadIdx.x & 63;
  unsigned f = 0;
  if (nblk > (unsigned)kTicketShards) {
    if (lane < (unsigned)kTicketShards) f = atomicExch(&st->ticket_sub[lane * 32 + 1], 0u);
  } else if (lane == 0) {
    f = atomicExch(&st->req_flags, 0u);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) f |= __shfl_xor(f, o);
  return f;
}

// A 64-bit value for the workgroup that ticket_last elects: stored past the L2.
__device__ __forceinline__ void publish_u64(unsigned long long* p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Adds the workgroup's total of `x` to one shard of the key counter. Every thread of
// the workgroup must call it. `red` holds kBlock/64 words of LDS.
__device__ __forceinline__ void block_count_add(DevState* st, unsigned x, unsigned* red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned t = 0;
#pragma unroll
    for (int w = 0; w < kBlock / 64; ++w) t += red[w];
    if (t) atomicAdd(&st->count_shard[(blockIdx.x % kCountShards) * kShardStride], (unsigned long long)t);
  }
}

// Workgroup-wide exclusive prefix sum of `x` plus the workgroup total; every thread must
// call it. `red` holds kBlock/64 + 1 words of LDS and may be reused after the next barrier.
__device__ __forceinline__ unsigned long long block_excl_scan_u64(unsigned long long x,
                                                                  unsigned long long* red,
                                                                  unsigned long long& total) {
  unsigned long long inc = x;
  const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    unsigned long long y = __shfl_up(inc, d);
    if (lane >= (unsigned)d) inc += y;
  }
  __syncthreads();
  if (lane == 63) red[wave] = inc;
  __syncthreads();
  unsigned long long before = 0, t = 0;
#pragma unroll
  for (unsigned w = 0; w < kBlock / 64; ++w) {
    if (w < wave) before += red[w];
    t += red[w];
  }
  total = t;
  return before + inc - x;
}

typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// One 128-bit read of a slot (key and payload together).
__device__ __forceinline__ u64x2 load_slot(const Slot* p) {
  return *reinterpret_cast<const u64x2*>(p);
}

// murmur3 finaliser: full avalanche, so evenly spaced keys (kMaxKey/n*i) spread out
__device__ __forceinline__ uint64_t mix64(uint64_t x) {
  x ^= x >> 33;
  x *= 0xff51afd7ed558ccdull;
  x ^= x >> 33;
  x *= 0xc4ceb9fe1a85ec53ull;
  x ^= x >> 33;
  return x;
}

// Home slot of a key in an array of mask + 1 slots (a power of two, at least 2): the TOP bits of
// the hash. A key's home in an array of G times the slots is then G * home + (a few more bits),
// so the keys of one stretch of an array are the keys of the G times longer stretch at the same
// relative place of the larger array, which lets a growth stream through both arrays instead of
// scattering every key (k_regrow).
__device__ __forceinline__ uint64_t home_slot(uint64_t key, uint64_t mask) {
  return mix64(key) >> __builtin_clzll(mask);
}

// Inclusive prefix sum over the 64 lanes of a wavefront. Every lane must call it.
__device__ __forceinline__ unsigned long long wave_incl_scan_u64(unsigned long long x) {
  const unsigned lane = __lane_id();
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    unsigned long long y = __shfl_up(x, d);
    if (lane >= (unsigned)d) x += y;
  }
  return x;
}

// Writes the table's counters to `out` (pinned host memory). Called by all 64 lanes of one
// wavefront, at a point of the stream where no kernel is changing the counters.
__device__ __forceinline__ void publish_snapshot(const DevState* st, Snapshot* out, uint64_t seq) {
  static_assert(kCountShards <= 64, "one lane per shard");
  const unsigned lane = threadIdx.x & 63;
  unsigned long long c = lane < kCountShards ? st->count_shard[lane * kShardStride] : 0ull;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
  const unsigned long long top = st->arena_top;
  if (lane != 0) return;
  auto tell = [](volatile uint64_t* to, uint64_t x) {
    __hip_atomic_store(const_cast<uint64_t*>(to), x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  };
  tell(&out->count, record_word(c, seq));
  tell(&out->arena_top, record_word(top, seq));
  tell(&out->seq, seq);
}

// Tries to settle `key` at slot `at`, whose contents `s` were read a moment ago: 1 = found (`seen` is the payload), 2 =
// claimed, 0 = the slot belongs to another key.
__device__ __forceinline__ int settle_slot(Slot* __restrict__ slots, uint64_t at, const u64x2& s, uint64_t key,
                                           uint64_t& seen) {
  if (s.x == key) {
    seen = s.y;
    return 1;
  }
  if (s.x == kEmptyKey) {
    unsigned long long old = atomicCAS(reinterpret_cast<unsigned long long*>(&slots[at].key),
                                       (unsigned long long)kEmptyKey, (unsigned long long)key);
    if (old == kEmptyKey) return 2;
    if (old == key) {  // same key twice in one request: undefined for callers, but stay sane
      seen = slots[at].payload;
      return 1;
    }
  }
  return 0;
}

// The walk behind slot `h`, which belongs to another key: three slots at once (a walk of one slot per round trip made
// a push a tenth slower at a fill of 0.4 than at 0.1). The first three may have been asked for already (`there`).
__device__ __forceinline__ uint64_t* walk_slots(Slot* __restrict__ slots, uint64_t mask, DevState* st, uint64_t key,
                                                uint64_t h, bool& is_new, uint64_t& seen, u64x2 s1, u64x2 s2, u64x2 s3,
                                                bool there) {
  for (uint64_t probes = 0; probes <= mask; probes += 3) {
    const uint64_t h1 = (h + 1) & mask, h2 = (h + 2) & mask, h3 = (h + 3) & mask;
    if (!there) s1 = load_slot(&slots[h1]), s2 = load_slot(&slots[h2]), s3 = load_slot(&slots[h3]);
    there = false;
    if (const int r = settle_slot(slots, h1, s1, key, seen)) return is_new = r == 2, &slots[h1].payload;
    if (const int r = settle_slot(slots, h2, s2, key, seen)) return is_new = r == 2, &slots[h2].payload;
    if (const int r = settle_slot(slots, h3, s3, key, seen)) return is_new = r == 2, &slots[h3].payload;
    h = h3;
  }
  atomicOr(&st->error, kDevErrFull);
  return nullptr;
}

// Key 2^64-1, which marks an empty slot, lives in the side slot.
__device__ __forceinline__ uint64_t* special_slot(DevState* st, bool& is_new, uint64_t& seen) {
  is_new = atomicExch(&st->special_present, 1u) == 0u;
  seen = st->special_payload;
  return reinterpret_cast<uint64_t*>(&st->special_payload);
}

// Finds `key` or claims an empty slot for it. Returns the address of the slot's
// payload (nullptr if the table has no free slot, which the host-side sizing
// rules out). `seen` is the payload read together with the key when the key was
// already present.
__device__ __forceinline__ uint64_t* find_or_insert(Slot* __restrict__ slots, uint64_t mask,
                                                    DevState* st, uint64_t key, bool& is_new,
                                                    uint64_t& seen) {
  is_new = false;
  seen = 0;
  if (key == kEmptyKey) return special_slot(st, is_new, seen);
  const uint64_t h = home_slot(key, mask);
  // The home slot alone first: at the fills this table runs at, most keys are settled there, and
  // one load per lane keeps the most wavefronts in flight.
  const u64x2 s = load_slot(&slots[h]);
  if (const int r = settle_slot(slots, h, s, key, seen)) return is_new = r == 2, &slots[h].payload;
  return walk_slots(slots, mask, st, key, h, is_new, seen, s, s, s, false);
}

// The same for the N keys of a lane, whose home slots have been read a moment ago, side by side: in a wavefront there
// is nearly always a lane that has to claim a slot or to walk on, and N keys one after the other are N round trips.
template <int N>
__device__ __forceinline__ void find_or_insert_all(Slot* __restrict__ slots, uint64_t mask, DevState* st,
                                                   const uint64_t (&key)[N], const u64x2 (&home)[N], const bool (&live)[N],
                                                   uint64_t* (&p)[N], bool (&is_new)[N], uint64_t (&seen)[N]) {
  unsigned long long old[N];
  bool walk[N];
#pragma unroll
  for (int j = 0; j < N; ++j) {
    p[j] = nullptr, is_new[j] = false, seen[j] = 0, old[j] = home[j].x;
    walk[j] = live[j] && key[j] != kEmptyKey;
    if (walk[j] && home[j].x == kEmptyKey)
      old[j] = atomicCAS(reinterpret_cast<unsigned long long*>(&slots[home_slot(key[j], mask)].key),
                         (unsigned long long)kEmptyKey, (unsigned long long)key[j]);
  }
  u64x2 s[N][3];
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const uint64_t h = home_slot(key[j], mask);
    s[j][0] = s[j][1] = s[j][2] = home[j];
    if (!walk[j]) continue;
    if (old[j] == kEmptyKey || old[j] == key[j]) {
      walk[j] = false;
      p[j] = &slots[h].payload;
      is_new[j] = old[j] == kEmptyKey;
      seen[j] = home[j].x == key[j] ? home[j].y : is_new[j] ? 0 : slots[h].payload;
    } else {
      s[j][0] = load_slot(&slots[(h + 1) & mask]);
      s[j][1] = load_slot(&slots[(h + 2) & mask]);
      s[j][2] = load_slot(&slots[(h + 3) & mask]);
    }
  }
#pragma unroll
  for (int j = 0; j < N; ++j) {
    if (walk[j])
      p[j] = walk_slots(slots, mask, st, key[j], home_slot(key[j], mask), is_new[j], seen[j], s[j][0], s[j][1], s[j][2], true);
    if (live[j] && key[j] == kEmptyKey) p[j] = special_slot(st, is_new[j], seen[j]);
  }
}

// Lookup without insertion. Returns false when the key is absent.
__device__ __forceinline__ bool find_only(const Slot* __restrict__ slots, uint64_t mask,
                                          const DevState* st, uint64_t key, uint64_t& payload) {
  if (key == kEmptyKey) {
    payload = st->special_payload;
    return st->special_present != 0u;
  }
  uint64_t h = home_slot(key, mask);
  for (uint64_t probes = 0; probes <= mask; ++probes) {
    const u64x2 s = load_slot(&slots[h]);
    if (s.x == key) {
      payload = s.y;
      return true;
    }
    if (s.x == kEmptyKey) return false;
    h = (h + 1) & mask;
  }
  return false;
}

}  // namespace pskv
#endif  // PSKV_DEVICE_COMMON_H_

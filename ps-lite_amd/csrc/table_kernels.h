// Device kernels of the HBM-resident key-value store (gfx950).
//
// They replace the body of KVServerDefaultHandle::operator()
// (include/ps/kv_app.h:442-461): `store[key] += val` becomes find-or-insert in an
// open-addressing table followed by a float add, `res.vals[i] = store[key]`
// becomes a gather. The row kernels extend the same two operations to the
// multi-float layouts of KVPairs (kv_app.h:17-31).
#ifndef PSKV_TABLE_KERNELS_H_
#define PSKV_TABLE_KERNELS_H_
#include "device_common.h"
#include "quads.h"
#include "scan.h"
#include "vote.h"

namespace pskv {

// What the kernels of a request need to know about ONE table's share of it. A launch carries up
// to kMaxBatch of these by value (blockIdx.y selects one), so that a request which the slicer
// has cut into per-server pieces (kv_app.h:562-612) costs one launch per step and not one per
// server; the single-table entry points launch with one of them.
// (The first half, all that the SCALAR kernels need, is a record of its own: a launch costs the calling thread by
// what it carries, 2.45 us with 64 bytes of arguments, 2.9 with 240, 3.8 with 3,840.)
struct TableHead {
  Slot* slots;
  uint64_t mask;
  DevState* st;
  const uint64_t* keys;  // n sorted unique keys
  const float* vals;     // SCALAR push: n values
  union {
    float* out;          // SCALAR pull: n values
    uint64_t ragged;     // VARLEN push: how the host would have ragged rows added (by_row)
  };
  uint64_t n;
  uint64_t* cache_keys;  // keys (and lens) of the request whose references the workspace holds
  // SCALAR key cache (a request that repeats the cached sorted key set is served from a
  // request-ordered value array): cache_keys above, the values in `arena`, the slot numbers in
  // `tile_key`
  float* arena;              // row storage
  uint32_t* tile_key;        // VARLEN: first key of every request-side tile, ntiles+1 entries
  Snapshot* snap;            // where the kernel that creates the request's keys leaves the counters
  uint64_t snap_seq;
  ReqTag tag;
  unsigned long long* outcome;  // pinned host word that learns how the comparison went, or null; SCALAR
                                // without the key cache: the word that takes tag.epoch when the request is done
  uint32_t nblk;        // workgroups of the launch in flight that serve this table
  uint32_t cache_mode;  // kCache* below; k_scalar_repeat: looks for the outcome before a workgroup leaves
};
struct TableReq : TableHead {
  const int32_t* lens;   // VARLEN push: n row lengths
  uint64_t nvals;        // VARLEN push: floats pushed; FIXED row kernels: the quad the launch starts at
  // row modes
  uint64_t* ref;             // n row references, written by the lookup kernel
  uint64_t* off;             // VARLEN: n+1 request-side row offsets in floats
  unsigned long long* part;  // VARLEN: per-workgroup totals of the lens scan
  TileNote* tile_aff;        // VARLEN: one note per tile
  uint64_t ntiles;           // VARLEN: tiles of the request (push) / room in the tile table (pull);
                             // FIXED row kernels: the quad the launch ends before
  int32_t* cache_lens;
  int32_t* out_lens;         // VARLEN pull: n answered lengths
  // row kernels
  float* req;             // push: request values (read); pull: response values (written)
  uint64_t total;         // floats in req
  uint64_t k;             // FIXED: floats per row
  union {
    uint32_t cached;      // FIXED lookup: the first so many positions of cache_keys and ref belong together
    uint32_t started;     // VARLEN row kernels: workgroups of the k_var_*_start in front of this one, or 0
  };
  uint32_t ignore_new;    // pull half of a push+pull: rows created by the push half hold data
  uint32_t total_on_device;  // VARLEN pull without a host round trip: the floats to move are
                             // DevState::scan_total and `total` is the room in req
  uint32_t tile_base;           // VARLEN row kernels: the launch starts at this tile of the request (a large
                                // host-resident request is served piece by piece as it arrives)
};
constexpr uint32_t kCacheOff = 0;     // SCALAR: the request neither uses nor fills the key cache
constexpr uint32_t kCacheOn = 1;      // SCALAR: serve from the cache when the keys match, else refill it
constexpr uint32_t kCachePerKey = 3;  // SCALAR pull, slots up to date: every key that sits at its cached
                                      // position is answered from the cache, the others through the slots
constexpr uint32_t kCacheOnBehind = 5;  // SCALAR: as kCacheOn, and the slots may lag behind the cache (k_scalar<BEHIND>)
constexpr uint32_t kCacheRecords = 3;   // the bits that say so: a request that is served from the cache, or fills it
constexpr uint32_t kSlotSpecial = 0xffffffffu;  // cached slot number of key 2^64-1 (the side slot)
// Every kernel comes for one, for up to four and for up to kMaxBatch tables: an argument of 3.8 KB costs the
// calling thread 4.6 us per launch, one of 240 bytes 3.
template <int TABLES>
struct ReqBatch {
  TableReq t[TABLES];
};
template <int TABLES>
struct HeadBatch {
  TableHead t[TABLES];
};
static_assert(sizeof(ReqBatch<kMaxBatch>) <= 3840, "kernel arguments are limited to 4 KiB");

// Small requests are bound by the loads that wait for each other. Left to itself the compiler puts a load where
// its value is first used, behind whatever branch that is, and a kernel argument likewise: what a kernel is going
// to need is asked for together, from where there is something to read (past the end: the last element again),
// and held here until all of it has arrived.
template <typename T>
__device__ __forceinline__ void arrived(T& x) {
  asm volatile("" : "+v"(x));
}

// ---------------------------------------------------------------------------------
// SCALAR mode: one float per key, kept in the low word of the slot payload (stored_value) so that a
// probe reads key and value with one 128-bit load.
// One lane per key. Keys are unique within a request (kv_app.h:17), so the value word of a
// slot is only ever touched by the lane that owns the key: no atomics on values, and the
// per-key sum order is the request order (requests are serialised on one stream).
// The reference's handle is a plain loop over the request (kv_app.h:451-459), so even a
// sorted request that repeats a key has a defined result there; it has the same result
// here: the lane of the first occurrence serves the whole run in order, the other lanes of
// the run stand back. Whether a lane starts or continues a run is read off the neighbouring
// lanes' keys (a shuffle; only the first and the last lane of a wavefront look at memory), which
// costs requests without repeats about 1 % of a push + pull step. One lane walks its run element
// by element, so this is for the odd repeat, not a reduction of long runs. An UNSORTED request
// that repeats a key remains a caller error with an unspecified sum.
// ---------------------------------------------------------------------------------
// Stable key sets (the idea of the reference's unused sorted-merge helper,
// include/ps/internal/parallel_kv_match.h:29-120: when both sides are sorted the same way no
// lookup is needed). The CACHE variant serves a request that repeats the cached sorted key set
// from a request-ordered value array: `cache_vals[i] += vals[i]`, fully coalesced, 12 bytes per
// key instead of a 128-byte line per probe; the slots are brought up to date (k_scalar_flush)
// before anything else looks at them. A request that does not repeat the cache goes the usual
// way and leaves its keys, their values and their slot numbers behind as the new cache.
// A pull that comes right behind the push that filled the cache (the slots are up to date then)
// needs no decision for the whole request: kCachePerKey compares key by key, in the same pass.
// PINNED: the request lies in pinned host memory, whose every read is a round trip over the host link
// (about 2 us): everything the lane needs of it is asked for at once, the neighbours of the wavefront's
// first and last key included. (From device memory the plain order is 2 % faster: those two reads are
// mostly in the cache by the time they are made.)
// BEHIND: the cached values may be ahead of the slots. Should the request name other keys than the cached one, k_same_keys has
// written back those of the positions where it does, which may be anybody's here; a position where it does not is this lane's
// alone, which takes the value from the cache. (Usually the request names the same keys: a launch in front of every request
// that found out whether there is something to write back took 4.7 us of the 75 of 16M keys and 4.3 of the 12.8 of 500,000.
// Workgroups that wrote everything back here and waited for each other took 706 us for 4M other keys, now 202 behind 98.)
// (Eight wavefronts per SIMD, said to the compiler: it came to 7 for pulls with BEHIND, 4M keys 20.4 us and not 20.0, and to
// 24.0 and not 23.0 for pushes.)
template <bool PUSH, bool PULL, bool CACHE, bool PINNED, bool BEHIND, int TABLES>
__global__ __launch_bounds__(kBlock, 8) void k_scalar(HeadBatch<TABLES> b) {
  const TableHead& d = b.t[blockIdx.y];
  unsigned blk = blockIdx.x;
  // (one fetch instead of three: a push of 1,000 keys from host memory occupies its stream for 4.22 us and not 4.45, a pull is back after
  // 11.5 and not 11.7. The other variants gain nothing beyond noise.)
  if (PINNED)
    PSKV_ASK_ARGS_FOR(blk, "s"(d.n), "s"(d.nblk), "s"(d.slots), "s"(d.mask), "s"(d.st), "s"(d.keys), "s"(d.vals), "s"(d.out),
                      "s"(d.cache_mode), "s"(d.snap), "s"(d.snap_seq), "s"(d.tag.epoch));
  const uint64_t n = d.n;
  const unsigned nblk = d.nblk;  // (the grid is sized for the table with the most workgroups)
  if (blk >= nblk) return;
  Slot* __restrict__ slots = d.slots;
  const uint64_t mask = d.mask;
  DevState* st = d.st;
  const uint64_t* __restrict__ keys = d.keys;
  const float* __restrict__ vals = d.vals;
  float* __restrict__ out = d.out;
  const bool record = CACHE && (d.cache_mode & kCacheRecords) == kCacheOn;
  if (CACHE && replay_blocked(st, d.tag)) return;
  if (record && __builtin_expect(cache_same(st, d.tag), BEHIND)) {
    // the keys are those of the cached request: position i of the request is position i of the cache
    float* __restrict__ cv = d.arena;
    if (PUSH && blk == 0 && threadIdx.x == 0) st->dirty_epoch = d.tag.epoch;  // the slots fall behind
    const bool vec = ((reinterpret_cast<uintptr_t>(vals) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
    const uint64_t stride = (uint64_t)nblk * kBlock * 4;
    for (uint64_t i = ((uint64_t)blk * kBlock + threadIdx.x) * 4; i < n; i += stride) {
      if (vec && i + 4 <= n) {
        f32x4 cur = *reinterpret_cast<const f32x4*>(cv + i);
        if (PUSH) cur = cur + __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(vals + i));
        if (PULL) __builtin_nontemporal_store(cur, reinterpret_cast<f32x4*>(out + i));
        if (PUSH) *reinterpret_cast<f32x4*>(cv + i) = cur;
      } else {
        for (uint64_t j = i; j < n && j < i + 4; ++j) {
          float cur = cv[j];
          if (PUSH) cur = cur + vals[j];
          if (PULL) out[j] = cur;
          if (PUSH) cv[j] = cur;
        }
      }
    }
    // (no key is created on this path: the counters are what they were)
    if (d.snap && blk == 0 && threadIdx.x < 64) publish_snapshot(st, d.snap, d.snap_seq);
    return;
  }
  const bool ahead = BEHIND && d.cache_mode == kCacheOnBehind && st->behind_epoch == d.tag.epoch;
  if (record && blk == 0 && threadIdx.x == 0) st->cache_epoch = d.tag.epoch;
  constexpr bool kPerKey = CACHE && PULL && !PUSH;
  bool per_key = false, differs = false;
  if (kPerKey) {
    // (nothing writes these two words while a pull of this kind runs)
    per_key = d.cache_mode == kCachePerKey && st->cache_epoch != 0ull && st->bad_epoch != st->cache_epoch;
  }
  __shared__ unsigned red[kBlock / 64];
  unsigned created = 0;
  if (kPerKey && per_key) {
    // Four keys per lane, 128 bits per load. The cached request had no repeats, so four keys that
    // equal their cached neighbours are four different keys; the key behind them says whether
    // the last of them starts a run, which goes through the slots as a whole.
    const uint64_t* __restrict__ ck = d.cache_keys;
    const float* __restrict__ cv = d.arena;
    const bool kvec = (reinterpret_cast<uintptr_t>(keys) & 15) == 0;
    const bool ovec = (reinterpret_cast<uintptr_t>(out) & 15) == 0;
    const uint64_t stride4 = (uint64_t)nblk * kBlock * 4;
    for (uint64_t i = ((uint64_t)blk * kBlock + threadIdx.x) * 4; i < n; i += stride4) {
      if (i + 4 <= n) {
        u64x2 x0, x1;
        if (kvec) {
          x0 = __builtin_nontemporal_load(reinterpret_cast<const u64x2*>(keys + i));
          x1 = __builtin_nontemporal_load(reinterpret_cast<const u64x2*>(keys + i + 2));
        } else {
          x0.x = keys[i], x0.y = keys[i + 1], x1.x = keys[i + 2], x1.y = keys[i + 3];
        }
        const u64x2 y0 = *reinterpret_cast<const u64x2*>(ck + i);
        const u64x2 y1 = *reinterpret_cast<const u64x2*>(ck + i + 2);
        const f32x4 v4 = *reinterpret_cast<const f32x4*>(cv + i);
        const uint64_t behind = i + 4 < n ? keys[i + 4] : ~x1.y;
        if (x0.x == y0.x && x0.y == y0.y && x1.x == y1.x && x1.y == y1.y && behind != x1.y) {
          if (ovec) {
            __builtin_nontemporal_store(v4, reinterpret_cast<f32x4*>(out + i));
          } else {
            out[i] = v4.x, out[i + 1] = v4.y, out[i + 2] = v4.z, out[i + 3] = v4.w;
          }
          continue;
        }
      }
      for (uint64_t j = i; j < n && j < i + 4; ++j) {  // key by key
        const uint64_t key = keys[j];
        if (j > 0 && keys[j - 1] == key) continue;  // inside a run: its first key answers for it
        const bool run = j + 1 < n && keys[j + 1] == key;
        if (!run && ck[j] == key) {
          out[j] = cv[j];
          continue;
        }
        differs = true;
        bool is_new;
        uint64_t seen;
        uint64_t* p = find_or_insert(slots, mask, st, key, is_new, seen);
        if (!p) continue;
        const float cur = is_new ? 0.0f : stored_value(seen);
        out[j] = cur;
        for (uint64_t r = j + 1; r < n && keys[r] == key; ++r) out[r] = cur;
        created += is_new ? 1u : 0u;
      }
    }
  }
  // every other request: one key per lane and turn through the slots
  const uint64_t n_turns = (kPerKey && per_key) ? 0 : n;
  const uint64_t stride = (uint64_t)nblk * kBlock;
  const unsigned lane = threadIdx.x & 63;
  // whole wavefronts stay in the loop together: the shuffles below need every lane
  for (uint64_t first = (uint64_t)blk * kBlock; first < n_turns; first += stride) {
    const uint64_t i = first + threadIdx.x;
    const bool live = i < n;
    uint64_t outside = 0;  // PINNED: the key next to the wavefront's 64 keys on this lane's side
    float v = 0.0f;
    if (PINNED) {
      const bool up = lane == 0 && i > 0 && live, down = lane == 63 && i + 1 < n;
      if (up || down) outside = keys[up ? i - 1 : i + 1];
      if (PUSH && live) v = vals[i];
    }
    const uint64_t key = live ? keys[i] : 0;
    uint64_t before = __shfl_up(key, 1);
    uint64_t after = __shfl_down(key, 1);
    // the first and the last lane look just outside the wavefront's 64 keys; their neighbours have
    // fetched those lines already
    if (PINNED) {
      if (lane == 0) before = outside;
      if (lane == 63) after = outside;
    } else {
      if (lane == 0) before = (live && i > 0) ? keys[i - 1] : ~key;
      if (lane == 63) after = (i + 1 < n) ? keys[i + 1] : ~key;
    }
    if (!live || (i > 0 && before == key)) continue;  // past the end, or inside a run
    const bool run = i + 1 < n && after == key;
    if (PUSH && !PINNED) v = vals[i];
    bool held = false;  // the cached value is the key's
    float held_value = 0.0f;
    if (BEHIND && ahead) {
      uint64_t at = i;  // (a run names the cached key of one of its positions at most)
      if (run)
        while (at + 1 < n && keys[at + 1] == key && d.cache_keys[at] != key) ++at;
      held = d.cache_keys[at] == key;
      held_value = d.arena[at];
    }
    bool is_new;
    uint64_t seen;
    uint64_t* p = find_or_insert(slots, mask, st, key, is_new, seen);
    if (record && (!p || run)) st->bad_epoch = d.tag.epoch;  // not a request the cache can stand for
    if (!p) continue;
    // an absent key starts from Val() == 0, then `+=` (kv_app.h:454): 0.0f + v, not a copy
    float cur = is_new ? 0.0f : held ? held_value : stored_value(seen);
    if (PUSH) cur = cur + v;
    if (PULL) out[i] = cur;
    if (run) {  // the rest of the run, element by element like the reference's loop
      for (uint64_t j = i + 1; j < n && keys[j] == key; ++j) {
        if (PUSH) cur = cur + vals[j];
        if (PULL) out[j] = cur;
      }
    }
    if (PUSH || held) store_value(p, cur);
    created += is_new ? 1u : 0u;
    if (record) {
      d.cache_keys[i] = key;
      d.arena[i] = cur;
      d.tile_key[i] = key == kEmptyKey ? kSlotSpecial
                                       : (uint32_t)((reinterpret_cast<Slot*>(p - 1) - slots));
    }
  }
  block_count_add(st, created, red);
  // The workgroup that finishes last tells the host, which never waits for either, whether every
  // key of a key-by-key pull sat at its cached position and, when the host asked for it (the
  // table is close to a limit), what the counters are after this request.
  // (A request without the key cache may have a host that watches a word for its end: the answers, in
  // pinned memory, come before the word.)
  const bool want_outcome = kPerKey && d.cache_mode == kCachePerKey;
  const bool want_done = !CACHE && d.outcome != nullptr;
  if (want_outcome || want_done || d.snap) {
    __shared__ unsigned s_last;
    const int any = want_outcome ? __syncthreads_or(differs ? 1 : 0) : 0;
    if (want_done) {
      __threadfence_system();
      __syncthreads();
    }
    if (threadIdx.x == 0) {
      if (any) report_facts(st, kReqDiffer, nblk);
      s_last = ticket_last(st, nblk) ? 1u : 0u;
    }
    __syncthreads();
    if (!s_last) return;
    if (want_outcome && threadIdx.x < 64) {
      const bool all = (take_facts(st, nblk) & kReqDiffer) == 0u && per_key;
      if (threadIdx.x == 0 && d.outcome) *d.outcome = (d.tag.epoch << 1) | (all ? 1ull : 0ull);
    }
    if (d.snap && threadIdx.x < 64) publish_snapshot(st, d.snap, d.snap_seq);
    if (want_done && threadIdx.x == 0)
      __hip_atomic_store(d.outcome, d.tag.epoch, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// Writes a cached value back to its slot.
__device__ __forceinline__ void write_back(const TableHead& d, uint64_t i) {
  const uint32_t slot = d.tile_key[i];
  const float v = d.arena[i];
  store_value(slot == kSlotSpecial ? reinterpret_cast<uint64_t*>(&d.st->special_payload) : &d.slots[slot].payload, v);
}

// Writes the cached values back to their slots. Launched before anything reads or changes the
// slots of a table whose cache may be ahead of them: a request that is not compared with the cached
// one, a growth, a dump.
__global__ __launch_bounds__(kBlock) void k_scalar_flush(HeadBatch<1> b) {
  const TableHead& d = b.t[0];
  if (blockIdx.x >= d.nblk) return;
  // nothing changes these two while this kernel runs except its own last workgroup, which writes
  // after every workgroup has read them
  const unsigned long long dirty = d.st->dirty_epoch;
  if (dirty <= d.st->clean_epoch) return;  // the slots are up to date
  __shared__ unsigned s_last;
  const uint64_t stride = (uint64_t)d.nblk * kBlock;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < d.n; i += stride) write_back(d, i);
  if (threadIdx.x == 0) s_last = ticket_last(d.st, d.nblk) ? 1u : 0u;
  __syncthreads();
  if (s_last && threadIdx.x == 0) d.st->clean_epoch = dirty;
}

// ---------------------------------------------------------------------------------
// Row modes, step 1: key -> row reference.
// ---------------------------------------------------------------------------------

// The decision about a request that may repeat the cached one, written down by one thread after
// every workgroup has compared its share (`same`: none found a difference and the cache was
// usable). If it is not the same, the request is going to refill the cache, so it becomes the cached request right here. Epochs start
// at 1.
__device__ __forceinline__ bool cache_usable(const DevState* st, const ReqTag& tag) {
  return tag.try_cache && st->cache_epoch != 0ull && st->bad_epoch != st->cache_epoch;
}
__device__ __forceinline__ void decide_same(DevState* st, const ReqTag& tag, bool same,
                                            unsigned long long* outcome = nullptr) {
  if (tag.replay && !same) {
    // (an earlier replay of this very request may have left its number here)
    st->same_epoch = 0ull;
    atomicOr(&st->error, kDevErrReplay);
    return;
  }
  if (same) {
    st->same_epoch = tag.epoch;
  } else {
    st->cache_epoch = tag.epoch;
  }
  // the host reads this when it gets to it (never waits for it): epoch << 1 | same; only a
  // request that was in fact compared reports
  if (outcome && tag.try_cache) *outcome = (tag.epoch << 1) | (same ? 1ull : 0ull);
}

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// What the workgroups of a comparison come to, found by the last of them. `how`: kComparesKeys, or kComparesPacked, or kPacksKeys,
// with kReqWide where this lane's could not be packed.
constexpr unsigned kComparesKeys = 0u, kComparesPacked = 1u, kPacksKeys = 2u;
// What the host is told in outcome[2] when it expects packed keys that are not there: packed again they may be, or, as they lie too
// far apart, never (then DevState::packed_epoch is the cached request's number and kCannotBePacked).
constexpr unsigned long long kNotPacked = 1ull, kNeverPacked = 2ull, kCannotBePacked = 1ull << 63;
__device__ __forceinline__ void same_keys_verdict(const TableHead& d, bool differ, unsigned how) {
  DevState* st = d.st;
  __shared__ unsigned s_last;
  const int any = __syncthreads_or(differ ? 1 : 0);
  const int wide = how & kPacksKeys ? __syncthreads_or(how & kReqWide ? 1 : 0) : 0;
  if (threadIdx.x == 0) {
    if (any || wide) report_facts(st, (any ? kReqDiffer : 0u) | (wide ? kReqWide : 0u), d.nblk);
    s_last = ticket_last(st, d.nblk) ? 1u : 0u;
  }
  __syncthreads();
  if (!s_last) return;
  if (threadIdx.x >= 64) return;
  const unsigned found = take_facts(st, d.nblk);
  const bool same = (found & kReqDiffer) == 0u && cache_usable(st, d.tag);
  if (threadIdx.x != 0) return;
  if (!same && d.cache_mode == kCacheOnBehind && st->dirty_epoch > st->clean_epoch) {
    st->behind_epoch = d.tag.epoch;
    st->clean_epoch = st->dirty_epoch;  // (by the end of the request)
  }
  if (how & kPacksKeys) {
    st->packed_epoch = same ? st->cache_epoch | (found & kReqWide ? kCannotBePacked : 0ull) : 0ull;
  }
  if (how != kComparesKeys && d.outcome && st->packed_epoch != st->cache_epoch)
    d.outcome[2] = st->packed_epoch == (st->cache_epoch | kCannotBePacked) ? kNeverPacked : kNotPacked;
  decide_same(st, d.tag, same, d.outcome);
}

// Compares the keys of a request with the cached ones and reaches the decision for the whole
// request: the workgroup that finishes last sees whether any workgroup found a difference and
// writes same_epoch. (A var-len push, whose lens count as well, compares in k_var_push_begin.)
constexpr int kSameKeysItems = 4;
template <int TABLES>
__global__ __launch_bounds__(kBlock) void k_same_keys(HeadBatch<TABLES> b) {
  const TableHead& d = b.t[blockIdx.y];
  if (blockIdx.x >= d.nblk) return;  // tables that have nothing to compare have no workgroups
  const uint64_t* __restrict__ keys = d.keys;
  const uint64_t* __restrict__ cache_keys = d.cache_keys;
  const uint64_t n = d.n;
  DevState* st = d.st;
  constexpr int kItems = kSameKeysItems;
  static_assert(kItems % 2 == 0, "two keys per 128-bit load");
  const uint64_t base = ((uint64_t)blockIdx.x * kBlock + threadIdx.x) * kItems;
  // all loads first, then the compares; 128 bits per load where the buffers allow it (the cached
  // keys always do), the request side read past the caches
  uint64_t a[kItems], c[kItems];
  const bool vec = (reinterpret_cast<uintptr_t>(keys) & 15) == 0 && base + kItems <= n;
  if (vec) {
#pragma unroll
    for (int j = 0; j < kItems; j += 2) {
      const u64x2 x = __builtin_nontemporal_load(reinterpret_cast<const u64x2*>(keys + base + j));
      const u64x2 y = *reinterpret_cast<const u64x2*>(cache_keys + base + j);
      a[j] = x.x, a[j + 1] = x.y;
      c[j] = y.x, c[j + 1] = y.y;
    }
  } else {
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      const bool in = base + j < n;
      a[j] = in ? keys[base + j] : 0;
      c[j] = in ? cache_keys[base + j] : 0;
    }
  }
  bool differ = false;
#pragma unroll
  for (int j = 0; j < kItems; ++j) differ |= a[j] != c[j];
  // Cached values that are ahead of the slots go back where the keys differ (a position past the end does not: both are 0).
  // The request's own kernel sees to the others; which way it goes is not known here. (Nothing changes these two words in
  // this launch before every workgroup has taken its ticket.)
  if (__builtin_expect(differ, 0)) {
    if (d.cache_mode == kCacheOnBehind && st->dirty_epoch > st->clean_epoch) {
#pragma unroll
      for (int j = 0; j < kItems; ++j)
        if (a[j] != c[j]) write_back(d, base + j);
    }
  }
  same_keys_verdict(d, differ, kComparesKeys);
}

// Cached keys are compared again and again while a request repeats, and of sorted keys not all has to be read for that.
// SCALAR tables keep, behind the cached keys, what each of them is above the one in front of it, in 48 bits. A wavefront compares
// its first key whole and the other 511 by what they add, which says that they are equal, or not, as surely; where they are
// not it reads the cached keys themselves. They lie as the lanes read them: per wavefront and lane the lower 32 bits of its
// eight keys, then the upper 16. PACK: a comparison with the cached keys themselves, which leaves them packed if they are the
// request's; not where two neighbours are 2^48 or more apart (one such gap is enough), nor for keys that are not sorted. A request
// whose keys are others than the packed ones pays for it (30 B per key), once or twice: comparisons that fail are left out.
// A table of the same launch whose keys are not packed is compared as by k_same_keys, 16 B per key. (With its words read for nothing and
// its keys twice, 30 B, two tables of 8M keys of which one cannot be packed took 53 us to compare and 163 to push and pull. They take 36
// and 127; as long as nothing was packed they took 38 and 131.)
// Bound by memory: 14 B per key instead of 16. Push and pull of 16M repeated keys took 130 us and take 122.6 (three tables on three
// streams in turn: 145.8 and 137), of 8M 73.1 and 69.1, of 2M 26 and 24.5. The packed words are left in the
// memory-side cache: loads that pass it by take 16M keys of three tables down to 121 us, but those of one alone up to 134-139.
// 52 registers: with the cached keys themselves held as well (140) three wavefronts per SIMD took longer than what was read less.
struct PackedKeys {
  static constexpr int kItems = 8, kPairs = kItems / 2;  // keys of a lane: pairs of neighbours, 128 keys apart
  static constexpr uint64_t kBlockKeys = 64 * kItems;
  __host__ __device__ static constexpr uint64_t blocks(uint64_t n) { return (n + kBlockKeys - 1) / kBlockKeys; }
  __host__ __device__ static constexpr size_t bytes(uint64_t n) { return blocks(n) * kBlockKeys * (8 + 6); }  // the keys' own included
  __device__ static u32x4* block(uint64_t* keys, uint64_t n, uint64_t b) {
    return reinterpret_cast<u32x4*>(keys + blocks(n) * kBlockKeys) + b * (kBlockKeys * 6 / 16);
  }
};
template <bool PACK, int TABLES>
__global__ __launch_bounds__(kBlock) void k_same_packed(HeadBatch<TABLES> b) {
  const TableHead& d = b.t[blockIdx.y];
  if (blockIdx.x >= d.nblk) return;
  const uint64_t* __restrict__ keys = d.keys;
  uint64_t* const cache_keys = d.cache_keys;
  const uint64_t n = d.n;
  const DevState* st = d.st;
  constexpr int kPairs = PackedKeys::kPairs;
  const uint64_t wave = (uint64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  const unsigned lane = threadIdx.x & 63;
  const uint64_t base = wave * PackedKeys::kBlockKeys + lane * 2;
  const bool there = wave * PackedKeys::kBlockKeys < n, first = lane == 0;
  u32x4* const block = PackedKeys::block(cache_keys, n, wave);
  const bool vec = (reinterpret_cast<uintptr_t>(keys) & 15) == 0;
  auto key_pair = [&](int q) {
    const uint64_t i = base + q * 128;
    u64x2 x;
    if (vec && i + 2 <= n) {
      x = __builtin_nontemporal_load(reinterpret_cast<const u64x2*>(keys + i));
    } else {
      x.x = i < n ? keys[i] : 0, x.y = i + 1 < n ? keys[i + 1] : 0;
    }
    return x;
  };
  auto cached_pair = [&](int q) {
    const uint64_t i = base + q * 128;
    u64x2 y;
    if (i + 2 <= n) {
      y = *reinterpret_cast<const u64x2*>(cache_keys + i);
    } else {
      y.x = i < n ? cache_keys[i] : 0, y.y = 0;
    }
    return y;
  };
  u64x2 a[kPairs];
#pragma unroll
  for (int q = 0; q < kPairs; ++q) a[q] = key_pair(q);
  // (one of the tables of the launch has been asked for this; whether its keys are there packed the device knows)
  const bool asked = d.tag.try_cache == (PACK ? kTryAndPack : kTryPacked);
  const bool packed = asked && (PACK || (st->packed_epoch == st->cache_epoch && st->cache_epoch != 0ull));
  const bool ahead = d.cache_mode == kCacheOnBehind && st->dirty_epoch > st->clean_epoch;  // (as in k_same_keys)
  bool differ = false, wide = false;
  if (!packed) {
    u64x2 c[kPairs];
#pragma unroll
    for (int q = 0; q < kPairs; ++q) c[q] = cached_pair(q);
#pragma unroll
    for (int q = 0; q < kPairs; ++q) differ |= a[q].x != c[q].x || a[q].y != c[q].y;
    if (__builtin_expect(differ && ahead, 0)) {
#pragma unroll
      for (int q = 0; q < kPairs; ++q) {
        if (a[q].x != c[q].x) write_back(d, base + q * 128);
        if (a[q].y != c[q].y) write_back(d, base + q * 128 + 1);
      }
    }
    return same_keys_verdict(d, differ, asked ? kComparesPacked : kComparesKeys);
  }
  u32x4 word[3] = {(u32x4)(0u), (u32x4)(0u), (u32x4)(0u)};
  uint64_t whole = 0;
  if (!PACK && there) {
#pragma unroll
    for (int w = 0; w < 3; ++w) word[w] = block[w * 64 + lane];
    if (first) whole = cache_keys[base];
  }
#pragma unroll
  for (int q = 0; q < kPairs; ++q) {
    const uint64_t i = base + q * 128;
    uint64_t before = __shfl_up((unsigned long long)a[q].y, 1);
    const uint64_t end = __shfl((unsigned long long)a[q ? q - 1 : 0].y, 63);
    if (first) before = end;
    const uint64_t x = a[q].x - before, y = a[q].y - a[q].x;
    const bool alone = first && q == 0;  // (the wavefront's first key is compared whole)
    if (!PACK) {
      const unsigned high = word[2][q];
      const bool equal = alone ? a[q].x == whole : x == ((uint64_t)(high & 0xffffu) << 32 | word[q / 2][q % 2 * 2]);
      differ |= i < n && !equal;
      differ |= i + 1 < n && y != ((uint64_t)(high >> 16) << 32 | word[q / 2][q % 2 * 2 + 1]);
    } else {
      wide |= (i < n && !alone && x >> 48) || (i + 1 < n && y >> 48);
      word[q / 2][q % 2 * 2] = (unsigned)x, word[q / 2][q % 2 * 2 + 1] = (unsigned)y;
      word[2][q] = (unsigned)(x >> 32 & 0xffffu) | (unsigned)(y >> 32) << 16;
    }
  }
  if (PACK && there) {
#pragma unroll
    for (int w = 0; w < 3; ++w) block[w * 64 + lane] = word[w];
  }
  if (PACK || __any(differ)) {  // the keys themselves
    differ = false;
#pragma unroll 1  // (rare: it may not take registers from the others)
    for (int q = 0; q < kPairs; ++q) {
      const u64x2 x = key_pair(q), y = cached_pair(q);
      differ |= x.x != y.x || x.y != y.y;
      if (ahead && x.x != y.x) write_back(d, base + q * 128);
      if (ahead && x.y != y.y) write_back(d, base + q * 128 + 1);
    }
  }
  same_keys_verdict(d, differ, PACK ? kPacksKeys | (wide ? kReqWide : 0u) : kComparesPacked);
}

// A recorded SCALAR request of up to kRepeatGroups workgroups: comparison and values in ONE launch. Nothing
// may change or be answered before every key of the table's share is known to be the cached one, so the
// workgroups of a table wait for each other in between: all loads are under way by then, and the wait (an atomic
// and a look at its outcome) is shorter than the end of one kernel and the start of the next (4 tables of 25,000
// keys: 4.6 + 3.6 us and the gap between them, now 5.5; the calling thread makes one launch instead of two, and a
// recorded step 8.8 -> 4.2 us).
// All workgroups have to be on the GPU together: 64 of 1,024 threads are an eighth of what it holds, so twice as
// many such launches fit side by side as a process has hardware queues to run them from. Something else may hold up
// a part of them all the same (a long kernel of small workgroups on another stream, another process): a workgroup
// that has looked for the outcome for about a second (kRepeatLooks) leaves, and nobody applies anything then
// (vote.h); the run counts as one that named other keys.
constexpr unsigned kRepeatBlock = 1024;
constexpr unsigned kRepeatGroups = 64;
constexpr unsigned kRepeatLooks = 1u << 20;
// Quads of keys per thread: one while the request fits into kRepeatGroups workgroups that way (262,144 keys), two
// up to twice that; beyond it the two kernels that fill the GPU are as quick (with four quads the registers spill).
constexpr unsigned kRepeatFew = 1, kRepeatMany = 2;
typedef unsigned long long u64x2u __attribute__((ext_vector_type(2), aligned(8)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
// (the memory of vote(): words that are only ever touched by atomics, past the per-XCD L2)
template <bool PUSH>
struct RepeatVotes {
  DevState* st;
  ReqTag tag;
  unsigned long long* told;   // (pinned: the outcome for the host)
  unsigned long long before;  // the verdict of the launch before this one
  __device__ unsigned add(unsigned x) { return atomicAdd(&st->repeat_arrived, x); }
  __device__ unsigned word() { return __hip_atomic_load(&st->repeat_arrived, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
  __device__ bool swap(unsigned from, unsigned to) { return atomicCAS(&st->repeat_arrived, from, to) == from; }
  __device__ bool publish(bool same) {
    decide_same(st, tag, same, told);
    if (PUSH && same) st->dirty_epoch = tag.epoch;  // the slots fall behind
    __hip_atomic_store(&st->repeat_arrived, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&st->repeat_verdict, ((before >> 1) + 1) << 1 | (same ? 1ull : 0ull), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    return same;
  }
  __device__ int outcome() {
    const unsigned long long now = __hip_atomic_load(&st->repeat_verdict, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return now == before ? -1 : (int)(now & 1ull);
  }
  __device__ void pause() { __builtin_amdgcn_s_sleep(1); }
};

template <bool PUSH, bool PULL, unsigned QUADS, int TABLES>
__global__ __launch_bounds__(kRepeatBlock) void k_scalar_repeat(HeadBatch<TABLES> b) {
  const TableHead& d = b.t[blockIdx.y];
  const unsigned nblk = d.nblk;
  if (blockIdx.x >= nblk) return;
  DevState* st = d.st;
  const unsigned looks = d.cache_mode;
  __shared__ unsigned s_same;
  // (nobody changes the verdict before this workgroup has voted, nor what says that the cache is usable; both are asked
  // for with the keys, and the arguments that the last vote needs as well: between the votes and the outcome nothing
  // is fetched)
  RepeatVotes<PUSH> votes{st, d.tag, d.outcome, 0ull};
  PSKV_ASK_ARGS("s"(votes.told), "s"(votes.tag.epoch), "s"(looks));
  bool usable = false;
  if (threadIdx.x == 0) {
    votes.before = __hip_atomic_load(&st->repeat_verdict, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    usable = cache_usable(st, votes.tag);
  }
  const uint64_t n = d.n;
  const uint64_t first = ((uint64_t)blockIdx.x * kRepeatBlock * QUADS + threadIdx.x) * 4;
  f32x4 cur[QUADS], add[QUADS];
  u64x2u x0[QUADS], x1[QUADS];
  u64x2 y0[QUADS], y1[QUADS];
#pragma unroll
  for (unsigned q = 0; q < QUADS; ++q) {
    const uint64_t i = first + (uint64_t)q * kRepeatBlock * 4;
    cur[q] = add[q] = (f32x4)(0.f);
    x0[q] = x1[q] = (u64x2u)(0ull);
    y0[q] = y1[q] = (u64x2)(0ull);
    if (i + 4 <= n) {
      x0[q] = *reinterpret_cast<const u64x2u*>(d.keys + i), x1[q] = *reinterpret_cast<const u64x2u*>(d.keys + i + 2);
      y0[q] = *reinterpret_cast<const u64x2*>(d.cache_keys + i);
      y1[q] = *reinterpret_cast<const u64x2*>(d.cache_keys + i + 2);
      cur[q] = *reinterpret_cast<const f32x4*>(d.arena + i);
      if (PUSH) add[q] = *reinterpret_cast<const f32x4u*>(d.vals + i);
    } else {
#pragma unroll
      for (unsigned j = 0; j < 4; ++j) {
        if (i + j >= n) continue;
        const uint64_t x = d.keys[i + j], y = d.cache_keys[i + j];
        if (j < 2) x0[q][j] = x, y0[q][j] = y; else x1[q][j - 2] = x, y1[q][j - 2] = y;
        cur[q][j] = d.arena[i + j];
        if (PUSH) add[q][j] = d.vals[i + j];
      }
    }
  }
  bool differ = false;
#pragma unroll
  for (unsigned q = 0; q < QUADS; ++q)
    differ |= x0[q].x != y0[q].x || x0[q].y != y0[q].y || x1[q].x != y1[q].x || x1[q].y != y1[q].y;
  const bool any = __syncthreads_or(differ ? 1 : 0) != 0;
  if (threadIdx.x == 0) {
    // (the old verdict has to be here before the vote goes out, behind which it may change)
    asm volatile("" : "+v"(votes.before) : : "memory");
    s_same = vote(votes, nblk, usable && !any, looks) ? 1u : 0u;
  }
  __syncthreads();
  if (!s_same) return;
#pragma unroll
  for (unsigned q = 0; q < QUADS; ++q) {
    const uint64_t i = first + (uint64_t)q * kRepeatBlock * 4;
    if (PUSH) cur[q] = cur[q] + add[q];
    if (i + 4 <= n) {
      if (PULL) *reinterpret_cast<f32x4u*>(d.out + i) = cur[q];
      if (PUSH) *reinterpret_cast<f32x4*>(d.arena + i) = cur[q];
    } else {
#pragma unroll
      for (unsigned j = 0; j < 4; ++j) {
        if (i + j >= n) continue;
        if (PULL) d.out[i + j] = cur[q][j];
        if (PUSH) d.arena[i + j] = cur[q][j];
      }
    }
  }
}

// The counter record of a request, written by the kernel that creates its keys once every
// workgroup has taken its rows (or at once when the request creates nothing): the record then
// holds the counters as they are AFTER the request. Every thread of the workgroup calls it;
// `s_last` is one word of LDS.
__device__ __forceinline__ void publish_after_lookup(DevState* st, Snapshot* snap, uint64_t seq,
                                                     unsigned nblk, unsigned* s_last) {
  if (!snap) return;
  if (threadIdx.x == 0) *s_last = ticket_last(st, nblk) ? 1u : 0u;
  __syncthreads();
  if (*s_last && threadIdx.x < 64) publish_snapshot(st, snap, seq);
}

// Keys per thread and round of the creating lookups: 4 for large requests (fewer atomic adds on
// the arena counter), 1 for small ones (enough workgroups to fill the GPU).
constexpr int kLookupItemsLarge = 4;
constexpr uint64_t kLookupLargeKeys = 1u << 20;

// FIXED: find or create the row of every key. Push and pull both create
// (pull of an absent key inserts a zero value, kv_app.h:457).
// A round handles kBlock*kLookupItems keys, kLookupItems consecutive ones per thread:
// every thread claims slots for its keys, then the workgroup takes the rows of all
// created keys from the arena with ONE atomic add and a workgroup-wide scan hands them
// out in request order, so rows of neighbouring keys are neighbours in the arena.
// A key's row never changes, so a reference that an earlier request has left at the key's position
// (cache_keys holds the key it was left for) is the key's still: it is used as it is, and only the other
// keys are looked up. A request that repeats the last one, or a push behind the pull of its keys, streams
// through 24 B per key here. (It used to be compared as a whole by a launch of its own in front of this one:
// 6.8 us of comparison and 4.5 us of a lookup that returned at once for 1M keys, and both for every small
// request.)
// FIXED: request `tag` repeats a key. Reported by the next wait; the request's row kernels
// change no stored value.
__device__ __forceinline__ void refuse_fixed(DevState* st, const ReqTag& tag) {
  atomicOr(&st->error, kDevErrDuplicate);
  st->bad_epoch = tag.epoch;
  st->refused_epoch = tag.epoch;
}

template <int kLookupItems, int TABLES>
__global__ __launch_bounds__(kBlock) void k_lookup_fixed(ReqBatch<TABLES> b) {
  const TableReq& d = b.t[blockIdx.y];
  PSKV_ASK_ARGS("s"(d.slots), "s"(d.mask), "s"(d.st), "s"(d.keys), "s"(d.n), "s"(d.ref), "s"(d.cache_keys),
                "s"(d.snap), "s"(d.tag.epoch), "s"(d.cached), "s"(d.nblk));
  const unsigned nblk = d.nblk;
  if (blockIdx.x >= nblk) return;
  Slot* __restrict__ slots = d.slots;
  const uint64_t mask = d.mask;
  DevState* st = d.st;
  const uint64_t* __restrict__ keys = d.keys;
  const uint64_t n = d.n;
  uint64_t* __restrict__ ref = d.ref;
  uint64_t* __restrict__ cache_keys = d.cache_keys;
  const ReqTag tag = d.tag;
  Snapshot* snap = d.snap;
  const uint64_t snap_seq = d.snap_seq;
  const uint64_t cached = d.cached;
  if (blockIdx.x == 0 && threadIdx.x == 0) st->cache_epoch = tag.epoch;
  __shared__ unsigned long long red[kBlock / 64];
  __shared__ unsigned cred[kBlock / 64];
  __shared__ unsigned long long s_first;
  __shared__ unsigned s_last;
  unsigned created = 0;
  constexpr uint64_t kRound = (uint64_t)kBlock * kLookupItems;
  for (uint64_t base = (uint64_t)blockIdx.x * kRound; base < n; base += (uint64_t)nblk * kRound) {
    uint64_t* p[kLookupItems];
    uint64_t seen[kLookupItems];
    uint64_t was[kLookupItems];  // the reference that is there already, if it is this key's
    bool is_new[kLookupItems];
    unsigned mine = 0;
    // (the buffers have room for n keys; what lies beyond `cached` is not looked at)
    uint64_t key[kLookupItems], left[kLookupItems], cached_key[kLookupItems], cached_ref[kLookupItems];
#pragma unroll
    for (int j = 0; j < kLookupItems; ++j) {
      const uint64_t i = base + (uint64_t)threadIdx.x * kLookupItems + j, at = i < n ? i : n - 1;
      key[j] = keys[at];
      left[j] = keys[at ? at - 1 : 0];
      cached_key[j] = cache_keys[at];
      cached_ref[j] = ref[at];
    }
#pragma unroll
    for (int j = 0; j < kLookupItems; ++j) arrived(key[j]), arrived(left[j]), arrived(cached_key[j]), arrived(cached_ref[j]);
#pragma unroll
    for (int j = 0; j < kLookupItems; ++j) {
      const uint64_t i = base + (uint64_t)threadIdx.x * kLookupItems + j;
      p[j] = nullptr;
      is_new[j] = false;
      seen[j] = 0;
      was[j] = kRefAbsent;
      if (i < n) {
        // keys are sorted and must be unique (kv_app.h:17): a key that equals its left neighbour
        // refuses the request, whether the key is new or has been in the table for long
        if (i > 0 && left[j] == key[j]) {
          refuse_fixed(st, tag);
          cache_keys[i] = key[j];
        } else if (i < cached && cached_key[j] == key[j] && cached_ref[j] != kRefAbsent) {
          was[j] = cached_ref[j];
        } else {
          cache_keys[i] = key[j];
          p[j] = find_or_insert(slots, mask, st, key[j], is_new[j], seen[j]);
        }
      }
      if (p[j] && !is_new[j] && seen[j] == kPayloadUnset) {
        // (unsorted request) another lane of this request is creating the very same key
        refuse_fixed(st, tag);
        p[j] = nullptr;
      }
      mine += (p[j] && is_new[j]) ? 1u : 0u;
    }
    unsigned long long total;
    unsigned long long at = block_excl_scan_u64(mine, red, total);
    if (threadIdx.x == 0 && total) s_first = atomicAdd(&st->arena_top, total);
    __syncthreads();
    at += total ? s_first : 0ull;
#pragma unroll
    for (int j = 0; j < kLookupItems; ++j) {
      const uint64_t i = base + (uint64_t)threadIdx.x * kLookupItems + j;
      if (i >= n) continue;
      if (was[j] != kRefAbsent) {  // (created by the request that left it, but not by this one)
        if (was[j] & kRefNew) ref[i] = was[j] & ~kRefNew;
        continue;
      }
      if (!p[j]) {
        ref[i] = kRefAbsent;
        continue;
      }
      uint64_t row = seen[j];
      if (is_new[j]) {
        row = at++;
        *p[j] = row;
      }
      ref[i] = row | (is_new[j] ? kRefNew : 0ull);
    }
    created += mine;
    __syncthreads();  // s_first and red are reused by the next round
  }
  block_count_add(st, created, cred);
  publish_after_lookup(st, snap, snap_seq, nblk, &s_last);
}

// Four consecutive keys of a request with a word each, starting at index `at`: 128-bit loads where all four are
// there (keys on any 8-byte, words on any 4-byte boundary), `fill` and zero keys past the end.
template <typename W>
struct FourKeys {
  uint64_t k[4];
  W v[4];
};
template <typename W>
__device__ __forceinline__ void load_four(FourKeys<W>& f, const uint64_t* keys, const W* words, uint64_t at, uint64_t n,
                                          W fill) {
  static_assert(kScanItems == 4, "four keys per thread");
  if (at + 4 <= n) {
    const u64x2u a = *reinterpret_cast<const u64x2u*>(keys + at);
    const u64x2u b = *reinterpret_cast<const u64x2u*>(keys + at + 2);
    typedef W W4 __attribute__((ext_vector_type(4), aligned(sizeof(W))));
    const W4 w = *reinterpret_cast<const W4*>(words + at);
    f.k[0] = a.x, f.k[1] = a.y, f.k[2] = b.x, f.k[3] = b.y;
    f.v[0] = w.x, f.v[1] = w.y, f.v[2] = w.z, f.v[3] = w.w;
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f.k[j] = at + j < n ? keys[at + j] : 0;
      f.v[j] = at + j < n ? words[at + j] : fill;
    }
  }
}

// Tells the host, in the word behind that of the outcomes, when a table's pushes come to have ragged rows or cease to.
__device__ __forceinline__ void tell_ragged(DevState* st, unsigned long long* outcome, unsigned flags) {
  const unsigned ragged = flags & kReqMisaligned ? 1u : 0u;
  if (!outcome || ragged == st->told_ragged) return;
  st->told_ragged = ragged;
  outcome[1] = ragged;
}

// TableHead::ragged of a VARLEN push whose rows the host takes to be ragged: 2^shift lanes per row, two or three turns of them, and the longest
// row for which that will do; 0: a wavefront per 256 floats.
constexpr unsigned kByRowBits = 8, kByRowThree = 1u << 7;
__host__ __device__ constexpr uint64_t by_row(unsigned shift, bool three, uint64_t longest) {
  return longest << kByRowBits | (three ? kByRowThree : 0u) | (shift + 1);
}
__host__ __device__ constexpr unsigned by_row_shift(uint64_t ragged) { return ((unsigned)ragged & (kByRowThree - 1)) - 1; }
__device__ __forceinline__ unsigned longest_by_row(const TableReq& d) { return d.ragged ? (unsigned)(d.ragged >> kByRowBits) : ~0u; }

// VARLEN push, first kernel: one pass over the request's keys and lens that
//   - compares them with the cached request (when the host found the cache usable),
//   - takes pass 1 of the lens scan (per-workgroup totals, flags),
// and whose last workgroup decides whether the request repeats the cached one and scans the
// totals. Always launched for a push, so the decision and the scan cost no launch of their
// own.
// (Bound by its tail, not by its bytes: the tickets, and the scan of the totals, which a request that
// repeats the cached one does without.)
template <int TABLES>
__global__ __launch_bounds__(kBlock) void k_var_push_begin(ReqBatch<TABLES> b) {
  const TableReq& d = b.t[blockIdx.y];
  const unsigned nblk = d.nblk;
  if (blockIdx.x >= nblk) return;
  const uint64_t* __restrict__ keys = d.keys;
  const int32_t* __restrict__ lens = d.lens;
  const uint64_t n = d.n;
  unsigned long long* __restrict__ part = d.part;
  DevState* st = d.st;
  constexpr unsigned max_len = PSKV_MAX_VARLEN_ROW;
  const unsigned longest = longest_by_row(d);
  const ReqTag tag = d.tag;
  __shared__ unsigned long long red[kBlock / 64];
  __shared__ unsigned fred[kBlock / 64];
  __shared__ unsigned long long carry_s;
  __shared__ unsigned s_last, s_same;
  const uint64_t base = ((uint64_t)blockIdx.x * kBlock + threadIdx.x) * kScanItems;
  // all loads first, then the arithmetic
  FourKeys<int32_t> mine, old;
  load_four(mine, keys, lens, base, n, 0);
  if (tag.try_cache) {
    load_four(old, d.cache_keys, d.cache_lens, base, n, 0);
  } else {
    old = mine;
  }
  // the key in front of this thread's first one (its neighbour has asked for that line already)
  const uint64_t left = (base > 0 && base < n) ? keys[base - 1] : 0;
  unsigned long long s = 0;
  unsigned flags = 0;
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    const int32_t l = mine.v[j];
    s += (unsigned long long)(long long)l;
    flags |= (unsigned)l & kReqMisaligned;
    flags |= (unsigned)l > longest ? kReqLong : 0u;
    flags |= (l < 0 || (unsigned)l > max_len) ? kReqBadLen : 0u;
    flags |= (mine.k[j] != old.k[j] || l != old.v[j]) ? kReqDiffer : 0u;
    // keys are sorted and must be unique (kv_app.h:17): a key that equals its left neighbour
    // refuses the request before anything of it is applied
    const bool has_left = base + j < n && base + j > 0;
    flags |= (has_left && mine.k[j] == (j ? mine.k[j - 1] : left)) ? kReqDuplicate : 0u;
  }
  if (!scan_pass1_block(s, flags, part, st, nblk, red, fred, &s_last)) return;
  flags = scan_pass1_facts(st, nblk);
  if (threadIdx.x == 0) s_same = !(flags & kReqDiffer) && cache_usable(st, tag) ? 1u : 0u;
  __syncthreads();
  const bool same = s_same != 0u;
  scan_pass1_last(part, st, nblk, tag.epoch, flags, same, red, &carry_s);
  if (threadIdx.x == 0) {
    decide_same(st, tag, same, d.outcome);
    tell_ragged(st, d.outcome, flags);
  }
}

// VARLEN push, second kernel: pass 2 of the lens scan (request-side offsets and the tile
// table) and, for the same keys, find-or-create: a created row gets ceil(len/4) 16-byte
// units of the arena, so every row starts 16-byte aligned; a present row must have the
// pushed length. A workgroup handles chunks of kBlock*kItems consecutive keys (one each, or, when the
// request is expected to repeat the cached one and the kernel to return at once, several): every thread
// claims slots for its keys, then the workgroup takes the rows of all created keys from the arena
// with ONE atomic add and a workgroup-wide scan hands them out in request order, so rows of
// neighbouring keys are neighbours in the arena.
constexpr unsigned kTileVar = 256;  // request-side floats per wavefront of the var-len row kernel: one quad per lane
constexpr unsigned long long kArenaPadUnits = 8;  // 128 bytes in 16-byte allocation units

template <int kItems, int TABLES>
__global__ __launch_bounds__(kBlock) void k_var_push_lookup(ReqBatch<TABLES> b) {
  const TableReq& d = b.t[blockIdx.y];
  const unsigned nblk = d.nblk;
  if (blockIdx.x >= nblk) return;
  Slot* __restrict__ slots = d.slots;
  const uint64_t mask = d.mask;
  DevState* st = d.st;
  const uint64_t* __restrict__ keys = d.keys;
  const int32_t* __restrict__ lens = d.lens;
  const uint64_t n = d.n, nvals = d.nvals;
  const unsigned long long* __restrict__ part = d.part;
  uint64_t* __restrict__ off = d.off;
  uint32_t* __restrict__ tile_key = d.tile_key;
  const uint64_t ntiles = d.ntiles;
  constexpr uint64_t tile = kTileVar;
  uint64_t* __restrict__ ref = d.ref;
  uint64_t* __restrict__ cache_keys = d.cache_keys;
  int32_t* __restrict__ cache_lens = d.cache_lens;
  const ReqTag tag = d.tag;
  Snapshot* snap = d.snap;
  const uint64_t snap_seq = d.snap_seq;
  if (cache_same(st, tag)) {  // offsets, tile table and references of the cached request hold
    if (snap && blockIdx.x == 0 && threadIdx.x < 64) publish_snapshot(st, snap, snap_seq);
    return;
  }
  if (tag.replay) return;
  // the request is refused as a whole when its lens are invalid or do not add up to vals.size(),
  // or when it repeats a key
  // (a refused request creates nothing, so the counter record the host may be waiting for holds
  // the counters as they are)
  if (st->req_error & (kDevErrBadLen | kDevErrSizeMismatch | kDevErrDuplicate)) {
    if (snap && blockIdx.x == 0 && threadIdx.x < 64) publish_snapshot(st, snap, snap_seq);
    return;
  }
  if (st->scan_total != nvals) {
    if (blockIdx.x == 0 && threadIdx.x == 0) raise_error(st, kDevErrSizeMismatch, tag.epoch);
    if (snap && blockIdx.x == 0 && threadIdx.x < 64) publish_snapshot(st, snap, snap_seq);
    return;
  }
  __shared__ unsigned long long wsum[kBlock / 64];
  __shared__ unsigned long long red[kBlock / 64];
  __shared__ unsigned cred[kBlock / 64];
  __shared__ unsigned long long s_first;
  __shared__ unsigned s_last;
  unsigned created = 0;
  constexpr uint64_t kChunk = (uint64_t)kBlock * kItems;
  static_assert(kScanPart % kChunk == 0, "a part of the scan is a whole number of chunks");
  for (uint64_t first_key = (uint64_t)blockIdx.x * kChunk; first_key < n; first_key += (uint64_t)nblk * kChunk) {
    const uint64_t base = first_key + (uint64_t)threadIdx.x * kItems;
    unsigned long long len[kItems];
#pragma unroll
    for (int j = 0; j < kItems; ++j) len[j] = base + j < n ? (unsigned long long)(uint32_t)lens[base + j] : 0ull;
    // where the chunk's first row starts in the request: the offset of its part of the scan, and the lens
    // of that part in front of the chunk
    const uint64_t part_key = first_key / kScanPart * kScanPart;
    unsigned long long start = 0;
    if (kChunk < kScanPart) {
      for (uint64_t i = part_key + threadIdx.x; i < first_key; i += kBlock) start += (unsigned long long)(uint32_t)lens[i];
      unsigned none = 0;
      block_sum_or(start, none, red, cred);
    }
    start += part[first_key / kScanPart];
    scan_pass2_offsets<kItems>(len, base, n, start, off, tile_key, ntiles, tile, wsum);

    uint64_t* p[kItems];
    uint64_t seen[kItems];
    bool is_new[kItems];
    unsigned long long units = 0;
    unsigned mine = 0;
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      const uint64_t i = base + j;
      p[j] = nullptr;
      is_new[j] = false;
      seen[j] = 0;
      if (i < n) {
        const uint64_t key = keys[i];
        cache_keys[i] = key;
        cache_lens[i] = (int32_t)len[j];
        p[j] = find_or_insert(slots, mask, st, key, is_new[j], seen[j]);
        if (p[j] && !is_new[j] && seen[j] == kPayloadUnset) {
          atomicOr(&st->error, kDevErrDuplicate);  // the same key twice in this request
          st->bad_epoch = tag.epoch;
          p[j] = nullptr;
        }
      }
      if (p[j] && is_new[j]) {
        units += (len[j] + 3) >> 2;
        ++mine;
      }
    }
    unsigned long long total;
    unsigned long long at = block_excl_scan_u64(units, red, total);
    if (threadIdx.x == 0 && total) {
      // kArenaPadUnits - 1 units of slack let the chunk's rows start at an arena address that
      // is congruent, modulo 128 bytes, to the request-side offset of the chunk's first key.
      // When all its keys are new (a first push) the rows then mirror the request 128-byte line
      // for 128-byte line, and the row kernels' arena accesses are as aligned as their
      // request-side ones (misaligned ones cost about 5 % of their bandwidth).
      const unsigned long long first = atomicAdd(&st->arena_top, total + (kArenaPadUnits - 1));
      const unsigned long long want = (start >> 2) & (kArenaPadUnits - 1);
      s_first = first + ((want - first) & (kArenaPadUnits - 1));
    }
    __syncthreads();
    at += total ? s_first : 0ull;
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      const uint64_t i = base + j;
      if (i >= n) continue;
      if (!p[j]) {
        ref[i] = kRefAbsent;
        continue;
      }
      uint64_t payload = seen[j];
      if (is_new[j]) {
        payload = ((uint64_t)at << kLenBits) | len[j];
        at += (len[j] + 3) >> 2;
        *p[j] = payload;
      } else if ((payload & kLenMask) != len[j]) {
        raise_error(st, kDevErrLenChanged, tag.epoch);
      }
      ref[i] = payload | (is_new[j] ? kRefNew : 0ull);
    }
    created += mine;
    __syncthreads();  // the shared words are reused by the next chunk
  }
  block_count_add(st, created, cred);
  publish_after_lookup(st, snap, snap_seq, nblk, &s_last);
}

// VARLEN pull, first kernel: the stored length of every key (an absent key answers length 0
// and is not created) together with pass 1 of the scan over those lengths. A key that sits where the
// cached push had it is present with the cached length, and its reference is in the workspace: only the
// others are looked up. When every key does, the offsets of that push are the offsets of this response
// as well, and the scan of the totals falls away. (The comparison was a launch of its own in front of this
// one; a recorded request, which must not answer anything before the decision is there, still has it.)
template <int TABLES>
__global__ __launch_bounds__(kBlock) void k_var_pull_lookup(ReqBatch<TABLES> b) {
  const TableReq& d = b.t[blockIdx.y];
  const unsigned nblk = d.nblk;
  if (blockIdx.x >= nblk) return;
  const Slot* __restrict__ slots = d.slots;
  const uint64_t mask = d.mask;
  DevState* st = d.st;
  const uint64_t* __restrict__ keys = d.keys;
  const uint64_t n = d.n;
  uint64_t* __restrict__ ref = d.ref;
  int32_t* __restrict__ out_lens = d.out_lens;
  unsigned long long* __restrict__ part = d.part;
  const ReqTag tag = d.tag;
  __shared__ unsigned long long red[kBlock / 64];
  __shared__ unsigned fred[kBlock / 64];
  __shared__ unsigned long long carry_s;
  __shared__ unsigned s_last, s_same;
  const uint64_t base = ((uint64_t)blockIdx.x * kBlock + threadIdx.x) * kScanItems;
  if (tag.replay) {
    if (!cache_same(st, tag)) return;
#pragma unroll
    for (int j = 0; j < kScanItems; ++j)
      if (base + j < n) out_lens[base + j] = d.cache_lens[base + j];
    return;
  }
  // (the last workgroup alone changes what this reads, after every workgroup has read it)
  const bool usable = cache_usable(st, tag);
  FourKeys<int32_t> old;
  uint64_t key[kScanItems];
  bool known[kScanItems], hit[kScanItems];
  uint64_t payload[kScanItems];
  int32_t l[kScanItems];
  if (base + kScanItems <= n) {
    const u64x2u a = *reinterpret_cast<const u64x2u*>(keys + base);
    const u64x2u c = *reinterpret_cast<const u64x2u*>(keys + base + 2);
    key[0] = a.x, key[1] = a.y, key[2] = c.x, key[3] = c.y;
  } else {
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) key[j] = base + j < n ? keys[base + j] : 0;
  }
  if (usable) load_four(old, d.cache_keys, d.cache_lens, base, n, 0);
  bool all = true;
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    known[j] = base + j >= n || (usable && old.k[j] == key[j]);
    l[j] = known[j] && base + j < n ? old.v[j] : 0;
    all = all && known[j];
  }
  unsigned bits = 0;
  if (!all) {
    bits = kReqDiffer;
    // the home slots of the thread's keys together: a probe is one line from memory
    u64x2 home[kScanItems];
#pragma unroll
    for (int j = 0; j < kScanItems; ++j)
      if (!known[j]) home[j] = load_slot(&slots[home_slot(key[j], mask)]);
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
      if (known[j]) continue;
      if (home[j].x == key[j] && key[j] != kEmptyKey) {
        hit[j] = true;
        payload[j] = home[j].y;
      } else {
        hit[j] = find_only(slots, mask, st, key[j], payload[j]);
      }
      l[j] = hit[j] ? (int32_t)(payload[j] & kLenMask) : 0;
      ref[base + j] = hit[j] ? payload[j] : kRefAbsent;
    }
  }
  unsigned long long s = 0;
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    s += (uint32_t)l[j];
    bits |= (unsigned)l[j] & kReqMisaligned;
  }
  if (base + kScanItems <= n) {
    typedef int32_t i32x4u __attribute__((ext_vector_type(4), aligned(4)));
    i32x4u w;
    w.x = l[0], w.y = l[1], w.z = l[2], w.w = l[3];
    *reinterpret_cast<i32x4u*>(out_lens + base) = w;
  } else {
#pragma unroll
    for (int j = 0; j < kScanItems; ++j)
      if (base + j < n) out_lens[base + j] = l[j];
  }
  if (!scan_pass1_block(s, bits, part, st, nblk, red, fred, &s_last)) return;
  const unsigned flags = scan_pass1_facts(st, nblk);
  if (threadIdx.x == 0) s_same = !(flags & kReqDiffer) && usable ? 1u : 0u;
  __syncthreads();
  const bool same = s_same != 0u;
  scan_pass1_last(part, st, nblk, tag.epoch, flags, same, red, &carry_s);
  if (threadIdx.x == 0) {
    if (same) {
      st->same_epoch = tag.epoch;
    } else {
      // this pull has rewritten references in the workspace, and its offsets will: the cached push is gone
      st->bad_epoch = st->cache_epoch;
    }
    if (d.outcome && tag.try_cache) *d.outcome = (tag.epoch << 1) | (same ? 1ull : 0ull);
  }
}

// VARLEN pull, second kernel: pass 2 of the scan over the answered lengths: the request-side
// offsets of the response and its tile table. `ntiles_cap` is the room in the table; the
// tiles in use follow from the scanned total.
template <int TABLES>
__global__ __launch_bounds__(kBlock) void k_var_offsets(ReqBatch<TABLES> b) {
  const TableReq& d = b.t[blockIdx.y];
  if (blockIdx.x >= d.nblk) return;
  const int32_t* __restrict__ lens = d.out_lens;  // the lengths the lookup kernel answered
  const uint64_t n = d.n;
  const unsigned long long* __restrict__ part = d.part;
  uint64_t* __restrict__ off = d.off;
  uint32_t* __restrict__ tile_key = d.tile_key;
  const uint64_t ntiles_cap = d.ntiles;
  constexpr uint64_t tile = kTileVar;
  const DevState* st = d.st;
  const ReqTag tag = d.tag;
  if (cache_same(st, tag) || tag.replay) return;  // offsets and tile table of the cached request hold
  __shared__ unsigned long long wsum[kBlock / 64];
  uint64_t ntiles = (st->scan_total + tile - 1) / tile;
  if (ntiles > ntiles_cap) ntiles = ntiles_cap;
  for (uint64_t first = (uint64_t)blockIdx.x * kScanPart; first < n; first += (uint64_t)d.nblk * kScanPart) {
    const uint64_t base = first + (uint64_t)threadIdx.x * kScanItems;
    unsigned long long len[kScanItems];
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) len[j] = base + j < n ? (unsigned long long)(uint32_t)lens[base + j] : 0ull;
    scan_pass2_offsets<kScanItems>(len, base, n, part[first / kScanPart], off, tile_key, ntiles, tile, wsum);
    __syncthreads();  // wsum is reused by the next part
  }
}

// ---------------------------------------------------------------------------------
// Row modes, step 2: stream the values.
// The unit of work is a quad: four consecutive floats of the request-side buffer (one 128-bit access
// per lane), so the load is balanced for any mix of row lengths. Quads need not lie on 16-byte
// boundaries: a 128-bit access to global memory may start at any float, and costs a wavefront of
// consecutive quads one 128-byte line in eight at most.
// FIXED cuts every row into quads of its own (the last one shorter when k is not a multiple of four) and
// locates the row of a quad by division; VARLEN cuts the request into quads, stages the offsets and row
// references of the keys that overlap a wavefront's stretch in LDS and locates rows by binary search
// there.
// ---------------------------------------------------------------------------------
struct RowsParams {
  float* req;                // push: request values (read); pull: response values (written)
  float* arena;              // row storage
  const uint64_t* ref;       // n row references from the lookup kernel
  const uint64_t* off;       // VARLEN: n+1 request-side row offsets in floats
  const uint32_t* tile_key;  // VARLEN: ntiles+1 entries
  TileNote* tile_aff;        // VARLEN: one note per tile
  DevState* st;
  uint64_t n;
  uint64_t total;         // VARLEN: floats in req
  uint64_t k;             // FIXED: floats per row
  uint32_t ignore_new;    // pull half of a push+pull: rows created by the push half hold data
  uint32_t total_on_device;  // VARLEN pull without a host round trip: the floats to move are
                             // DevState::scan_total and `total` is the room in req
  uint32_t blk;              // VARLEN: the workgroup's number among those that cover the request
  ReqTag tag;
};

constexpr int kOpAcc = 0;
constexpr int kOpGather = 1;

// Four (three, two) floats that start at any float. STREAM selects non-temporal accesses: a
// request far larger than the caches is read and written once per launch, and telling
// the memory system so is worth 10-15 % of bandwidth on this GPU.
typedef float f32x3u __attribute__((ext_vector_type(3), aligned(4)));
typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));
template <bool STREAM>
__device__ __forceinline__ f32x4 load_quad(const float* p) {
  const f32x4u* q = reinterpret_cast<const f32x4u*>(p);
  return STREAM ? __builtin_nontemporal_load(q) : *q;
}
template <bool STREAM>
__device__ __forceinline__ void store_quad(f32x4 v, float* p) {
  f32x4u* q = reinterpret_cast<f32x4u*>(p);
  if (STREAM) __builtin_nontemporal_store((f32x4u)v, q); else *q = v;
}
// The first `count` (1 to 4) floats of a quad, one access each.
template <bool STREAM>
__device__ __forceinline__ f32x4 load_part(const float* p, unsigned count) {
  f32x4 v = (f32x4)(0.f);
  if (count == 4) {
    v = load_quad<STREAM>(p);
  } else if (count == 3) {
    const f32x3u* q = reinterpret_cast<const f32x3u*>(p);
    const f32x3u w = STREAM ? __builtin_nontemporal_load(q) : *q;
    v.x = w.x, v.y = w.y, v.z = w.z;
  } else if (count == 2) {
    const f32x2u* q = reinterpret_cast<const f32x2u*>(p);
    const f32x2u w = STREAM ? __builtin_nontemporal_load(q) : *q;
    v.x = w.x, v.y = w.y;
  } else {
    v.x = STREAM ? __builtin_nontemporal_load(p) : *p;
  }
  return v;
}
template <bool STREAM>
__device__ __forceinline__ void store_part(f32x4 v, float* p, unsigned count) {
  if (count == 4) {
    store_quad<STREAM>(v, p);
  } else if (count == 3) {
    f32x3u* q = reinterpret_cast<f32x3u*>(p);
    const f32x3u w = {v.x, v.y, v.z};
    if (STREAM) __builtin_nontemporal_store(w, q); else *q = w;
  } else if (count == 2) {
    f32x2u* q = reinterpret_cast<f32x2u*>(p);
    const f32x2u w = {v.x, v.y};
    if (STREAM) __builtin_nontemporal_store(w, q); else *q = w;
  } else {
    if (STREAM) __builtin_nontemporal_store(v.x, p); else *p = v.x;
  }
}

// FIXED rows: one quad per lane. `quads` = ceil(k/4) per row, `rest` = k mod 4 floats in a row's last one
// (REST: not zero). A row's quads are its own, so a lane deals with one row whatever k is. (Rows with a
// rest used to go float by float, four 32-bit accesses and four divisions per lane: 500,000 rows of 33
// floats 78 us to accumulate and 47 to gather, now 49 and 35; 160 rows of 825,153 floats 1.39 times faster.)
template <int OP, bool STREAM, bool REST>
__device__ __forceinline__ void rows_quads_fixed(const RowsParams& p, uint64_t q0, uint64_t q_end) {
  // a refused push (it repeats a key) changes no stored value; rows it created stay, as zero rows
  const bool rejected = OP == kOpAcc && p.st->refused_epoch == p.tag.epoch;
  const uint64_t quads = (p.k + 3) >> 2;
  const unsigned rest = REST ? (unsigned)p.k & 3u : 0u;
  const bool live = threadIdx.x < q_end - q0;
  f32x4 x = (f32x4)(0.f);
  // Without a rest the request side depends on nothing but the quad's number: asked for first, so that
  // it is in flight while the row reference is fetched.
  if (OP == kOpAcc && !REST && live) x = load_quad<STREAM>(p.req + (q0 + threadIdx.x) * 4);
  // one division per workgroup; a lane is at most kBlock quads further on
  const uint64_t row0 = q0 / quads;
  const uint64_t c0 = q0 - row0 * quads + threadIdx.x;
  uint64_t over, c;
  if (quads >= kBlock) {
    over = c0 >= quads ? 1u : 0u;
    c = over ? c0 - quads : c0;
  } else {
    const unsigned o32 = (unsigned)c0 / (unsigned)quads;
    over = o32;
    c = (unsigned)c0 - o32 * (unsigned)quads;
  }
  if (!live) return;
  const uint64_t row = row0 + over;
  const unsigned count = REST && c + 1 == quads ? rest : 4u;
  float* side = p.req + row * p.k + c * 4;
  // (a shorter quad is read whole: what follows it is other rows, or the room behind the last row of the
  // arena; only the end of the request's values is the end of what may be read)
  if (OP == kOpAcc && REST)
    x = count == 4 || whole_quads(row + 1, p.k, p.n) ? load_quad<STREAM>(side) : load_part<STREAM>(side, rest);
  const uint64_t r = p.ref[row];
  if (r == kRefAbsent) return;  // a key the lookup refused (duplicate in the request, full table)
  const bool fresh = (r & kRefNew) != 0 && !p.ignore_new;
  float* dst = p.arena + (r & ~kRefNew) * p.k + c * 4;
  f32x4 y = (f32x4)(0.f);
  if (!fresh) y = load_quad<STREAM>(dst);
  if (OP == kOpAcc) {
    if (rejected) {
      if (!fresh) return;
    } else {
      y = y + x;  // a created row is a zero row first (0.0f + v), kv_app.h:454
    }
    if (!REST || count == 4) store_quad<STREAM>(y, dst); else store_part<STREAM>(y, dst, rest);
  } else {
    if (!REST || count == 4) store_quad<STREAM>(y, side); else store_part<STREAM>(y, side, rest);
    if (fresh) {  // pull created the row: zeros
      if (!REST || count == 4) store_quad<STREAM>(y, dst); else store_part<STREAM>(y, dst, rest);
    }
  }
}

// The same for rows of kWideRow floats and more, which a workgroup meets one or two of. Bound by memory, as long as a wavefront asks
// early: all arguments in one fetch, then the request's values, then the two references, through the scalar cache, so that nothing
// waits for anything but the row for its reference. Above, arguments, facts and reference are four waits one behind the other
// and the values are waited for with the reference: 64 rows of 4M floats, four pushes and a pull of three tables in turn, 2,460 us
// against 2,395 here (6.1 and 6.3 TB/s), 300 of 100,010 318 and 308, 3 of 4.9M 178 and 170. Pulls by themselves gain less: 300
// rows of 100,010 41.2 and 39.0, 3 of 4.9M 20.9 and 20.0, 5,000 of 4,100 28.3 and 27.5, 64 of 4M 334 both. Shorter rows, scattered over the
// arena, gain nothing from it (64 floats 633 and 634-639, 48 floats 158 and 161: the memory has enough to do).
constexpr uint64_t kWideRow = 1024;
typedef const __attribute__((address_space(4))) uint64_t* ScalarWords;  // what no workgroup of this launch writes
template <int OP, bool STREAM, bool REST>
__device__ __forceinline__ void rows_quads_wide(const TableReq& d, uint64_t q0) {
  // (asked for first, and not waited for before the references have come)
  unsigned long long same_epoch = d.st->same_epoch, refused = OP == kOpAcc ? d.st->refused_epoch : 0ull;
  const uint64_t quads = (d.k + 3) >> 2;
  const unsigned rest = REST ? (unsigned)d.k & 3u : 0u;
  if (threadIdx.x >= d.ntiles - q0) return;
  f32x4 x = (f32x4)(0.f);
  if (OP == kOpAcc && !REST) x = load_quad<STREAM>(d.req + (q0 + threadIdx.x) * 4);
  const uint64_t row0 = q0 / quads;
  const uint64_t c0 = q0 - row0 * quads + threadIdx.x;
  const bool over = c0 >= quads;
  const ScalarWords refs = (ScalarWords)reinterpret_cast<uintptr_t>(d.ref);
  uint64_t ra = refs[row0], rb = refs[row0 + 1 < d.n ? row0 + 1 : row0];
  const uint64_t row = row0 + (over ? 1u : 0u), c = over ? c0 - quads : c0;
  const unsigned count = REST && c + 1 == quads ? rest : 4u;
  float* side = d.req + row * d.k + c * 4;
  if (OP == kOpAcc && REST)  // (as in rows_quads_fixed)
    x = count == 4 || whole_quads(row + 1, d.k, d.n) ? load_quad<STREAM>(side) : load_part<STREAM>(side, rest);
  asm volatile("" : "+" PSKV_SCALAR(ra), "+" PSKV_SCALAR(rb), "+v"(same_epoch), "+v"(refused));
  const uint64_t r = over ? rb : ra;
  const bool same = same_epoch == d.tag.epoch;
  if (d.tag.replay && !same) return;
  if (r == kRefAbsent) return;  // a key the lookup refused (duplicate in the request, full table)
  const bool rejected = OP == kOpAcc && refused == d.tag.epoch;
  const bool fresh = (r & kRefNew) != 0 && !d.ignore_new && !same;
  float* dst = d.arena + (r & ~kRefNew) * d.k + c * 4;
  f32x4 y = (f32x4)(0.f);
  if (!fresh) y = load_quad<STREAM>(dst);
  if (OP == kOpAcc) {
    if (rejected) {
      if (!fresh) return;
    } else {
      y = y + x;  // a created row is a zero row first (0.0f + v), kv_app.h:454
    }
    if (!REST || count == 4) store_quad<STREAM>(y, dst); else store_part<STREAM>(y, dst, rest);
  } else {
    if (!REST || count == 4) store_quad<STREAM>(y, side); else store_part<STREAM>(y, side, rest);
    if (fresh) {  // pull created the row: zeros
      if (!REST || count == 4) store_quad<STREAM>(y, dst); else store_part<STREAM>(y, dst, rest);
    }
  }
}

// VARLEN rows: a WAVEFRONT owns WTILE consecutive request-side floats. The tile table names
// the first key that overlaps them; the wavefront stages the offsets and row references of
// the keys that overlap its tile in its own piece of LDS (no workgroup barrier: the four
// wavefronts of a workgroup never wait for each other) and finds the row of each element by
// binary search there. Tiles that overlap more than kWaveSpan keys (rows of a float or two)
// search the global arrays instead.
constexpr unsigned kWaveSpan = 128;

// What a wavefront can ask for knowing nothing but its tile index: the tile's shortcut note (read
// even when it turns out not to be needed, so that it is not a second round trip after the
// decision) and the request-side values. `bound` is what the host knows of the request's
// length; the data may be shorter.
template <int OP, bool STREAM>
__device__ __forceinline__ void rows_wave_ask(const RowsParams& p, uint64_t bound, f32x4& x, TileNote& aff) {
  const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t wt = (uint64_t)p.blk * (kBlock / 64) + wave;
  const uint64_t f0 = wt * kTileVar;
  const uint64_t left = bound > f0 ? bound - f0 : 0;  // 0: the tile lies past the data
  const uint32_t floats = (uint32_t)(left < (uint64_t)kTileVar ? left : (uint64_t)kTileVar);
  aff.first = kTileNotAffine;
  aff.second = 0;
  if (left && p.tag.try_cache) {
    const u64x2 w = *reinterpret_cast<const u64x2*>(&p.tile_aff[wt]);  // one 128-bit load
    aff.first = w.x;
    aff.second = w.y;
  }
  x = (f32x4)(0.f);
  if (OP == kOpAcc) {
    const uint32_t lf = lane * 4;
    if (lf + 4 <= floats) {
      x = load_quad<STREAM>(p.req + f0 + lf);
    } else if (lf < floats) {  // the end of the request
      x = load_part<STREAM>(p.req + f0 + lf, floats - lf);
    }
  }
}

// Shortcut of a request that repeats the cached one: if the rows of this tile lie in the arena
// as one or two unbroken pieces (two: the tile straddles the rows of two workgroups of the
// lookup that created them), the note the row kernel of the cached request left maps every
// float with an offset and neither the row table nor a search is needed. Returns false when the
// tile has to take the general way. Wavefront-uniform.
template <int OP, bool STREAM>
__device__ __forceinline__ bool rows_wave_affine(const RowsParams& p, uint64_t total, const f32x4& x,
                                                 const TileNote& aff) {
  static_assert(kTileVar < (1u << kTileSplitBits), "the split index does not fit the note");
  if (aff.first == kTileNotAffine) return false;
  const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t f0 = ((uint64_t)p.blk * (kBlock / 64) + wave) * kTileVar;
  if (f0 >= total) return true;
  const uint32_t lf = lane * 4;
  if (lf >= (total - f0 < (uint64_t)kTileVar ? (uint32_t)(total - f0) : kTileVar)) return true;
  // rows start on multiples of four floats here, so no quad straddles the split
  const uint32_t split = aff.second ? (uint32_t)(aff.second & ((1u << kTileSplitBits) - 1)) : ~0u;
  const int64_t first = (int64_t)aff.first;
  const int64_t second = (int64_t)(aff.second >> kTileSplitBits) - kTileNoteBias;  // may be negative
  float* dst = p.arena + ((lf >= split ? second : first) + (int64_t)lf);
  const f32x4 y = load_quad<STREAM>(dst);
  if (OP == kOpAcc) {
    store_quad<STREAM>(y + x, dst);
  } else {
    store_quad<STREAM>(y, p.req + f0 + lf);
  }
  return true;
}

// The second half of it: moves the tile's floats. STAGED: offsets and references lie in LDS (all of it in 32 bits:
// a row is shorter than 2^28 floats), else where they were.
template <int OP, bool RAGGED, bool STREAM, bool STAGED>
__device__ __forceinline__ void rows_wave_move(const RowsParams& p, uint64_t f0, uint32_t tile_floats, uint64_t j_lo,
                                               uint32_t span, const int32_t* s_off, const uint64_t* s_ref, bool rejected,
                                               const f32x4& x) {
  const unsigned lane = threadIdx.x & 63;
  const uint32_t lf = lane * 4;
  if (lf >= tile_floats) return;
  // offsets (from the tile's first float; those of a row that ends far behind the tile are cut off) and references
  // of the keys that overlap the tile
  auto off_of = [&](uint32_t s) -> int32_t {
    if (STAGED) return s_off[s];
    const int64_t o = (int64_t)(p.off[j_lo + s] - f0);
    return (int32_t)(o < (int64_t)PSKV_MAX_VARLEN_ROW * 2 ? o : (int64_t)PSKV_MAX_VARLEN_ROW * 2);
  };
  auto ref_of = [&](uint32_t s) { return STAGED ? s_ref[s] : p.ref[j_lo + s]; };
  auto place = [&](uint64_t r, int32_t within) {
    return p.arena + (((r & ~kRefNew) >> kLenBits) << 2) + within;
  };
  // the key that holds the quad's first float: the last one whose first float is at or before it
  // (zero-length rows repeat an offset)
  uint32_t lo = 0, hi = span;
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (off_of(mid) <= (int32_t)lf) lo = mid + 1; else hi = mid;
  }
  const uint64_t r = ref_of(lo - 1);
  float* dst = place(r, (int32_t)lf - off_of(lo - 1));
  // a key the lookup refused (duplicate in the request, full table) is neither read nor written
  const bool here = r != kRefAbsent;
  const bool fresh = (r & kRefNew) != 0 && !p.ignore_new;
  float* side = p.req + f0 + lf;
  if (!RAGGED) {
    if (!here) return;
    f32x4 y = (f32x4)(0.f);
    if (!fresh) y = load_quad<STREAM>(dst);
    if (OP == kOpGather) {
      store_quad<STREAM>(y, side);
    } else if (!rejected) {
      store_quad<STREAM>(y + x, dst);  // a created row is a zero row first (0.0f + v)
    } else if (fresh) {
      // a refused push changes no stored value; rows it created stay, as zero rows
      store_quad<STREAM>(y, dst);
    }
    return;
  }
  const uint32_t upto = tile_floats - lf < 4u ? tile_floats - lf : 4u;
  const int32_t end = off_of(lo);
  const uint32_t count = end - (int32_t)lf < (int32_t)upto ? (uint32_t)(end - (int32_t)lf) : upto;
  // the next row, when the quad reaches into it
  uint64_t r2 = kRefAbsent;
  float* dst2 = nullptr;
  uint32_t two = upto;  // floats of the quad that the two rows hold
  if (count < upto) {
    uint32_t key = lo;  // (zero-length rows are stepped over; the key table closes with the end of the request)
    while (off_of(key + 1) <= end) ++key;
    r2 = ref_of(key);
    dst2 = place(r2, 0);
    const int32_t end2 = off_of(key + 1);
    if (end2 - (int32_t)lf < (int32_t)upto) two = (uint32_t)(end2 - (int32_t)lf);
  }
  const bool here2 = r2 != kRefAbsent;
  const bool fresh2 = (r2 & kRefNew) != 0 && !p.ignore_new;
  if (two == upto) {
    // (reading a quad whole is safe: what follows its row is another row, or the room behind the arena's last)
    f32x4 y = (f32x4)(0.f), y2 = (f32x4)(0.f);
    if (here && !fresh) y = load_quad<false>(dst);
    if (here2 && !fresh2) y2 = load_quad<false>(dst2);
    if (OP == kOpGather) {
      f32x4 v = y;
      if (count == 1) v.y = y2.x, v.z = y2.y, v.w = y2.z;
      if (count == 2) v.z = y2.x, v.w = y2.y;
      if (count == 3) v.w = y2.x;
      if (upto == 4 && here && (here2 || count == 4)) {
        store_quad<STREAM>(v, side);
      } else {
        if (here) store_part<false>(y, side, count);
        if (here2) store_part<false>(y2, side + count, upto - count);
      }
      return;
    }
    if (here && (!rejected || fresh)) store_part<false>(rejected ? y : y + x, dst, count);
    if (here2 && (!rejected || fresh2)) {
      f32x4 x2 = x;
      if (count == 1) x2.x = x.y, x2.y = x.z, x2.z = x.w;
      if (count == 2) x2.x = x.z, x2.y = x.w;
      if (count == 3) x2.x = x.w;
      store_part<false>(rejected ? y2 : y2 + x2, dst2, upto - count);
    }
    return;
  }
  // three rows or more
  float* at[4];
  float cur[4];
  bool made[4];
  uint32_t key = lo - 1;
#pragma unroll
  for (uint32_t e = 0; e < 4; ++e) {
    at[e] = nullptr;
    made[e] = false;
    if (e >= upto) continue;
    while (off_of(key + 1) <= (int32_t)(lf + e)) ++key;
    const uint64_t q = ref_of(key);
    if (q == kRefAbsent) continue;
    made[e] = (q & kRefNew) != 0 && !p.ignore_new;
    at[e] = place(q, (int32_t)(lf + e) - off_of(key));
  }
#pragma unroll
  for (uint32_t e = 0; e < 4; ++e) cur[e] = at[e] && !made[e] ? *at[e] : 0.f;
#pragma unroll
  for (uint32_t e = 0; e < 4; ++e) {
    if (!at[e]) continue;
    if (OP == kOpGather) {
      side[e] = cur[e];
    } else if (!rejected) {
      *at[e] = cur[e] + x[e];
    } else if (made[e]) {
      *at[e] = cur[e];
    }
  }
}

// `x` comes from rows_wave_ask; it is used only below `total`. RAGGED: some row's length is not a
// multiple of four, so a quad may hold the end of one row and the start of the next (rows themselves
// start on multiples of four floats in the arena). The part in the row of its first float and the part in
// the next row are one access each, both asked for before either is used; where rows of one or two floats
// make it more than two parts, the floats are moved one by one, their loads together. (Every float used to
// be looked up and moved on its own.) The arena side of such rows is read and written through the caches
// whatever the size of the request: a 128-byte line holds pieces of several rows, and lines that are
// written piecewise past the caches cost a third of the bandwidth (1M rows of 1 to 60 floats: 345 us per
// push + pull against 221).
template <int OP, bool RAGGED, bool STREAM>
__device__ __forceinline__ void rows_wave_varlen(const RowsParams& p, uint64_t total,
                                                 int32_t* s_off_all, uint64_t* s_ref_all,
                                                 bool rejected, bool same, const f32x4& x) {
  const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t wt = (uint64_t)p.blk * (kBlock / 64) + wave;
  const uint64_t f0 = wt * kTileVar;
  if (f0 >= total) return;  // the whole wavefront leaves; nothing below synchronises workgroups
  const uint32_t tile_floats = (uint32_t)((total - f0 < (uint64_t)kTileVar) ? (total - f0) : (uint64_t)kTileVar);

  const uint64_t j_lo = p.tile_key[wt];
  const uint32_t span = (uint32_t)((uint64_t)p.tile_key[wt + 1] - j_lo + 1);
  const bool staged = span <= kWaveSpan;
  int32_t* s_off = s_off_all + wave * (kWaveSpan + 1);
  uint64_t* s_ref = s_ref_all + wave * kWaveSpan;
  if (staged) {
    for (uint32_t s = lane; s <= span; s += 64) {
      uint64_t at = p.off[j_lo + s], r = p.ref[j_lo + (s < span ? s : span - 1)];  // (one trip, not two)
      arrived(at), arrived(r);
      s_off[s] = (int32_t)(int64_t)(at - f0);
      if (s < span) s_ref[s] = r;
    }
    // the wavefront's own LDS writes, visible to all of its lanes before the reads below
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  if (!same && !RAGGED) {  // (nobody looks at the notes of a request with ragged rows)
    // Leave a note for requests that repeat this one. Every row with floats in the tile has a
    // distance between its place in the arena and its place in the request; the tile is one
    // piece when all distances are equal (the rows lie back to back, in request order, without
    // padding between them) and two pieces when they change once.
    TileNote note = {kTileNotAffine, 0};
    if (staged) {
      bool absent = false;
      int64_t d[(kWaveSpan + 63) / 64];
      bool has[(kWaveSpan + 63) / 64];
#pragma unroll
      for (uint32_t it = 0; it < (kWaveSpan + 63) / 64; ++it) {
        const uint32_t s = it * 64 + lane;
        has[it] = s < span && s_off[s + 1] > s_off[s] && s_off[s] < (int32_t)tile_floats;
        d[it] = 0;
        if (has[it]) {
          const uint64_t r = s_ref[s];
          absent |= r == kRefAbsent;
          d[it] = (int64_t)(((r & ~kRefNew) >> kLenBits) << 2) - (int64_t)s_off[s];
        }
      }
      // the first row with floats, its distance, and the first row whose distance differs
      uint32_t s0 = ~0u, s1 = ~0u;
#pragma unroll
      for (uint32_t it = 0; it < (kWaveSpan + 63) / 64; ++it) {
        const uint64_t m = __ballot(has[it]);
        if (s0 == ~0u && m) s0 = it * 64 + (uint32_t)__builtin_ctzll(m);
      }
      if (s0 != ~0u && __ballot(absent) == 0ull) {
        const uint64_t r0 = s_ref[s0];
        const int64_t d0 = (int64_t)(((r0 & ~kRefNew) >> kLenBits) << 2) - (int64_t)s_off[s0];
#pragma unroll
        for (uint32_t it = 0; it < (kWaveSpan + 63) / 64; ++it) {
          const uint64_t m = __ballot(has[it] && d[it] != d0);
          if (s1 == ~0u && m) s1 = it * 64 + (uint32_t)__builtin_ctzll(m);
        }
        if (s1 == ~0u) {
          note.first = (uint64_t)d0;
        } else {
          const uint64_t r1 = s_ref[s1];
          const int32_t at = s_off[s1];  // > 0: row s0 comes first and has floats in the tile
          const int64_t d1 = (int64_t)(((r1 & ~kRefNew) >> kLenBits) << 2) - (int64_t)at;
          bool other = false;
#pragma unroll
          for (uint32_t it = 0; it < (kWaveSpan + 63) / 64; ++it)
            other |= has[it] && it * 64 + lane > s1 && d[it] != d1;
          if (__ballot(other) == 0ull && at > 0) {
            note.first = (uint64_t)d0;
            note.second = ((uint64_t)(d1 + kTileNoteBias) << kTileSplitBits) | (uint64_t)(uint32_t)at;
          }
        }
      }
    }
    if (lane == 0) p.tile_aff[wt] = note;
  }

  if (staged) {
    rows_wave_move<OP, RAGGED, STREAM, true>(p, f0, tile_floats, j_lo, span, s_off, s_ref, rejected, x);
  } else {
    rows_wave_move<OP, RAGGED, STREAM, false>(p, f0, tile_floats, j_lo, span, s_off, s_ref, rejected, x);
  }
}

// Ragged rows of a push, the other way round: 2^shift lanes a row (as many as it takes, by the host's reckoning, ragged_by_row),
// a lane a quad of it, kTurns turns asked for together. A wavefront that starts from its tile makes five trips to memory that follow
// from each other (facts, tile table, offsets and references, rows, values), one that starts from its rows two: what it needs of the offsets
// and references is asked for with the facts (behind them the kernel took 27.3 us where it takes 25.8). Its
// accesses to the arena are whole quads on their own boundaries (the end of a row's last one is nobody's), where a tile's
// straddle them. Bound by the lines of the rows, which lie scattered: 200,000 of 600,000 rows of 1 to 100 floats 31.8 -> 25.8 us,
// of 1 to 16 10.6 -> 8.9. Not for pulls (30 -> 33: their stores would be the ones that straddle), and not
// where a row is far longer than the others, whose wavefront everybody would wait for.
struct RowOfLane {
  uint64_t first, end, ref;  // kRefAbsent behind the last row
};
__device__ __forceinline__ RowOfLane row_of_lane(const RowsParams& p, unsigned shift) {
  const uint64_t wave = (uint64_t)p.blk * (kBlock / 64) + (threadIdx.x >> 6);
  const uint64_t row = (wave << (6 - shift)) + ((threadIdx.x & 63) >> shift);
  if (row >= p.n) return RowOfLane{0, 0, kRefAbsent};
  return RowOfLane{p.off[row], p.off[row + 1], p.ref[row]};
}
template <bool STREAM, unsigned kTurns>
__device__ __forceinline__ void rows_by_row(const RowsParams& p, uint64_t total, unsigned shift, const RowOfLane& mine, bool rejected) {
  const unsigned lane = threadIdx.x & 63, lanes = 1u << shift;
  const uint64_t first = mine.first, end = mine.end, r = mine.ref;
  if (r == kRefAbsent) return;  // a key the lookup refused
  const bool fresh = (r & kRefNew) != 0 && !p.ignore_new;
  if (rejected && !fresh) return;
  const uint32_t len = (uint32_t)(end - first), quads = (len + 3) >> 2;
  float* dst = p.arena + (((r & ~kRefNew) >> kLenBits) << 2);
  const float* side = p.req + first;
  for (uint32_t q0 = lane & (lanes - 1); q0 < quads; q0 += kTurns * lanes) {
    f32x4 x[kTurns], y[kTurns];
#pragma unroll
    for (unsigned u = 0; u < kTurns; ++u) {
      const uint32_t q = q0 + u * lanes;
      x[u] = y[u] = (f32x4)(0.f);
      if (q >= quads) continue;
      if (!fresh) y[u] = load_quad<false>(dst + q * 4);
      if (!rejected)  // (what follows a row's last float is the next row, but for the last row's)
        x[u] = first + q * 4 + 4 <= total ? load_quad<STREAM>(side + q * 4) : load_part<STREAM>(side + q * 4, len - q * 4);
    }
#pragma unroll
    for (unsigned u = 0; u < kTurns; ++u) {
      const uint32_t q = q0 + u * lanes, left = len - q * 4;
      if (q >= quads) continue;
      f32x4 sum = rejected ? y[u] : y[u] + x[u];  // a created row is a zero row first (0.0f + v)
      if (left < 2) sum.y = y[u].y;
      if (left < 3) sum.z = y[u].z;
      if (left < 4) sum.w = y[u].w;
      store_quad<false>(sum, dst + q * 4);
    }
  }
}

// Quads per workgroup (fixed rows) and request-side floats per wavefront (var-len rows). One
// 128-bit access per lane and many small workgroups stream fastest on this GPU (6.5 TB/s for
// `row += in` against 5.5 TB/s with four accesses per lane).
constexpr unsigned kQuadsFixed = kBlock;
constexpr unsigned kRowsVarPerBlock = kTileVar * (kBlock / 64);

// Behind k_var_push_start and k_var_pull_start (one_launch.h): takes away what their workgroups have told each other, and
// leaves the counter record that the host asked for. One workgroup.
__device__ __forceinline__ void finish_start(const TableReq& d) {
  for (unsigned i = threadIdx.x; i < d.started; i += kBlock) d.st->parts[i] = 0ull;
  if (d.snap && threadIdx.x < 64) publish_snapshot(d.st, d.snap, d.snap_seq);
}

// STARTED: VARLEN, behind one of those two kernels. (A kernel of its own: with the end of such a request in the way of the
// others, 2M rows over 16 tables took 374 us to push and pull, not 357.)
// BY_ROW: a push in which the host takes some table's rows to be ragged.
template <int OP, bool VARLEN, bool STREAM, bool STARTED, bool BY_ROW, int TABLES>
__global__ __launch_bounds__(kBlock) void k_rows(ReqBatch<TABLES> b) {
  const TableReq& d = b.t[blockIdx.y];
  // the grid is sized for the largest table of the launch: workgroups (VARLEN: wavefronts) past
  // this table's floats leave before they touch anything
  const bool by_row = BY_ROW && d.ragged != 0;
  unsigned blk = blockIdx.x;
  if (VARLEN) {
    // every argument the common path uses, asked for at once (the compiler otherwise fetches them group by group where they
    // are first used, one wait each)
    PSKV_ASK_ARGS_FOR(blk, "s"(d.tile_base), "s"(d.total), "s"(d.st), "s"(d.req), "s"(d.arena), "s"(d.tile_aff), "s"(d.total_on_device),
        "s"(d.tag.epoch), "s"(d.tag.try_cache), "s"(d.tag.replay), "s"(d.ignore_new), "s"(d.ref), "s"(d.off), "s"(d.tile_key), "s"(d.n));
    const bool behind = by_row ? blk + (STARTED && d.started ? 1u : 0u) >= d.nblk
                               : (((uint64_t)blk + d.tile_base) * (kBlock / 64) + (threadIdx.x >> 6)) * kTileVar >= d.total;
    if (behind) {
      if (STARTED && d.started && blockIdx.x == d.nblk - 1) finish_start(d);  // (a workgroup behind the last one with floats)
      return;
    }
  } else {
    if (d.nvals + (uint64_t)blockIdx.x * kQuadsFixed >= d.ntiles) return;
  }
  RowsParams p;
  p.req = d.req;
  p.arena = d.arena;
  p.ref = d.ref;
  p.off = d.off;
  p.tile_key = d.tile_key;
  p.tile_aff = d.tile_aff;
  p.st = d.st;
  p.n = d.n;
  p.total = d.total;
  p.k = d.k;
  p.ignore_new = d.ignore_new;
  p.total_on_device = d.total_on_device;
  p.blk = blk + d.tile_base;
  p.tag = d.tag;
  __shared__ int32_t s_off[VARLEN ? (kWaveSpan + 1) * (kBlock / 64) : 1];
  __shared__ uint64_t s_ref[VARLEN ? kWaveSpan * (kBlock / 64) : 1];
  // What the device knows about the request: one load, one wait per wavefront.
  const ReqFacts facts = load_req_facts(p.st);
  const unsigned long long refused = STARTED && OP == kOpAcc ? p.st->refused_epoch : 0ull;
  if (VARLEN) {
    // the grid covers the room in the caller's buffer, which may be more than the data; the loads
    // that need no facts are on their way before the facts are looked at
    uint64_t total = p.total;
    f32x4 x;
    TileNote aff = {kTileNotAffine, 0};
    RowOfLane mine;
    if (by_row) mine = row_of_lane(p, by_row_shift(d.ragged)); else rows_wave_ask<OP, STREAM>(p, total, x, aff);
    // a request served from the cached references creates nothing and cannot have been refused
    const bool same = facts.same_epoch == p.tag.epoch;
    if (p.tag.replay && !same) return;
    if (same) p.ignore_new = 1;
    const unsigned err = same ? 0u : facts.req_error;
    if (err & (kDevErrBadLen | kDevErrSizeMismatch | kDevErrDuplicate)) return;
    const bool rejected =
        (err & kDevErrLenChanged) != 0 || (STARTED && OP == kOpAcc && refused == p.tag.epoch);
    if (p.total_on_device) {
      total = facts.scan_total;
      if (total > p.total) {  // the response does not fit the caller's buffer: write nothing
        if (p.blk == 0 && threadIdx.x == 0) atomicOr(&p.st->error, kDevErrNoRoom);
        return;
      }
    }
    if (by_row) {
      if ((facts.misaligned & kReqMisaligned) && !(facts.misaligned & kReqLong)) {
        if (d.ragged & kByRowThree)
          rows_by_row<STREAM, 3>(p, total, by_row_shift(d.ragged), mine, rejected);
        else
          rows_by_row<STREAM, 2>(p, total, by_row_shift(d.ragged), mine, rejected);
        return;
      }
      rows_wave_ask<OP, STREAM>(p, total, x, aff);  // (the host was wrong)
    }
    if (facts.misaligned & kReqMisaligned) {
      rows_wave_varlen<OP, true, STREAM>(p, total, s_off, s_ref, rejected, same, x);
    } else {
      if (same && rows_wave_affine<OP, STREAM>(p, total, x, aff)) return;
      rows_wave_varlen<OP, false, STREAM>(p, total, s_off, s_ref, rejected, same, x);
    }
  } else {
    if (p.tag.replay && facts.same_epoch != p.tag.epoch) return;
    if (facts.same_epoch == p.tag.epoch) p.ignore_new = 1;
    const uint64_t q0 = d.nvals + (uint64_t)blockIdx.x * kQuadsFixed;
    if (p.k & 3) {
      // (short rows share 128-byte lines with their neighbours, which lie in other workgroups' hands: lines
      // written piecewise past the caches made rows of 33 floats a third slower)
      if (p.k >= 1024) {
        rows_quads_fixed<OP, STREAM, true>(p, q0, d.ntiles);
      } else {
        rows_quads_fixed<OP, false, true>(p, q0, d.ntiles);
      }
    } else {
      rows_quads_fixed<OP, STREAM, false>(p, q0, d.ntiles);
    }
  }
}

template <int OP, bool STREAM, int TABLES>
__global__ __launch_bounds__(kBlock) void k_rows_wide(ReqBatch<TABLES> b) {
  const TableReq& d = b.t[blockIdx.y];
  unsigned blk = blockIdx.x;
  // (the arguments asked for at once: fetched group by group where they are first used, each group is a wait)
  PSKV_ASK_ARGS_FOR(blk, "s"(d.nvals), "s"(d.ntiles), "s"(d.req), "s"(d.arena), "s"(d.ref), "s"(d.st), "s"(d.n), "s"(d.k),
      "s"(d.ignore_new), "s"(d.tag.epoch), "s"(d.tag.replay));
  const uint64_t q0 = d.nvals + (uint64_t)blk * kQuadsFixed;
  if (q0 >= d.ntiles) return;
  if (d.k & 3) {
    rows_quads_wide<OP, STREAM, true>(d, q0);
  } else {
    rows_quads_wide<OP, STREAM, false>(d, q0);
  }
}

// ---------------------------------------------------------------------------------
// Maintenance kernels.
// ---------------------------------------------------------------------------------

// Growth, the general way: every live slot of the old array is re-inserted into the new one
// (which starts as all ones); payloads move bit for bit, so stored sums are unchanged.
__global__ __launch_bounds__(kBlock) void k_rehash(const Slot* __restrict__ old_slots,
                                                  uint64_t old_cap, Slot* __restrict__ slots,
                                                  uint64_t mask, DevState* st) {
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < old_cap; i += stride) {
    const ulonglong2 s = *reinterpret_cast<const ulonglong2*>(&old_slots[i]);
    if (s.x == kEmptyKey) continue;
    uint64_t h = home_slot(s.x, mask);
    bool placed = false;
    for (uint64_t probes = 0; probes <= mask; ++probes) {
      if (slots[h].key == kEmptyKey) {
        unsigned long long old =
            atomicCAS(reinterpret_cast<unsigned long long*>(&slots[h].key),
                      (unsigned long long)kEmptyKey, (unsigned long long)s.x);
        if (old == kEmptyKey) {
          slots[h].payload = s.y;
          placed = true;
          break;
        }
      }
      h = (h + 1) & mask;
    }
    if (!placed) atomicOr(&st->error, kDevErrFull);
  }
}

// Growth by a small power of two G, as two streaming passes instead of a scatter. A key's home
// slot is the top bits of its hash, so the keys whose homes lie in the old slots [a, a + R) are
// exactly the keys whose new homes lie in [G * a, G * (a + R)): one workgroup builds that
// stretch of the new array in LDS from its R old slots and writes it out whole, empty slots
// included, with coalesced 128-bit stores (the new array needs no fill, and no atomics reach
// memory). What it cannot place there is left for the second pass: keys that sit in its old
// slots but have their home in an earlier stretch (a probe chain that crossed the boundary, or
// wrapped around the end of the array), and keys whose probe chain would leave the LDS stretch.
// The workgroup writes those, packed, over the front of its own old slots (it is the only one
// that reads them) with an empty slot behind the last; k_regrow_rest inserts them the general
// way once every stretch of the new array is in place. At a fill of one half about one key in
// 250 takes the second pass. Payloads move bit for bit.
// One launch serves all tables of a request that grow (blockIdx.y): four tables of 64 MB each, one after the other, took
// 51 + 5.5 us and the gaps of two launches for each of them (20 pushes of 1M new keys into four tables 2,003 -> 1,966 us).
constexpr int kRegrowOld = kBlock;  // old slots per workgroup, one per thread
constexpr int kRegrowMaxFactor = 8;
struct RegrowOf {
  Slot* old_slots;
  Slot* slots;
  uint64_t old_mask, mask;
  DevState* st;
  uint64_t factor;
  uint64_t stretch;  // old slots per workgroup: a multiple of kRestLanes
};
struct RegrowBatch {
  RegrowOf t[kMaxBatch];
};
__global__ __launch_bounds__(kBlock) void k_regrow(RegrowBatch b) {
  extern __shared__ unsigned long long regrow_lds[];  // keys of the stretch, then its payloads
  const RegrowOf& d = b.t[blockIdx.y];
  Slot* __restrict__ old_slots = d.old_slots;
  Slot* __restrict__ slots = d.slots;
  const uint64_t old_mask = d.old_mask, mask = d.mask;
  const unsigned factor = (unsigned)d.factor;
  if ((uint64_t)blockIdx.x * kRegrowOld > old_mask) return;  // (the grid is as wide as the largest table needs)
  const unsigned T = kRegrowOld * factor;
  unsigned long long* tkey = regrow_lds;
  unsigned long long* tpay = regrow_lds + T;
  __shared__ unsigned long long red[kBlock / 64 + 1];
  const uint64_t a = (uint64_t)blockIdx.x * kRegrowOld;
  const uint64_t A = a * factor;
  const u64x2 s = __builtin_nontemporal_load(reinterpret_cast<const u64x2*>(&old_slots[a + threadIdx.x]));
  for (unsigned j = threadIdx.x; j < T; j += kBlock) {
    tkey[j] = kEmptyKey;
    tpay[j] = kPayloadUnset;
  }
  __syncthreads();
  const bool live = s.x != kEmptyKey;
  bool rest = false;
  if (live) {
    const uint64_t oh = home_slot(s.x, old_mask);
    if (oh >= a && oh <= a + threadIdx.x) {
      unsigned j = (unsigned)(home_slot(s.x, mask) - A);
      rest = true;
      for (; j < T; ++j) {
        if (atomicCAS(&tkey[j], (unsigned long long)kEmptyKey, (unsigned long long)s.x) == kEmptyKey) {
          tpay[j] = s.y;
          rest = false;
          break;
        }
      }
    } else {
      rest = true;  // its home lies in another workgroup's stretch
    }
  }
  unsigned long long total;
  const unsigned long long at = block_excl_scan_u64(rest ? 1ull : 0ull, red, total);  // (two barriers)
  u64x2* out = reinterpret_cast<u64x2*>(slots + A);
  for (unsigned j = threadIdx.x; j < T; j += kBlock) {
    u64x2 v;
    v.x = tkey[j];
    v.y = tpay[j];
    __builtin_nontemporal_store(v, &out[j]);
  }
  // every thread has read its old slot (the barriers of the scan lie in between)
  if (rest) *reinterpret_cast<u64x2*>(&old_slots[a + at]) = s;
  if (threadIdx.x == 0 && total < (unsigned long long)kRegrowOld) old_slots[a + total].key = kEmptyKey;
}

// Second pass of a growth: sixteen lanes per stretch of old slots read the keys the first pass left at its front, up to the
// first empty slot, and insert them the general way. A key that a pushed request has created in the new array meanwhile
// (k_stream_push) gets both values: what was pushed came to 0.0f + v, and a stored value is never -0.0f.
constexpr int kRestLanes = 16;
__global__ __launch_bounds__(kBlock) void k_regrow_rest(RegrowBatch b) {
  const RegrowOf& d = b.t[blockIdx.y];
  const Slot* __restrict__ old_slots = d.old_slots;
  Slot* __restrict__ slots = d.slots;
  const uint64_t old_cap = d.old_mask + 1, mask = d.mask, length = d.stretch;
  DevState* st = d.st;
  const uint64_t stretch = ((uint64_t)blockIdx.x * kBlock + threadIdx.x) / kRestLanes;
  const unsigned l = threadIdx.x % kRestLanes;
  const unsigned group_shift = (threadIdx.x & 63) / kRestLanes * kRestLanes;
  const uint64_t a = stretch * length;
  bool more = a < old_cap;
  for (uint64_t c = 0; c < length; c += kRestLanes) {
    u64x2 s;
    s.x = kEmptyKey, s.y = 0;
    if (more) s = *reinterpret_cast<const u64x2*>(&old_slots[a + c + l]);
    // the lanes of a wavefront stay together for the ballot; a group that is done reads nothing
    const unsigned long long ends = __ballot(more && s.x == kEmptyKey);
    const unsigned mine = (unsigned)(ends >> group_shift) & ((1u << kRestLanes) - 1u);
    const unsigned first_end = mine ? (unsigned)__builtin_ctz(mine) : (unsigned)kRestLanes;
    if (more && l < first_end) {
      uint64_t h = home_slot(s.x, mask);
      bool placed = false;
      for (uint64_t probes = 0; probes <= mask; ++probes) {
        unsigned long long k = slots[h].key;
        if (k == kEmptyKey) {
          k = atomicCAS(reinterpret_cast<unsigned long long*>(&slots[h].key), (unsigned long long)kEmptyKey,
                        (unsigned long long)s.x);
          if (k == kEmptyKey) {
            slots[h].payload = s.y;
            placed = true;
            break;
          }
        }
        if (k == s.x) {
          store_value(&slots[h].payload, sum_in_order(stored_value(slots[h].payload), stored_value(s.y)));
          atomicAdd(&st->count_shard[stretch % kCountShards * kShardStride], ~0ull);  // (it has been counted twice)
          placed = true;
          break;
        }
        h = (h + 1) & mask;
      }
      if (!placed) atomicOr(&st->error, kDevErrFull);
    }
    if (mine) more = false;
    if (!__any(more)) break;
  }
}

// Collects the keys of all live slots (unordered); *counter must start at 0.
__global__ __launch_bounds__(kBlock) void k_collect_keys(const Slot* __restrict__ slots,
                                                        uint64_t cap, uint64_t* __restrict__ out,
                                                        uint64_t out_cap,
                                                        unsigned long long* counter) {
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t base = (uint64_t)blockIdx.x * kBlock; base < cap; base += stride) {
    const uint64_t i = base + threadIdx.x;
    uint64_t key = kEmptyKey;
    if (i < cap) key = slots[i].key;
    const unsigned long long need = key != kEmptyKey ? 1ull : 0ull;
    const unsigned long long inc = wave_incl_scan_u64(need);
    const unsigned long long tot = __shfl(inc, 63);
    unsigned long long first = 0;
    if ((threadIdx.x & 63) == 63 && tot) first = atomicAdd(counter, tot);
    first = __shfl(first, 63);
    const unsigned long long at = first + inc - need;
    if (need && at < out_cap) out[at] = key;
  }
}

// VARLEN: total floats of all stored rows.
__global__ __launch_bounds__(kBlock) void k_sum_lens(const Slot* __restrict__ slots, uint64_t cap,
                                                    const DevState* st,
                                                    unsigned long long* total) {
  unsigned long long s = 0;
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < cap; i += stride) {
    const ulonglong2 v = *reinterpret_cast<const ulonglong2*>(&slots[i]);
    if (v.x != kEmptyKey) s += v.y & kLenMask;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0 && st->special_present) s += st->special_payload & kLenMask;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
  if ((threadIdx.x & 63) == 0 && s) atomicAdd(total, s);
}

// Plain streaming copy: one non-temporal 16-byte load and store per lane.
__global__ __launch_bounds__(kBlock) void k_copy(f32x4* __restrict__ dst,
                                                const f32x4* __restrict__ src, uint64_t n16) {
  const uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n16) __builtin_nontemporal_store(__builtin_nontemporal_load(&src[i]), &dst[i]);
}

}  // namespace pskv
#endif  // PSKV_TABLE_KERNELS_H_

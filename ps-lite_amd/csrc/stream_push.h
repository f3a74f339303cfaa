// Pushes of many keys into a SCALAR table that is not much larger than they are, or that is moving to a larger array anyway
// (gfx950). Through the slots (k_scalar) a key costs two or three requests to memory, wherever its slot is, and the GPU
// serves 38 to 45 of those per ns; a pass over the whole array costs its bytes. So the keys are put in the order of their
// home slots first, and the array is then streamed through LDS, a stretch at a time, with the stretch's keys applied there:
//   k_split        cuts the request into tiles of 8,192 keys and leaves each tile's keys (and values) sorted by bin, a bin
//                  being the keys whose homes lie in one stretch of the array (the top bits of the hash)
//   k_stream_push  a workgroup per bin: reads its keys from all tiles, builds the new slots of its stretch in LDS, writes them
//                  out whole. Growing, it reads the old array and builds the new one (as k_regrow does), so that the keys of the
//                  request that makes a table grow come along for next to nothing
//   k_regrow_rest  growing: the keys of the old array whose probe chains cross from stretch to stretch
//   k_push_left    the keys of the request whose probe chains do, and those that the tiles do not carry: runs of one key,
//                  the key that marks an empty slot
// 4M keys, 40 % of them held, us of all kernels (through the slots -> here): into 16M slots 232 -> 141, from 4M to 16M slots 290 -> 120, from
// 16M to 32M 351 -> 201, from 32M to 64M 475 -> 334. The same bins with plain stores to the slots in place of the pass
// over the array (no compare-and-swap): 250 for the first, not worth it.
#ifndef PSKV_STREAM_PUSH_H_
#define PSKV_STREAM_PUSH_H_
#include "device_common.h"
#include "stream_rule.h"
#include "table_kernels.h"

namespace pskv {

constexpr unsigned kSplitBlock = 1024;
constexpr unsigned kSplitItems = kSplitTile / kSplitBlock;
constexpr unsigned kStreamBlock = 1024;
constexpr unsigned kStreamItems = kBinKeys / kStreamBlock;  // keys of its bin that a lane holds

// A key that k_push_left looks up the general way, by where it lies: its place among the tiles' keys, or, with kOfRequest, its index in
// the request (where a run of it may follow).
constexpr unsigned kOfRequest = 1u << 31;
static_assert(kMostTiles * kSplitTile < kOfRequest, "places and indexes fit");

struct StreamOf {
  Slot* slots;
  uint64_t mask;
  Slot* old_slots;  // where the keys held are: another array where the table grows
  uint64_t old_mask;
  DevState* st;
  const uint64_t* keys;
  const float* vals;
  uint64_t n;
  unsigned long long* parts;  // per tile: room for its keys, behind them for its values
  uint16_t* starts;           // per tile: where each bin's keys start in it, and its number of keys; a row is bins + kStartsPad
  unsigned* left;             // room for n
  Snapshot* snap;             // counters after the request, or null
  uint64_t snap_seq;
  unsigned long long* told;   // pinned: whether the request named the keys of the one before it (by the sum of their hashes)
  uint32_t tiles;
  uint32_t bins, bin_bits;
  uint32_t images;  // of kImageSlots slots, per bin
  uint32_t turn;    // which of the two counters of left keys
};
struct StreamBatch {
  StreamOf t[kMaxBatch];
};
static_assert(sizeof(StreamBatch) <= 3840, "kernel arguments are limited to 4 KiB");

// The tiles' key and value at a place.
__device__ __forceinline__ const unsigned long long* key_at(const StreamOf& d, unsigned at) {
  return d.parts + (uint64_t)(at / kSplitTile) * kTileWords + at % kSplitTile;
}
__device__ __forceinline__ const float* value_at(const StreamOf& d, unsigned at) {
  return reinterpret_cast<const float*>(d.parts + (uint64_t)(at / kSplitTile) * kTileWords + kSplitTile) + at % kSplitTile;
}

// Room for the left keys of the lanes that call it together.
__device__ __forceinline__ unsigned left_room(DevState* st, unsigned turn) {
  const unsigned long long lanes = __ballot(1);
  const unsigned lane = threadIdx.x & 63, lead = (unsigned)__builtin_ctzll(lanes);
  unsigned at = 0;
  if (lane == lead) at = atomicAdd(&st->left_keys[turn], (unsigned)__popcll(lanes));
  return __shfl(at, lead) + (unsigned)__popcll(lanes & ((1ull << lane) - 1ull));
}

// One workgroup per tile. Bound by memory (12 bytes read and 12 written per key; 4M keys 24.4 us, 3.9 TB/s). A bin's place of a
// key is its rank among the tile's keys of that bin (an LDS atomic per key, two 16-bit counters a word, which leaves LDS for
// two workgroups per compute unit), keys and values travel through the same LDS one after the other, so that all
// that is written is written in whole lines. With one atomic per key and tile to counters in memory in place of rows
// of starts, and with keys and values stored straight to their places: 54 us.
__global__ __launch_bounds__(kSplitBlock, 8) void k_split(StreamBatch b) {
  const StreamOf& d = b.t[blockIdx.y];
  if (blockIdx.x >= d.tiles) return;
  __shared__ unsigned s_bins[kMostBins / 2];
  __shared__ unsigned long long s_keys[kSplitTile];
  __shared__ unsigned red[kSplitBlock / 64];
  __shared__ unsigned s_left, s_left_at;
  __shared__ unsigned long long s_sum;
  const uint64_t n = d.n, at = (uint64_t)blockIdx.x * kSplitTile;
  const uint64_t* __restrict__ keys = d.keys;
  const float* __restrict__ vals = d.vals;
  const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // (a wavefront's keys are neighbours: it looks at two more to know which of them start or continue a run)
  const uint64_t mine0 = at + (wave * kSplitItems) * 64 + lane;
  uint64_t key[kSplitItems];
#pragma unroll
  for (unsigned q = 0; q < kSplitItems; ++q) {
    const uint64_t i = mine0 + q * 64;
    key[q] = __builtin_nontemporal_load(keys + (i < n ? i : n - 1));
  }
  uint64_t outside = 0;
  {
    const uint64_t i = lane == 0 ? mine0 - 1 : mine0 + kSplitItems * 64 - 63;
    if ((lane == 0 && mine0 > 0 && i < n) || (lane == 63 && i < n)) outside = keys[i];
  }
  for (unsigned x = threadIdx.x; x < kMostBins / 2; x += kSplitBlock) s_bins[x] = 0;
  if (threadIdx.x == 0) s_left = 0, s_sum = 0;
  __syncthreads();
  constexpr unsigned kInLeft = 1u << 31, kNowhere = ~0u;
  float v[kSplitItems];
  unsigned place[kSplitItems];  // bin << 16 | rank in it; kInLeft | rank among the tile's left keys; kNowhere
  unsigned long long sum = 0;
#pragma unroll
  for (unsigned q = 0; q < kSplitItems; ++q) {
    const uint64_t i = mine0 + q * 64;
    uint64_t before = __shfl_up(key[q], 1), after = __shfl_down(key[q], 1);
    const uint64_t last = q ? __shfl(key[q ? q - 1 : 0], 63) : outside;
    const uint64_t next = q + 1 < kSplitItems ? __shfl(key[q + 1 < kSplitItems ? q + 1 : 0], 0) : outside;
    if (lane == 0) before = last;
    if (lane == 63) after = next;
    place[q] = kNowhere;
    if (i >= n || (i > 0 && before == key[q])) continue;  // past the end, or inside a run
    const bool run = i + 1 < n && after == key[q];
    const uint64_t hash = mix64(key[q]);
    sum += hash;
    if (run || key[q] == kEmptyKey) {
      place[q] = kInLeft | atomicAdd(&s_left, 1u);
      continue;
    }
    const unsigned bin = (unsigned)(hash >> (64 - d.bin_bits)), half = (bin & 1) * 16;
    place[q] = bin << 16 | ((atomicAdd(&s_bins[bin >> 1], 1u << half) >> half) & 0xffffu);
  }
#pragma unroll
  for (unsigned q = 0; q < kSplitItems; ++q) {
    const uint64_t i = mine0 + q * 64;
    v[q] = __builtin_nontemporal_load(vals + (i < n ? i : n - 1));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
  if (lane == 0) atomicAdd(&s_sum, sum);
  __syncthreads();
  if (threadIdx.x == 0) {
    if (s_left) s_left_at = atomicAdd(&d.st->left_keys[d.turn], s_left);
    atomicAdd(&d.st->count_shard[blockIdx.x % kCountShards * kShardStride + 1], s_sum);
  }
  // where each bin starts: a prefix sum over the counters
  constexpr unsigned kWords = kMostBins / 2 / kSplitBlock;
  unsigned w[kWords], mine = 0;
#pragma unroll
  for (unsigned q = 0; q < kWords; ++q) {
    w[q] = s_bins[threadIdx.x * kWords + q];
    mine += (w[q] & 0xffffu) + (w[q] >> 16);
  }
  unsigned inc = mine;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned y = __shfl_up(inc, o);
    if (lane >= (unsigned)o) inc += y;
  }
  if (lane == 63) red[wave] = inc;
  __syncthreads();
  unsigned run = inc - mine, total = 0;
  for (unsigned x = 0; x < kSplitBlock / 64; ++x) {
    if (x < wave) run += red[x];
    total += red[x];
  }
  unsigned* starts = reinterpret_cast<unsigned*>(d.starts + (uint64_t)blockIdx.x * (d.bins + kStartsPad));
#pragma unroll
  for (unsigned q = 0; q < kWords; ++q) {
    const unsigned x = threadIdx.x * kWords + q, first = w[q] & 0xffffu, second = w[q] >> 16;
    w[q] = run | (run + first) << 16;
    run += first + second;
    s_bins[x] = w[q];
    if (x < d.bins / 2) starts[x] = w[q];
  }
  if (threadIdx.x == 0) starts[d.bins / 2] = total;
  __syncthreads();
  unsigned long long* out = d.parts + (uint64_t)blockIdx.x * kTileWords;
#pragma unroll
  for (unsigned q = 0; q < kSplitItems; ++q) {
    if (place[q] == kNowhere) continue;
    if (place[q] & kInLeft) {
      d.left[s_left_at + (place[q] & 0xffffu)] = kOfRequest | (unsigned)(mine0 + q * 64);
      place[q] = kNowhere;
      continue;
    }
    const unsigned bin = place[q] >> 16;
    place[q] = (s_bins[bin >> 1] >> ((bin & 1) * 16) & 0xffffu) + (place[q] & 0xffffu);
    s_keys[place[q]] = key[q];
  }
  __syncthreads();
#pragma unroll
  for (unsigned q = 0; q < kSplitItems; ++q) {
    const unsigned j = q * kSplitBlock + threadIdx.x;
    if (j < total) out[j] = s_keys[j];
  }
  __syncthreads();
  float* s_vals = reinterpret_cast<float*>(s_keys);
#pragma unroll
  for (unsigned q = 0; q < kSplitItems; ++q)
    if (place[q] != kNowhere) s_vals[place[q]] = v[q];
  __syncthreads();
  float* out_vals = reinterpret_cast<float*>(out + kSplitTile);
#pragma unroll
  for (unsigned q = 0; q < kSplitItems; ++q) {
    const unsigned j = q * kSplitBlock + threadIdx.x;
    if (j < total) out_vals[j] = s_vals[j];
  }
}

// One workgroup per bin: images of kImageSlots slots (keys and values, 48 KiB of LDS, 54 in all, so two workgroups of 1,024 lanes per
// compute unit: one streams while the other looks for its keys), the next one asked for while the keys of this one are
// placed. Bound by memory: 4.3 (from 4M to 16M) to 5.8 TB/s (32M that stay) of slots. 4M keys into 16M slots 105 us; workgroups of 512 lanes with images of
// 2,048 slots 131, with 4,096 113, one image per bin instead of two 113 (as many lines read for half the keys). Keys whose
// probe chains leave their image, and those of a bin that has more than its lanes hold, are left to k_push_left.
// What a growth leaves in the old array is as with k_regrow: packed over the front of each image's old slots. A
// key of the request may be among those; it is created in its image then, and k_regrow_rest adds the two up.
// The runs of the bin's keys have LDS of their own, so that a key that is left can be named by its place (where the values go, they were
// gone by then): from 16M to 32M slots 179 -> 158 us, from 32M to 64M 310 -> 293, arrays that stay as before.
// SLOTS: of the array that the keys are in, per lane and image: 4 where it stays, 2 for one that becomes twice as large, 1 beyond.
template <unsigned SLOTS>
__global__ __launch_bounds__(kStreamBlock, 8) void k_stream_push(StreamBatch b) {
  constexpr bool GROW = SLOTS * kStreamBlock < kImageSlots;
  const StreamOf& d = b.t[blockIdx.y];
  if (blockIdx.x >= d.bins) return;
  __shared__ unsigned long long s_key[kImageSlots];
  __shared__ float s_val[kImageSlots];
  __shared__ unsigned red[kStreamBlock / 64];
  __shared__ unsigned s_rest;
  // where each tile's keys of this bin lie
  __shared__ unsigned s_before[kMostTiles];
  __shared__ uint16_t s_from[kMostTiles];
  // (workgroups are dealt out to the eight XCDs in turn: bins next to each other, whose keys share lines, to one of them)
  const unsigned bin = d.bins % 8 == 0 ? blockIdx.x % 8 * (d.bins / 8) + blockIdx.x / 8 : blockIdx.x;
  const uint64_t mask = d.mask, base = (uint64_t)bin * d.images * kImageSlots;
  const unsigned factor = GROW ? (unsigned)((mask + 1) / (d.old_mask + 1)) : 1u;
  const unsigned olds = kImageSlots / factor;  // slots of the old array per image
  Slot* __restrict__ from = d.old_slots + base / factor;
  u64x2 s[SLOTS];
  auto ask = [&](unsigned image) {
#pragma unroll
    for (unsigned q = 0; q < SLOTS; ++q) {
      const unsigned j = q * kStreamBlock + threadIdx.x;
      s[q].x = kEmptyKey, s[q].y = kPayloadUnset;
      if (j < olds) s[q] = __builtin_nontemporal_load(reinterpret_cast<const u64x2*>(&from[(uint64_t)image * olds + j]));
    }
  };
  const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const unsigned tiles = d.tiles;
  unsigned total = 0;  // keys of the bin
  {
    static_assert(kMostTiles == kStreamBlock, "a lane looks at a tile");
    const unsigned t = threadIdx.x;
    unsigned first = 0, many = 0;
    if (t < tiles) {
      const uint16_t* row = d.starts + (uint64_t)t * (d.bins + kStartsPad) + bin;
      first = row[0];
      many = row[1] - first;
    }
    ask(0);
    unsigned inc = many;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const unsigned y = __shfl_up(inc, o);
      if (lane >= (unsigned)o) inc += y;
    }
    if (lane == 63) red[wave] = inc;
    __syncthreads();
    unsigned before = inc - many;
    for (unsigned x = 0; x < kStreamBlock / 64; ++x) {
      if (x < wave) before += red[x];
      total += red[x];
    }
    if (t < tiles) {
      s_before[t] = before;
      s_from[t] = (uint16_t)first;
    }
    __syncthreads();
  }
  // key j of the bin: its place among the tiles' keys
  auto find = [&](unsigned j) {
    unsigned t = 0;
    for (unsigned many = tiles; many > 1;) {
      const unsigned half = many >> 1;
      const bool up = s_before[t + half] <= j;
      t = up ? t + half : t;
      many = up ? many - half : half;
    }
    return t * kSplitTile + s_from[t] + (j - s_before[t]);
  };
  unsigned long long key[kStreamItems];
  float v[kStreamItems];
#pragma unroll
  for (unsigned q = 0; q < kStreamItems; ++q) {
    const unsigned j = q * kStreamBlock + threadIdx.x;
    key[q] = 0, v[q] = 0.0f;
    if (j < total) {
      const unsigned at = find(j);
      key[q] = *key_at(d, at);
      v[q] = *value_at(d, at);
    }
  }
  for (unsigned j = kBinKeys + threadIdx.x; j < total; j += kStreamBlock) d.left[left_room(d.st, d.turn)] = find(j);
  if (GROW) {
    for (unsigned j = threadIdx.x; j < kImageSlots; j += kStreamBlock) s_key[j] = kEmptyKey, s_val[j] = 0.0f;
  }
  unsigned created = 0, left = 0;  // left: a bit for each of the lane's keys that found no place
  for (unsigned image = 0; image < d.images; ++image) {
    if (GROW) {
      const uint64_t old_base = base / factor + (uint64_t)image * olds;
      if (threadIdx.x == 0) s_rest = 0;
      // (nobody writes into the old slots before everybody's have arrived)
#pragma unroll
      for (unsigned q = 0; q < SLOTS; ++q) arrived(s[q]);
      __syncthreads();
      bool rest[SLOTS];
#pragma unroll
      for (unsigned q = 0; q < SLOTS; ++q) {
        const unsigned at = q * kStreamBlock + threadIdx.x;
        rest[q] = false;
        if (at >= olds || s[q].x == kEmptyKey) continue;
        rest[q] = true;
        // (a home in another stretch, in front of this one or, around the end of the array, behind it: for the second pass)
        if (home_slot(s[q].x, d.old_mask) - old_base > at) continue;
        for (unsigned j = (unsigned)home_slot(s[q].x, mask) % kImageSlots; j < kImageSlots; ++j) {
          if (atomicCAS(&s_key[j], (unsigned long long)kEmptyKey, (unsigned long long)s[q].x) != kEmptyKey) continue;
          s_val[j] = stored_value(s[q].y);
          rest[q] = false;
          break;
        }
      }
#pragma unroll
      for (unsigned q = 0; q < SLOTS; ++q)
        if (rest[q]) *reinterpret_cast<u64x2*>(&from[(uint64_t)image * olds + atomicAdd(&s_rest, 1u)]) = s[q];
    } else {
#pragma unroll
      for (unsigned q = 0; q < SLOTS; ++q) {
        const unsigned j = q * kStreamBlock + threadIdx.x;
        s_key[j] = s[q].x;
        s_val[j] = stored_value(s[q].y);
      }
    }
    if (image + 1 < d.images) ask(image + 1);
    __syncthreads();
    if (GROW && threadIdx.x == 0 && s_rest < olds) from[(uint64_t)image * olds + s_rest].key = kEmptyKey;
#pragma unroll
    for (unsigned q = 0; q < kStreamItems; ++q) {
      const unsigned home = (unsigned)(home_slot(key[q], mask) - base);
      if (q * kStreamBlock + threadIdx.x >= total || home / kImageSlots != image) continue;
      bool placed = false;
      for (unsigned j = home % kImageSlots; j < kImageSlots && !placed; ++j) {
        unsigned long long k = s_key[j];
        if (k == kEmptyKey) {
          k = atomicCAS(&s_key[j], (unsigned long long)kEmptyKey, key[q]);
          if (k == kEmptyKey) {  // an absent key starts from 0.0f, then `+=` (kv_app.h:454)
            s_val[j] = 0.0f + v[q];
            ++created;
            placed = true;
          }
        }
        if (k == key[q]) {
          s_val[j] = sum_in_order(v[q], s_val[j]);
          placed = true;
        }
      }
      if (!placed) left |= 1u << q;
    }
    __syncthreads();
    u64x2* __restrict__ out = reinterpret_cast<u64x2*>(d.slots + base + (uint64_t)image * kImageSlots);
#pragma unroll
    for (unsigned q = 0; q < kImageSlots / kStreamBlock; ++q) {
      const unsigned j = q * kStreamBlock + threadIdx.x;
      u64x2 w;
      w.x = s_key[j];
      w.y = kPayloadUnset ^ __float_as_uint(s_val[j]);
      __builtin_nontemporal_store(w, &out[j]);
      if (GROW) s_key[j] = kEmptyKey, s_val[j] = 0.0f;
    }
    // (what a lane writes in front of the next barrier, it has read itself)
  }
  for (unsigned q = 0; q < kStreamItems; ++q)
    if (left >> q & 1u) d.left[left_room(d.st, d.turn)] = find(q * kStreamBlock + threadIdx.x);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) created += __shfl_xor(created, o);
  if (lane == 0) red[wave] = created;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned all = 0;
    for (unsigned x = 0; x < kStreamBlock / 64; ++x) all += red[x];
    if (all) atomicAdd(&d.st->count_shard[blockIdx.x % kCountShards * kShardStride], (unsigned long long)all);
  }
}

// The keys that the pass over the array has left, a lane each; a run is added up in the order of the request, as k_scalar
// does. Usually some hundred of 4M: three trips to memory that follow from each other.
__global__ __launch_bounds__(kBlock) void k_push_left(StreamBatch b) {
  const StreamOf& d = b.t[blockIdx.y];
  DevState* st = d.st;
  const unsigned left = st->left_keys[d.turn];
  __shared__ unsigned red[kBlock / 64];
  unsigned created = 0;
  for (unsigned x = blockIdx.x * kBlock + threadIdx.x; x < left; x += gridDim.x * kBlock) {
    const unsigned at = d.left[x], i = at & ~kOfRequest;
    const bool of_request = (at & kOfRequest) != 0;
    const unsigned long long key = of_request ? d.keys[i] : *key_at(d, i);
    const float v = of_request ? d.vals[i] : *value_at(d, i);
    bool is_new;
    uint64_t seen;
    uint64_t* p = find_or_insert(d.slots, d.mask, st, key, is_new, seen);
    if (!p) continue;
    float cur = sum_in_order(v, is_new ? 0.0f : stored_value(seen));
    if (of_request)
      for (uint64_t j = (uint64_t)i + 1; j < d.n && d.keys[j] == key; ++j) cur = sum_in_order(cur, d.vals[j]);
    store_value(p, cur);
    created += is_new ? 1u : 0u;
  }
  if (blockIdx.x * kBlock < left) block_count_add(st, created, red);
  if (blockIdx.x == 0) {
    if (threadIdx.x == 0) st->left_keys[d.turn ^ 1u] = 0;  // (for the next request; this one's may yet be read)
    if (threadIdx.x < 64) {
      unsigned long long sum = threadIdx.x < kCountShards ? atomicExch(&st->count_shard[threadIdx.x * kShardStride + 1], 0ull) : 0ull;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
      if (threadIdx.x == 0) {
        __hip_atomic_store(d.told, sum == st->keys_sum ? 1ull : 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        st->keys_sum = sum;
      }
    }
  }
  if (!d.snap) return;
  __shared__ unsigned s_last;
  if (threadIdx.x == 0) s_last = ticket_last(st, gridDim.x) ? 1u : 0u;
  __syncthreads();
  if (s_last && threadIdx.x < 64) publish_snapshot(st, d.snap, d.snap_seq);
}

}  // namespace pskv
#endif  // PSKV_STREAM_PUSH_H_

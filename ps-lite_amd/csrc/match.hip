// Ordered match of two sorted key sets on the GPU (gfx950): the merge-join that the reference
// sketches in ParallelOrderedMatch (include/ps/internal/parallel_kv_match.h:29-120) with the
// operators of assign_op.h:12-41:
//     if (dst_key[i] == src_key[j]) dst_val[i] op= src_val[j]        (k floats per key)
// Both key sets are sorted, so the keys of one that can match a tile of the other's are
// one contiguous stretch. A first small kernel finds where every tile's stretch begins (one
// search per tile, all tiles at once; where there are few, the workgroups do so themselves); a workgroup then stages its
// stretch in LDS, or samples it there where it is long, and resolves its keys, so where the sets are of like size all key traffic is streamed, once. For
// k == 1 the values are combined in the same kernel; for longer values the kernel leaves the index of every key's match
// behind and a second kernel streams the rows.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <mutex>
#include <new>
#include <type_traits>

#include "device_common.h"
#include "host_common.h"
#include "search.h"

namespace pskv {
namespace {

constexpr unsigned kMatchBlock = 256;
// Keys per lane: four neighbouring ones, the first found by halving and the others a few keys further on; one where
// four would leave the GPU with fewer than two workgroups per compute unit, or a tile's stretch would not fit into LDS
// because the other set is twice as large or more.
constexpr unsigned kMatchItems = 4;
constexpr uint64_t kFewKeys = 2ull * 256 * kMatchBlock * kMatchItems;
constexpr unsigned kMatchLds = 1536;    // source keys (and values) a workgroup holds in LDS at a time (18 KiB)
constexpr unsigned kMatchTurn = kMatchLds / kMatchBlock;  // source keys a lane asks for: all that there is room for
// A longer stretch than so many pieces is sampled, not staged. (Pieces follow from each other, but read in one go
// what the sampled search reads key by key: they pay while there are workgroups enough to fill the GPU.)
constexpr unsigned kMatchPieces = 8, kMatchPiecesFew = 3;
// Tiles (of kMatchItems keys a lane, and of one) up to which the workgroups search for themselves, without a launch in front of them;
// tiles of kMatchItems keys a lane up to as many as those of one, too, where the other set is small (own_search).
constexpr unsigned kOwnSpans = 2560, kOwnSpansFew = 4096;
// What the search in front costs a call hardly depends on the sets; the workgroups' own costs by the tiles and by how many rounds each
// takes. us per call, with the launch in front and without: 30,000 into 3M keys 27.0 and 25.3, 1M into 3M 33.1 and 31.6, 2M into 3M 35.4
// and 34.7, 2.6M into 3M 36.4 and 36.6; 1M into 3.5M 34.3 and 33.9, 1.5M into 3.5M 35.3 and 35.8; 100,000 into 4.1M 31.7 and 31.0, 700,000
// into 4.1M 35.1 and 35.5.
constexpr bool own_search(uint64_t n_near, uint64_t n_far, unsigned blocks, bool few) {
  return blocks <= kOwnSpans || (blocks <= kOwnSpansFew && (few || n_near * 7 / 4 + n_far <= 29ull << 18));
}
constexpr uint64_t kNoMatch = ~0ull;
constexpr unsigned kCounts = 64;        // counters of matched keys, each on a line of its own
constexpr unsigned kCountStride = 16;

// assign_op.h:26-36: right op= left
__device__ __forceinline__ float combine(int op, float d, float s) {
  switch (op) {
    case PSKV_OP_PLUS: return d + s;
    case PSKV_OP_MINUS: return d - s;
    case PSKV_OP_TIMES: return d * s;
    case PSKV_OP_DIVIDE: return d / s;
    default: return s;
  }
}
__device__ __forceinline__ f32x4 combine(int op, f32x4 d, f32x4 s) {
  f32x4 r;
  r.x = combine(op, d.x, s.x), r.y = combine(op, d.y, s.y);
  r.z = combine(op, d.z, s.z), r.w = combine(op, d.w, s.w);
  return r;
}

// The match walks the tiles of one key set and finds their keys in the other. spans[t] = first key of the set that is
// searched (`src`, n_src keys) not below the first key of tile t of the other; spans[tiles] = n_src.
// The stretch of tile t is [spans[t], spans[t+1]): it may hold keys that lie between two
// tiles, which match nothing. Bound by the lines it reads (16 probes for each of 15,625 tiles are 6 us) and by the round trips
// that follow from each other: a workgroup samples the whole source evenly into LDS (one round trip, the same lines for every
// workgroup), its kSpanTiles tiles find the step they lie in there, and kSpanLanes lanes per tile look at kSpanWindow keys,
// a line or two or three, around the place where the tile's first key should be if the keys between the two that enclose it are spread evenly. A
// step of 12,000 keys spread by a hash takes two or three looks; what is not found after kSpanLooks of them is narrowed down by a
// factor of 16 per round. 12M into 16M keys: 17.5 us -> 10.6 (4,096 samples and three rounds of 16 probes without a guess), the
// whole call 103 -> 96.5; into keys in 2,000 clusters, where guesses are no good, 96.3 -> 95.4, squares 89.8 -> 88.3.
constexpr unsigned kSpanLanes = 16;
constexpr unsigned kSpanTiles = 64;
constexpr unsigned kSpanBlock = kSpanTiles * kSpanLanes;
constexpr unsigned kSpanSamples = kSpanBlock;
constexpr unsigned kSpanWindow = 2 * kSpanLanes;
constexpr unsigned kSpanLooks = 4;
__global__ __launch_bounds__(kSpanBlock) void k_match_spans(const uint64_t* __restrict__ src, uint64_t n_src,
                                                            const uint64_t* __restrict__ dst, uint64_t tiles,
                                                            unsigned tile, uint64_t* __restrict__ spans) {
  __shared__ uint64_t s_sample[kSpanSamples];
  const uint64_t t = (uint64_t)blockIdx.x * kSpanTiles + threadIdx.x / kSpanLanes;
  const unsigned lane = threadIdx.x & 63, sub = threadIdx.x % kSpanLanes;
  const bool live = t < tiles;
  const uint64_t key = live ? dst[t * tile] : 0;
  const uint64_t step = (n_src + kSpanSamples - 1) / kSpanSamples;
  const unsigned samples = (unsigned)((n_src + step - 1) / step);
  s_sample[threadIdx.x] = src[(threadIdx.x < samples ? threadIdx.x : samples - 1) * step];
  if (t == 0 && sub == 0) spans[tiles] = n_src;
  __syncthreads();
  unsigned a = 0, b = samples;  // samples before a are below the key, none from b on is
  while (a < b) {
    const unsigned mid = (a + b) >> 1;
    if (s_sample[mid] < key) a = mid + 1; else b = mid;
  }
  // every source key before lo is below the key, none from hi on is
  uint64_t lo = a ? (a - 1) * step + 1 : 0, hi = !live ? lo : a < samples ? a * step : n_src;
  if (a == 0) hi = lo;  // (the first sample is the first key)
  const unsigned of_group = lane / kSpanLanes * kSpanLanes;
  // (the lanes of a group stay together)
  auto count = [&](bool x) { return (unsigned)__popcll((__ballot(x) >> of_group) & ((1ull << kSpanLanes) - 1)); };
  const bool enclosed = a > 0 && a < samples;
  uint64_t under = enclosed ? s_sample[a - 1] : 0, over = enclosed ? s_sample[a] : 0;  // the keys at lo - 1 and at hi
  for (unsigned look = 0; look < kSpanLooks && __any(enclosed && lo < hi); ++look) {
    const float share = (float)(key - under) / (float)(over - under);
    const uint64_t guess = lo + (uint64_t)(fminf(fmaxf(share, 0.0f), 1.0f) * (float)(hi - lo));
    uint64_t from = guess > lo + kSpanWindow / 2 ? guess - kSpanWindow / 2 : lo;
    if (from + kSpanWindow > hi) from = hi - lo > kSpanWindow ? hi - kSpanWindow : lo;
    const uint64_t p0 = from + sub, p1 = p0 + kSpanLanes;
    const bool in0 = enclosed && p0 < hi, in1 = enclosed && p1 < hi;
    const uint64_t x0 = in0 ? src[p0] : ~0ull, x1 = in1 ? src[p1] : ~0ull;
    const unsigned looked = count(in0) + count(in1), below = count(in0 && x0 < key) + count(in1 && x1 < key);
    const uint64_t first = __shfl(x0, (int)of_group), last = __shfl(x1, (int)(of_group + kSpanLanes - 1));
    if (looked == 0) continue;  // found before
    if (below == 0 && from > lo) {
      hi = from, over = first;
    } else if (below == looked && from + looked < hi) {
      lo = from + looked, under = last;  // (a whole window: it ends before hi)
    } else {
      lo = hi = from + below;
    }
  }
  // (a wavefront takes as many rounds as the longest of its groups)
  while (__any(lo < hi)) {
    const uint64_t stride = (hi - lo + kSpanLanes - 1) / kSpanLanes;
    const uint64_t p = lo + sub * stride;
    const unsigned cnt = count(p < hi && src[p] < key);
    // the probes are sorted: the first cnt are below
    if (cnt == 0) {
      hi = lo;
    } else {
      const uint64_t next = lo + cnt * stride;  // the first probe that is not below, if there is one
      lo += (cnt - 1) * stride + 1;
      if (cnt < kSpanLanes && next < hi) hi = next;
    }
  }
  if (live && sub == 0) spans[t] = lo;
}

// One workgroup per tile of kMatchBlock * ITEMS keys of `near`, which it finds in `far`. Those are the destination's
// and the source's keys, or with SWAP, where the source is much the smaller set, the other way round: the walk then
// reads, and the row kernel visits, what there is in the source. Bound by memory once the loads do not wait for each
// other: 12M source against 16M destination keys, the whole call, took 125 us with one source key per lane asked for at a
// time, 104.7 with three under a condition each, 101 without it, and 99.5 with all six that LDS has room for.
// OWN: the workgroup finds where its stretch begins and ends itself (a wavefront each) instead of reading it from `spans`:
// the search is hidden behind the keys of the tile, and a launch in front of this one falls away, but every
// workgroup reads lines for it that nobody else needs. Up to kOwnSpans tiles that is the better way (us per call:
// 45,928 into 44,225 keys 16.6 -> 13.5, 1M into 1M 28.0 -> 21.4, 2.6M into 1.4M 39.3 -> 32.6; against the search as it is now 3M
// into 3M 41.3 -> 42.1, 4M into 4M 45.9 -> 50.3, but 1M into 16M, tiles of 256 keys, 70.7 -> 66.3).
// K1: values are single floats and are combined here; otherwise where[i] receives the index in `far` of the match of
// key i, or kNoMatch.
template <bool K1, bool SWAP, unsigned ITEMS, bool OWN>
__global__ __launch_bounds__(kMatchBlock) void k_match_keys(const uint64_t* __restrict__ far, uint64_t n_far,
                                                            const uint64_t* __restrict__ near, uint64_t n_near,
                                                            const uint64_t* __restrict__ spans,
                                                            uint64_t* __restrict__ where,
                                                            const float* __restrict__ src_vals,
                                                            float* __restrict__ dst_vals, int op,
                                                            unsigned long long* __restrict__ counts) {
  static_assert(ITEMS == 4 || ITEMS == 1, "128-bit accesses of four keys, or one key");
  __shared__ uint64_t s_keys[kMatchLds];
  __shared__ float s_vals[K1 && !SWAP ? kMatchLds : 1];
  __shared__ unsigned s_red[kMatchBlock / 64];
  constexpr unsigned kTile = kMatchBlock * ITEMS;
  const uint64_t first = (uint64_t)blockIdx.x * kTile;
  const uint64_t tile_n = n_near - first < kTile ? n_near - first : kTile;
  const unsigned idx0 = threadIdx.x * ITEMS;
  const uint64_t i0 = first + idx0;
  uint64_t key[ITEMS];
  const bool whole = ITEMS == 4 && idx0 + ITEMS <= tile_n;
  if (whole && (reinterpret_cast<uintptr_t>(near) & 15) == 0) {
    const u64x2 x = *reinterpret_cast<const u64x2*>(near + i0);
    const u64x2 y = *reinterpret_cast<const u64x2*>(near + i0 + 2);
    key[0] = x.x, key[1 % ITEMS] = x.y, key[2 % ITEMS] = y.x, key[3 % ITEMS] = y.y;
  } else {
#pragma unroll
    for (unsigned r = 0; r < ITEMS; ++r) key[r] = near[idx0 + r < tile_n ? i0 + r : first];
  }
  __shared__ uint64_t s_span[OWN ? 2 : 1];
  if (OWN) {
    const unsigned wave = threadIdx.x >> 6;
    if (wave < 2) {
      const uint64_t at = first + wave * kTile;
      const uint64_t end = at < n_near ? wave_lower_bound(far, n_far, near[at], threadIdx.x & 63) : n_far;
      if ((threadIdx.x & 63) == 0) s_span[wave] = end;
    }
    __syncthreads();
  }
  const uint64_t lo = OWN ? s_span[0] : spans[blockIdx.x], hi = OWN ? s_span[OWN ? 1 : 0] : spans[blockIdx.x + 1];
  const uint64_t span = hi > lo ? hi - lo : 0;  // (hi >= lo when the keys are sorted)
  // K1: the values follow the keys without waiting for what the search finds: those of this side are
  // asked for here (a line of 32 of them without a match is rare), those of a stretch that fits into LDS come
  // with its keys.
  const float* near_vals = SWAP ? src_vals : dst_vals;
  const bool vec = K1 && whole && (reinterpret_cast<uintptr_t>(near_vals) & 15) == 0;
  const bool vals_here = K1 && !SWAP && span <= kMatchLds;
  f32x4 mine = (f32x4)(0.f);
  if (vec) {
    mine = *reinterpret_cast<const f32x4*>(near_vals + i0);
  } else if (K1) {
#pragma unroll
    for (unsigned r = 0; r < ITEMS; ++r) mine[r] = near_vals[idx0 + r < tile_n ? i0 + r : first];
  }
  uint64_t j[ITEMS];
  bool open[ITEMS];
#pragma unroll
  for (unsigned r = 0; r < ITEMS; ++r) {
    j[r] = kNoMatch;
    open[r] = idx0 + r < tile_n;
  }
  if (span <= (uint64_t)kMatchLds * (ITEMS == 1 ? kMatchPiecesFew : kMatchPieces)) {
    // The stretch goes through LDS in pieces of kMatchLds keys. A key is looked up in the first
    // piece whose last key is not below it (or in the last piece).
    for (uint64_t base = 0; base < span; base += kMatchLds) {
      const unsigned len = span - base < kMatchLds ? (unsigned)(span - base) : kMatchLds;
      const bool last_piece = base + len == span;
      if (base) __syncthreads();  // everyone is done with the piece before
      // (all loads before the first of them is waited for; with values, a lane behind the end asks for the last key, as a
      // load under a condition waits for those in front of it)
      {
        const unsigned t0 = threadIdx.x;
        uint64_t ks[kMatchTurn];
        float vs[kMatchTurn] = {};
#pragma unroll
        for (unsigned q = 0; q < kMatchTurn; ++q) {
          const unsigned t = t0 + q * kMatchBlock;
          ks[q] = K1 ? far[lo + base + (t < len ? t : len - 1)] : t < len ? far[lo + base + t] : 0;
        }
        if (vals_here) {
#pragma unroll
          for (unsigned q = 0; q < kMatchTurn; ++q) {
            const unsigned t = t0 + q * kMatchBlock;
            vs[q] = src_vals[lo + base + (t < len ? t : len - 1)];
          }
        }
#pragma unroll
        for (unsigned q = 0; q < kMatchTurn; ++q) {
          const unsigned t = t0 + q * kMatchBlock;
          if (t >= len) continue;
          s_keys[t] = ks[q];
          if (vals_here) s_vals[t] = vs[q];
        }
      }
      __syncthreads();
      const uint64_t top = s_keys[len - 1];
      unsigned pos = 0;     // the lane's open keys are above every key before this one
      bool on_foot = false;  // whether a key of this lane has been placed in this piece already
#pragma unroll
      for (unsigned r = 0; r < ITEMS; ++r) {
        if (!open[r] || !(key[r] <= top || last_piece)) continue;
        unsigned at = pos;
        if (on_foot) {
          for (unsigned step = 0; step < 4 && at < len && s_keys[at] < key[r]; ++step) ++at;
        }
        if (at < len && s_keys[at] < key[r]) {  // halve what is left
          unsigned end = len;
          ++at;
          while (at < end) {
            const unsigned mid = (at + end) >> 1;
            if (s_keys[mid] < key[r]) at = mid + 1; else end = mid;
          }
        }
        if (at < len && s_keys[at] == key[r]) j[r] = lo + base + at;
        open[r] = false;
        pos = at;
        on_foot = true;
      }
    }
  } else {
    // Far more keys there than here: the stretch is sampled evenly into LDS, a key finds the step it lies in there and
    // halves that step where it lies, a line or two. (Halving the whole stretch in memory took 14 trips that follow
    // from each other for 13,000 keys, 50 us.)
    const uint64_t step = (span + kMatchLds - 1) / kMatchLds;
    const unsigned samples = (unsigned)((span + step - 1) / step);
    {
      const unsigned t0 = threadIdx.x;
      uint64_t ks[kMatchTurn];
#pragma unroll
      for (unsigned q = 0; q < kMatchTurn; ++q) {
        const unsigned t = t0 + q * kMatchBlock;
        ks[q] = far[lo + (t < samples ? t : samples - 1) * step];
      }
#pragma unroll
      for (unsigned q = 0; q < kMatchTurn; ++q)
        if (t0 + q * kMatchBlock < samples) s_keys[t0 + q * kMatchBlock] = ks[q];
    }
    __syncthreads();
    uint64_t a[ITEMS], b[ITEMS];  // every key before a is below the lane's, none from b on is
#pragma unroll
    for (unsigned r = 0; r < ITEMS; ++r) {
      unsigned at = 0, end = samples;
      while (at < end) {
        const unsigned mid = (at + end) >> 1;
        if (s_keys[mid] < key[r]) at = mid + 1; else end = mid;
      }
      a[r] = at ? lo + (at - 1) * step + 1 : lo;
      b[r] = at < samples ? lo + at * step : hi;
      if (!open[r]) b[r] = a[r];
    }
    for (uint64_t left = step; left > 0; left >>= 1) {  // (the lane's keys side by side)
#pragma unroll
      for (unsigned r = 0; r < ITEMS; ++r) {
        if (a[r] >= b[r]) continue;
        const uint64_t mid = a[r] + ((b[r] - a[r]) >> 1);
        if (far[mid] < key[r]) a[r] = mid + 1; else b[r] = mid;
      }
    }
#pragma unroll
    for (unsigned r = 0; r < ITEMS; ++r)
      if (open[r] && a[r] < n_far && far[a[r]] == key[r]) j[r] = a[r];
  }
  unsigned found = 0;
#pragma unroll
  for (unsigned r = 0; r < ITEMS; ++r) found += j[r] != kNoMatch ? 1u : 0u;
  if (K1 && SWAP) {
    float d[ITEMS];
#pragma unroll
    for (unsigned r = 0; r < ITEMS; ++r) d[r] = op != PSKV_OP_ASSIGN && j[r] != kNoMatch ? dst_vals[j[r]] : 0.0f;
#pragma unroll
    for (unsigned r = 0; r < ITEMS; ++r)
      if (j[r] != kNoMatch) dst_vals[j[r]] = combine(op, d[r], mine[r]);
  } else if (K1) {
#pragma unroll
    for (unsigned r = 0; r < ITEMS; ++r)
      if (j[r] != kNoMatch) mine[r] = combine(op, mine[r], vals_here ? s_vals[j[r] - lo] : src_vals[j[r]]);
    if (vec) {
      if (found) *reinterpret_cast<f32x4*>(dst_vals + i0) = mine;
    } else {
#pragma unroll
      for (unsigned r = 0; r < ITEMS; ++r)
        if (j[r] != kNoMatch) dst_vals[i0 + r] = mine[r];
    }
  } else {
    if (whole) {
      u64x2 x, y;
      x.x = j[0], x.y = j[1 % ITEMS], y.x = j[2 % ITEMS], y.y = j[3 % ITEMS];
      *reinterpret_cast<u64x2*>(where + i0) = x;  // (the workspace is 256-byte aligned)
      *reinterpret_cast<u64x2*>(where + i0 + 2) = y;
    } else {
#pragma unroll
      for (unsigned r = 0; r < ITEMS; ++r)
        if (idx0 + r < tile_n) where[i0 + r] = j[r];
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) found += __shfl_xor(found, o);
  if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = found;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned total = 0;
    for (unsigned w = 0; w < kMatchBlock / 64; ++w) total += s_red[w];
    // (spread over kCounts lines: adds on one address take turns)
    if (total) atomicAdd(&counts[(blockIdx.x % kCounts) * kCountStride], (unsigned long long)total);
  }
}

// The matched keys of all tiles, for the host to see, and the counts clear for the next call. One wavefront,
// behind the kernels of the match: when `done` shows `seq`, what those have written is there.
struct MatchDone {
  unsigned long long count, seq;
};
__global__ void k_match_total(unsigned long long* counts, MatchDone* done, unsigned long long seq) {
  static_assert(kCounts == 64, "one lane per count");
  unsigned long long x = counts[threadIdx.x * kCountStride];
  counts[threadIdx.x * kCountStride] = 0ull;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
  if (threadIdx.x != 0) return;
  done->count = x;
  __hip_atomic_store(&done->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Rows of kq units (floats, or groups of four floats): dst row i op= src row where[i], or with SWAP dst row where[i]
// op= src row i.
template <typename V, bool SWAP>
__global__ __launch_bounds__(kMatchBlock) void k_match_rows(const uint64_t* __restrict__ where, uint64_t n_near,
                                                            uint64_t kq, const V* __restrict__ src,
                                                            V* __restrict__ dst, int op) {
  const uint64_t total = n_near * kq;
  const uint64_t stride = (uint64_t)gridDim.x * kMatchBlock;
  for (uint64_t base = (uint64_t)blockIdx.x * kMatchBlock; base < total; base += stride) {
    // one division per workgroup and turn; a lane is at most kMatchBlock units further on
    const uint64_t row0 = base / kq;
    const uint64_t c = base - row0 * kq + threadIdx.x;
    const uint64_t over = kq >= kMatchBlock ? (c >= kq ? 1u : 0u) : (uint64_t)((unsigned)c / (unsigned)kq);
    const uint64_t row = row0 + over, col = c - over * kq;
    if (row >= n_near) continue;
    const uint64_t j = where[row];
    if (j == kNoMatch) continue;
    const V s = __builtin_nontemporal_load(src + (SWAP ? row : j) * kq + col);
    V* p = dst + (SWAP ? j : row) * kq + col;
    if (op == PSKV_OP_ASSIGN) {
      __builtin_nontemporal_store(s, p);
    } else {
      __builtin_nontemporal_store(combine(op, __builtin_nontemporal_load(p), s), p);
    }
  }
}

// Per device: a stream, the index workspace and, for host-resident calls, staging room. A call
// holds the lock for its whole duration (calls on one device take turns).
struct MatchCtx {
  std::mutex mu;
  hipStream_t stream = nullptr;
  MatchDone* done = nullptr;            // pinned; the last kernel of a call writes it
  unsigned long long seq = 0;           // number of the newest call
  unsigned long long* counts = nullptr;  // kCounts lines, zero between calls
  hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};  // begin/end of the key kernel and of the row kernel
  struct Buf {
    void* ptr = nullptr;
    size_t cap = 0;
  } where, spans, stage[4];
};

int room(MatchCtx::Buf* b, size_t bytes, hipStream_t stream) {
  if (bytes <= b->cap) return PSKV_OK;
  if (b->ptr) {
    PSKV_HIP(hipStreamSynchronize(stream));
    PSKV_HIP(hipFree(b->ptr));
    b->ptr = nullptr;
    b->cap = 0;
  }
  const size_t want = (bytes + (bytes >> 2) + 255) & ~(size_t)255;
  PSKV_HIP(hipMalloc(&b->ptr, want));
  b->cap = want;
  return PSKV_OK;
}

MatchCtx* match_ctx(int device, bool create = true) {
  constexpr int kMaxDevices = 64;
  static std::mutex* mu = new std::mutex();
  static MatchCtx* table[kMaxDevices] = {nullptr};
  if (device < 0 || device >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lk(*mu);
  if (table[device] || !create) return table[device];
  MatchCtx* c = new (std::nothrow) MatchCtx();  // kept until the process ends
  if (!c) return nullptr;
  bool ok = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) == hipSuccess;
  ok = ok && hipHostMalloc(reinterpret_cast<void**>(&c->done), sizeof(MatchDone), hipHostMallocCoherent) == hipSuccess;
  ok = ok && hipMalloc(reinterpret_cast<void**>(&c->counts), kCounts * kCountStride * 8) == hipSuccess;
  ok = ok && hipMemset(c->counts, 0, kCounts * kCountStride * 8) == hipSuccess;
  for (int e = 0; ok && e < 4; ++e) ok = hipEventCreate(&c->ev[e]) == hipSuccess;
  if (!ok) {
    (void)hipGetLastError();
    for (int e = 0; e < 4; ++e)
      if (c->ev[e]) (void)hipEventDestroy(c->ev[e]);
    if (c->done) (void)hipHostFree(c->done);
    if (c->counts) (void)hipFree(c->counts);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
    return nullptr;
  }
  c->done->seq = 0;
  table[device] = c;
  return c;
}

}  // namespace

// Gives back the workspaces and staging buffers the device's match context has grown to (they
// only grow, and a model-size host-resident call leaves several GiB behind).
int match_trim(int device) {
  MatchCtx* c = match_ctx(device, false);
  if (!c) return PSKV_OK;
  DeviceGuard guard(device);
  if (!guard.ok()) return set_error(PSKV_EHIP, "cannot select device %d", device);
  std::lock_guard<std::mutex> lk(c->mu);
  MatchCtx::Buf* bufs[] = {&c->where, &c->spans, &c->stage[0], &c->stage[1], &c->stage[2], &c->stage[3]};
  for (MatchCtx::Buf* b : bufs) {
    if (b->ptr) PSKV_HIP(hipFree(b->ptr));
    b->ptr = nullptr;
    b->cap = 0;
  }
  return PSKV_OK;
}

}  // namespace pskv

using namespace pskv;

extern "C" int pskv_match(int device, const uint64_t* src_keys, size_t n_src, const float* src_vals,
                          const uint64_t* dst_keys, size_t n_dst, float* dst_vals, size_t k, int op,
                          uint64_t* matched, float* kernel_ms, int memkind) {
  clear_error();
  if (matched) *matched = 0;
  if (kernel_ms) kernel_ms[0] = kernel_ms[1] = 0.0f;
  if (op < PSKV_OP_ASSIGN || op > PSKV_OP_DIVIDE)
    return set_error(PSKV_EINVAL, "op %d: only ASSIGN, PLUS, MINUS, TIMES and DIVIDE apply to floats", op);
  if (k == 0) return set_error(PSKV_EINVAL, "k must be at least 1");
  if (memkind != PSKV_MEM_DEVICE && memkind != PSKV_MEM_HOST) return set_error(PSKV_EINVAL, "bad memkind");
  if (n_src == 0 || n_dst == 0) return PSKV_OK;  // parallel_kv_match.h:36
  if (!src_keys || !src_vals || !dst_keys || !dst_vals) return set_error(PSKV_EINVAL, "null buffer");
  if (k > (1ull << 31) || n_src > (1ull << 40) || n_dst > (1ull << 40) ||
      (n_src > n_dst ? n_src : n_dst) > (1ull << 44) / k)  // (2^44 floats: no product below overflows)
    return set_error(PSKV_EINVAL, "sizes beyond what one call handles");
  DeviceGuard guard(device);
  if (!guard.ok()) return set_error(PSKV_EHIP, "cannot select device %d", device);
  MatchCtx* c = match_ctx(device);
  if (!c) return set_error(PSKV_EHIP, "cannot set up the match context of device %d", device);
  std::lock_guard<std::mutex> lk(c->mu);
  hipStream_t st = c->stream;
  const uint64_t* d_src = src_keys;
  const uint64_t* d_dst = dst_keys;
  const float* d_sv = src_vals;
  float* d_dv = dst_vals;
  if (memkind == PSKV_MEM_HOST) {
    const size_t bytes[4] = {n_src * 8, n_dst * 8, n_src * k * 4, n_dst * k * 4};
    const void* from[4] = {src_keys, dst_keys, src_vals, dst_vals};
    for (int b = 0; b < 4; ++b) {
      int rc = room(&c->stage[b], bytes[b], st);
      if (rc) return rc;
      PSKV_HIP(hipMemcpyAsync(c->stage[b].ptr, from[b], bytes[b], hipMemcpyHostToDevice, st));
    }
    d_src = static_cast<const uint64_t*>(c->stage[0].ptr);
    d_dst = static_cast<const uint64_t*>(c->stage[1].ptr);
    d_sv = static_cast<const float*>(c->stage[2].ptr);
    d_dv = static_cast<float*>(c->stage[3].ptr);
  }
  const bool vec = k % 4 == 0 && ((reinterpret_cast<uintptr_t>(d_sv) | reinterpret_cast<uintptr_t>(d_dv)) & 15) == 0;
  const uint64_t kq = vec ? k / 4 : k;
  // The walk goes over the destination's keys, which streams through everything once, unless the source is so much
  // smaller that finding its keys in the destination reads less. Single values: from 16 times on, and where the
  // destination is not a matter of a few microseconds anyway (320,000 into 6.6M keys: 41 -> 36 us, but 44,000 into
  // 1M 25 -> 27, 1.3M into 8.7M 53 -> 108). Longer ones: the row kernel visits the walk's keys, so from twice or four
  // times on (450,000 into 1.6M keys with 3 floats: 53 -> 39 us; 1M into 3M with 4: 58 -> 62).
  const uint64_t ratio = n_dst / n_src;
  const bool swap = k == 1 ? ratio >= 16 && n_dst >= (4u << 20) : ratio >= (kq == 1 ? 4 : 2);
  const uint64_t n_near = swap ? n_src : n_dst, n_far = swap ? n_dst : n_src;
  const uint64_t *near = swap ? d_src : d_dst, *far = swap ? d_dst : d_src;
  const bool few = n_near < kFewKeys || n_far / n_near >= 2;
  const unsigned tile = kMatchBlock * (few ? 1 : kMatchItems);
  const unsigned blocks = (unsigned)((n_near + tile - 1) / tile);
  const bool own = own_search(n_near, n_far, blocks, few);
  if (!own) {
    int rc = room(&c->spans, ((size_t)blocks + 1) * sizeof(uint64_t), st);
    if (rc) return rc;
  }
  uint64_t* spans = static_cast<uint64_t*>(c->spans.ptr);
  if (!own)
    hipLaunchKernelGGL(k_match_spans, dim3((blocks + kSpanTiles - 1) / kSpanTiles), dim3(kSpanBlock), 0, st, far, n_far, near,
                       (uint64_t)blocks, tile, spans);
  // (a launch can carry events of its own, which read the begin and the end of that very dispatch)
  hipEvent_t e0 = kernel_ms ? c->ev[0] : nullptr, e1 = kernel_ms ? c->ev[1] : nullptr;
  hipEvent_t e2 = kernel_ms ? c->ev[2] : nullptr, e3 = kernel_ms ? c->ev[3] : nullptr;
  uint64_t* where = nullptr;
  if (k > 1) {
    int rc = room(&c->where, n_near * sizeof(uint64_t), st);
    if (rc) return rc;
    where = static_cast<uint64_t*>(c->where.ptr);
  }
  auto pick = [&](auto o) {
    constexpr bool OWN = decltype(o)::value;
    return k == 1 ? (swap ? (few ? k_match_keys<true, true, 1, OWN> : k_match_keys<true, true, kMatchItems, OWN>)
                          : (few ? k_match_keys<true, false, 1, OWN> : k_match_keys<true, false, kMatchItems, OWN>))
                  : (few ? k_match_keys<false, false, 1, OWN> : k_match_keys<false, false, kMatchItems, OWN>);
  };
  auto keys = own ? pick(std::true_type()) : pick(std::false_type());
  hipExtLaunchKernelGGL(keys, dim3(blocks), dim3(kMatchBlock), 0, st, e0, e1, 0, far, n_far, near, n_near, spans, where, d_sv,
                        d_dv, op, c->counts);
  if (k > 1) {
    const unsigned grid = grid_for(n_near * kq, kMatchBlock, 1u << 20);
    if (vec) {
      auto rows = swap ? k_match_rows<f32x4, true> : k_match_rows<f32x4, false>;
      hipExtLaunchKernelGGL(rows, dim3(grid), dim3(kMatchBlock), 0, st, e2, e3, 0, where, n_near, kq,
                            reinterpret_cast<const f32x4*>(d_sv), reinterpret_cast<f32x4*>(d_dv), op);
    } else {
      auto rows = swap ? k_match_rows<float, true> : k_match_rows<float, false>;
      hipExtLaunchKernelGGL(rows, dim3(grid), dim3(kMatchBlock), 0, st, e2, e3, 0, where, n_near, kq, d_sv, d_dv, op);
    }
  }
  const unsigned long long seq = ++c->seq;
  hipLaunchKernelGGL(k_match_total, dim3(1), dim3(64), 0, st, c->counts, c->done, seq);
  PSKV_HIP(hipGetLastError());
  if (memkind == PSKV_MEM_HOST)
    PSKV_HIP(hipMemcpyAsync(dst_vals, d_dv, n_dst * k * 4, hipMemcpyDeviceToHost, st));
  if (memkind == PSKV_MEM_HOST || kernel_ms || !seen_in_time(&c->done->seq, seq)) PSKV_HIP(hipStreamSynchronize(st));
  if (matched) *matched = (uint64_t)c->done->count * k;  // values, not keys (:52)
  if (kernel_ms) {
    PSKV_HIP(hipEventElapsedTime(&kernel_ms[0], c->ev[0], c->ev[1]));
    if (k > 1) PSKV_HIP(hipEventElapsedTime(&kernel_ms[1], c->ev[2], c->ev[3]));
  }
  return PSKV_OK;
}

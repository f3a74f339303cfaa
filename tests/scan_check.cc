// The first kernel of a var-len push and of a var-len pull (csrc/table_kernels.h) on the CPU, wavefronts in every
// order: the totals that the last workgroup leaves are the offsets of the parts, whichever wavefront is ahead.
#include <hip/hip_runtime.h>
#include <stdio.h>

#include <algorithm>
#include <vector>

#include "pskv/capi.h"
#include "table_kernels.h"

namespace pskv {
thread_local unsigned long long regrow_lds[1];  // (a kernel that is not run here wants it)
}
using namespace pskv;

struct Launch {
  ReqBatch<1> b;
  bool push;
};

static bool check(bool push, uint64_t n, int longest, const std::vector<unsigned>& order) {
  const unsigned nblk = (unsigned)scan_num_parts(n);
  std::vector<uint64_t> keys(n), cache_keys(n), ref(n), slot_words(8, kEmptyKey);
  std::vector<int32_t> lens(n), cache_lens(n), out_lens(n);
  std::vector<unsigned long long> part(nblk, 7);
  std::vector<Slot> slots(4 * 1024);
  for (Slot& s : slots) s.key = kEmptyKey, s.payload = kPayloadUnset;
  DevState* st = static_cast<DevState*>(aligned_alloc(32, sizeof(DevState)));
  memset(static_cast<void*>(st), 0, sizeof(DevState));
  for (uint64_t i = 0; i < n; ++i) {
    keys[i] = 3 * i + 1;
    lens[i] = longest == 0 ? 4 : (int32_t)((i * 7) % (unsigned)longest);  // (0: rows of four floats, no fact to report)
  }
  Launch l;
  memset(static_cast<void*>(&l), 0, sizeof(l));
  l.push = push;
  TableReq& d = l.b.t[0];
  d.keys = keys.data(), d.lens = lens.data(), d.n = n, d.part = part.data(), d.st = st, d.nblk = nblk;
  d.cache_keys = cache_keys.data(), d.cache_lens = cache_lens.data(), d.ref = ref.data(), d.out_lens = out_lens.data();
  d.slots = slots.data(), d.mask = slots.size() - 1;
  d.tag.epoch = 5;
  std::vector<unsigned long long> want(nblk, 0);
  unsigned long long total = 0;
  for (unsigned p = 0; p < nblk; ++p) {
    want[p] = total;
    if (push)
      for (uint64_t i = p * kScanPart; i < std::min<uint64_t>(n, (p + 1) * kScanPart); ++i) total += (unsigned)lens[i];
  }
  host_waves().grid.x = nblk;
  for (unsigned b = 0; b < nblk; ++b) {
    host_waves().block.x = b, host_waves().block.y = 0;
    host_workgroup(kBlock, order, [](void* a) {
      Launch& x = *static_cast<Launch*>(a);
      if (x.push) k_var_push_begin<1>(x.b); else k_var_pull_lookup<1>(x.b);
    }, &l);
  }
  bool ok = part == want && st->scan_total == total && st->ticket_top == 0 && st->req_flags == 0;
  if (!ok)
    printf("%s of %llu keys, rows up to %d, wavefronts %u %u %u %u: total %llu, expected %llu\n", push ? "push" : "pull",
           (unsigned long long)n, longest, order[0], order[1], order[2], order[3], st->scan_total, total);
  free(st);
  return ok;
}

int main() {
  for (bool push : {true, false})
    for (int longest : {0, 30})
      for (uint64_t n : {1ull, 1023ull, 1024ull, 1025ull, 5000ull, 33ull * 1024 + 1}) {
        std::vector<unsigned> order = {0, 1, 2, 3};
        do {
          if (!check(push, n, longest, order)) return 1;
        } while (n < 5000 && std::next_permutation(order.begin(), order.end()));
      }
  printf("ok\n");
  return 0;
}

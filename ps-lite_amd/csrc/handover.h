// How a workgroup that has waited long enough for the verdict on its launch leaves its share of the work to the workgroup
// that reaches the verdict, which is the last of them to start on it and so is there for certain. Either the share's owner
// gets to know the verdict, or the last workgroup gets to know the share, never both and never neither.
// (constexpr: the host's tests run the same code over a memory of their own.)
#ifndef PSKV_HANDOVER_H_
#define PSKV_HANDOVER_H_

namespace pskv {

// The word of the verdict, which every launch exchanges once: launches so far << 2, whether somebody has left a share to
// the one in flight, the verdict on the newest that is done.
constexpr unsigned long long kVerdictYes = 1, kSharesLeft = 2;
constexpr unsigned long long next_verdict(unsigned long long before, bool yes) {
  return ((before >> 2) + 1) << 2 | (yes ? kVerdictYes : 0);
}
constexpr bool has_verdict(unsigned long long word, unsigned long long before) { return word >> 2 != before >> 2; }

// One thread of the workgroup that leaves; whoever works on the share must be able to see what it needs by now. `before`:
// the word as it was in front of the launch. Returns 1 or 0, the verdict, which has come after all, or -1: the share is the
// last workgroup's. Mem, every operation at its place before the next one:
//   void mark()                                   marks the share as one that is left
//   bool unmark()                                 takes the mark away; false: somebody has taken it already
//   unsigned long long swap(from, to)             exchanges the word of the verdict if it is `from`; returns what it was
// The last workgroup exchanges the word for next_verdict() first, and if kSharesLeft was in it takes the marks away, once
// and one by one, and works on those shares.
template <typename Mem>
constexpr int leave_share(Mem& m, unsigned long long before) {
  m.mark();
  const unsigned long long word = m.swap(before, before | kSharesLeft);
  // (no verdict yet: it will be exchanged for a word that says so, and the mark be found)
  if (!has_verdict(word, before)) return -1;
  return m.unmark() ? (int)(word & kVerdictYes) : -1;
}

}  // namespace pskv
#endif  // PSKV_HANDOVER_H_

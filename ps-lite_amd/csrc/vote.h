// How the workgroups of one launch agree on whether all of them go on, when nobody may go on alone and nobody
// knows that the others have started: every workgroup votes once, the last vote settles the outcome for all of
// them, and a workgroup that tires of waiting for it may leave only by making the outcome a no.
// (constexpr: the host's tests run the same code over a memory of their own.)
#ifndef PSKV_VOTE_H_
#define PSKV_VOTE_H_

namespace pskv {

// The word of the votes: how many there are (low half), those against, and the mark of those that have left.
constexpr unsigned kVoteAgainst = 1u << 16;
constexpr unsigned kVoteLeft = 1u << 31;
constexpr unsigned vote_count(unsigned word) { return word & 0xffffu; }

// One thread of every one of `nblk` (below 2^15) workgroups calls it once; it returns whether the workgroup goes
// on, which is the same in all of them, but that those who left have said no before the last vote, so that the
// others get a no as well. Mem:
//   unsigned add(unsigned)                   adds to the word of the votes and returns what it was
//   unsigned word()                          the word as it is
//   bool swap(unsigned from, unsigned to)    exchanges it if it is `from`
//   bool publish(bool yes)                   called by the last vote: clears the word, lets the others see the
//                                            outcome and returns it
//   int outcome()                            1 or 0, and -1 while it has not been published
//   void pause()
// `looks`: how often a workgroup looks for the outcome before it means to leave.
template <typename Mem>
constexpr bool vote(Mem& m, unsigned nblk, bool agrees, unsigned looks) {
  const unsigned old = m.add(agrees ? 1u : 1u + kVoteAgainst);
  if (vote_count(old) == nblk - 1) return m.publish(agrees && old == vote_count(old));
  for (unsigned i = 0; i < looks; ++i) {
    const int now = m.outcome();
    if (now >= 0) return now != 0;
    m.pause();
  }
  for (;;) {
    const unsigned word = m.word();
    // every vote is in (the word is full, or cleared already): there is nothing left to change, the outcome is a
    // few instructions of a running workgroup away
    if (vote_count(word) == 0u || vote_count(word) == nblk) break;
    if ((word & kVoteLeft) != 0u || m.swap(word, word | kVoteLeft)) return false;
  }
  int now = m.outcome();
  for (; now < 0; now = m.outcome()) m.pause();
  return now != 0;
}

}  // namespace pskv
#endif  // PSKV_VOTE_H_

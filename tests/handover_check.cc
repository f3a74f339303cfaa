// Runs pskv::leave_share (csrc/handover.h) and the last workgroup's side of it under every order in which their steps can
// take turns (a few workgroups, each a context of its own, one switch per access to memory), for two launches in a row, and
// checks that every workgroup's share is worked on once and under the verdict of its launch, and that no mark is left.
// `--keep`: a workgroup that finds the verdict works on its share without a look at its mark, the mistake that look is there
// against; the program then ends with an error.
#include <stdio.h>
#include <string.h>
#include <ucontext.h>

#include <vector>

#include "handover.h"

static bool g_keep = false;
constexpr unsigned kMost = 4;

struct Run {
  unsigned nblk = 0, looks = 0;
  bool yes = false;
  unsigned long long word = 0, before = 0;
  unsigned tickets = 0, marks = 0;
  unsigned done[kMost] = {0};  // how often the share has been worked on
  bool wrong = false, over[kMost] = {false};
  ucontext_t ctx[kMost], main_ctx;
  char stack[kMost][16384];
  unsigned running = 0;
};
static Run* g_run;

static void turn() { swapcontext(&g_run->ctx[g_run->running], &g_run->main_ctx); }
static void work(unsigned share, bool yes) {
  ++g_run->done[share];
  g_run->wrong = g_run->wrong || yes != g_run->yes;
}

struct Mem {
  unsigned me;
  void mark() {
    turn();
    g_run->marks |= 1u << me;
  }
  bool unmark() {
    turn();
    const bool there = (g_run->marks >> me & 1u) != 0;
    g_run->marks &= ~(1u << me);
    return there || g_keep;
  }
  unsigned long long swap(unsigned long long from, unsigned long long to) {
    turn();
    const unsigned long long was = g_run->word;
    if (was == from) g_run->word = to;
    return was;
  }
};

static void body() {
  Run& r = *g_run;
  const unsigned me = r.running;
  turn();
  if (++r.tickets == r.nblk) {
    turn();
    const unsigned long long was = r.word;
    r.word = pskv::next_verdict(r.before, r.yes);
    work(me, r.yes);
    if (was & pskv::kSharesLeft) {
      turn();
      const unsigned left = r.marks;
      r.marks = 0;
      for (unsigned i = 0; i < r.nblk; ++i)
        if (left >> i & 1u) work(i, r.yes);
    }
  } else {
    int verdict = -1;
    for (unsigned l = 0; l < r.looks && verdict < 0; ++l) {
      turn();
      if (pskv::has_verdict(r.word, r.before)) verdict = (int)(r.word & pskv::kVerdictYes);
    }
    Mem m{me};
    if (verdict < 0) verdict = pskv::leave_share(m, r.before);
    if (verdict >= 0) work(me, verdict != 0);
  }
  r.over[me] = true;
  turn();
}

// One launch under the order `taken` (then everyone in turn); the numbers of workgroups that could have taken each turn go
// to `could`.
static bool one(unsigned nblk, unsigned looks, bool yes, const std::vector<unsigned>& taken, std::vector<unsigned>& could) {
  Run r;
  g_run = &r;
  could.clear();
  r.nblk = nblk, r.looks = looks;
  for (int launch = 0; launch < 2; ++launch) {
    r.yes = launch ? !yes : yes;
    r.before = r.word;
    r.tickets = 0;
    memset(r.done, 0, sizeof(r.done));
    memset(r.over, 0, sizeof(r.over));
    for (unsigned i = 0; i < nblk; ++i) {
      getcontext(&r.ctx[i]);
      r.ctx[i].uc_stack.ss_sp = r.stack[i];
      r.ctx[i].uc_stack.ss_size = sizeof(r.stack[i]);
      r.ctx[i].uc_link = &r.main_ctx;
      makecontext(&r.ctx[i], body, 0);
    }
    unsigned next = 0;
    for (;;) {
      std::vector<unsigned> live;
      for (unsigned i = 0; i < nblk; ++i)
        if (!r.over[i]) live.push_back(i);
      if (live.empty()) break;
      const size_t step = could.size();
      could.push_back((unsigned)live.size());
      r.running = live[step < taken.size() ? taken[step] : next++ % live.size()];
      swapcontext(&r.main_ctx, &r.ctx[r.running]);
    }
    for (unsigned i = 0; i < nblk; ++i)
      if (r.done[i] != 1) return printf("share %u worked on %u times\n", i, r.done[i]), false;
    if (r.wrong) return printf("a share under another verdict\n"), false;
    if (r.marks || r.word != pskv::next_verdict(r.before, r.yes))
      return printf("marks %x, word %llx\n", r.marks, r.word), false;
  }
  return true;
}

int main(int argc, char** argv) {
  g_keep = argc > 1 && !strcmp(argv[1], "--keep");
  unsigned long long runs = 0;
  const struct { unsigned nblk, looks, depth; } sizes[] = {{1, 0, 4}, {2, 0, 10}, {2, 1, 11}, {3, 0, 11}, {3, 1, 10}, {4, 0, 8}};
  for (auto s : sizes) {
    for (int yes = 0; yes < 2; ++yes) {
      std::vector<unsigned> taken, could;
      for (;;) {  // every order of the first `depth` turns
        if (!one(s.nblk, s.looks, yes != 0, taken, could)) return printf("%u workgroups, %u looks\n", s.nblk, s.looks), 1;
        ++runs;
        const size_t n = could.size() < s.depth ? could.size() : s.depth;
        std::vector<unsigned> now(taken);
        now.resize(n, 0);
        size_t at = n;
        while (at > 0 && now[at - 1] + 1 >= could[at - 1]) --at;
        if (at == 0) break;
        ++now[at - 1];
        now.resize(at);
        taken = now;
      }
    }
  }
  printf("ok: %llu runs\n", runs);
  return 0;
}

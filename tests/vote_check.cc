// Runs pskv::vote (csrc/vote.h) under every order in which its steps can take turns (a few workgroups, each a
// context of its own, one switch per access to memory) and checks that the workgroups that come out with a yes are
// all of them or none, that the outcome is a yes when all agree and nobody left, and that the word of the votes is
// left at zero. `--leave-unmarked`: a workgroup that leaves does not say so, the mistake the mark is there against;
// the program then ends with an error.
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <ucontext.h>

#include <vector>

#include "vote.h"

static bool g_unmarked = false;

struct Run {
  unsigned nblk, looks, differs;  // (differs: bit i = workgroup i votes against)
  unsigned word = 0;
  int settled = -1;
  bool left = false;
  std::vector<int> answer;  // -1: not done
  std::vector<ucontext_t> ctx;
  std::vector<std::vector<char>> stack;
  ucontext_t main_ctx;
  unsigned running = 0;
};
static Run* g_run;

static void turn() { swapcontext(&g_run->ctx[g_run->running], &g_run->main_ctx); }

struct Mem {
  Run& r;
  unsigned add(unsigned x) {
    turn();
    const unsigned old = r.word;
    r.word += x;
    return old;
  }
  unsigned word() {
    turn();
    return r.word;
  }
  bool swap(unsigned from, unsigned to) {
    turn();
    if (g_unmarked) return r.left = true;
    if (r.word != from) return false;
    r.word = to;
    return r.left = true;
  }
  bool publish(bool yes) {
    turn();
    r.word = 0;
    turn();
    r.settled = yes ? 1 : 0;
    return yes;
  }
  int outcome() {
    turn();
    return r.settled;
  }
  void pause() {}
};

static void body() {
  Run& r = *g_run;
  const unsigned me = r.running;
  Mem m{r};
  r.answer[me] = pskv::vote(m, r.nblk, (r.differs >> me & 1u) == 0u, r.looks) ? 1 : 0;
  turn();
}

// One run under the order `taken` (then always the first that can go on); the numbers of workgroups that could
// have taken each turn go to `could`.
static bool one(unsigned nblk, unsigned looks, unsigned differs, const std::vector<unsigned>& taken,
                std::vector<unsigned>& could) {
  Run r;
  r.nblk = nblk, r.looks = looks, r.differs = differs;
  r.answer.assign(nblk, -1);
  r.ctx.resize(nblk);
  r.stack.assign(nblk, std::vector<char>(32768));
  g_run = &r;
  for (unsigned i = 0; i < nblk; ++i) {
    getcontext(&r.ctx[i]);
    r.ctx[i].uc_stack.ss_sp = r.stack[i].data();
    r.ctx[i].uc_stack.ss_size = r.stack[i].size();
    r.ctx[i].uc_link = &r.main_ctx;
    makecontext(&r.ctx[i], body, 0);
  }
  could.clear();
  unsigned next = 0;
  for (size_t step = 0; step < 400; ++step) {
    std::vector<unsigned> live;
    for (unsigned i = 0; i < nblk; ++i)
      if (r.answer[i] < 0) live.push_back(i);
    if (live.empty()) break;
    could.push_back((unsigned)live.size());
    // (past the order that is tried everyone gets a turn, so that whoever waits sees an end of it)
    const unsigned who = live[step < taken.size() ? taken[step] : next++ % live.size()];
    r.running = who;
    swapcontext(&r.main_ctx, &r.ctx[who]);
  }
  unsigned yes = 0;
  for (int a : r.answer) {
    if (a < 0) return printf("a workgroup waits for good\n"), false;
    yes += (unsigned)a;
  }
  if (yes != 0 && yes != nblk) return printf("%u of %u workgroups go on\n", yes, nblk), false;
  if (yes && differs) return printf("they go on although one voted against\n"), false;
  if (!yes && !differs && !r.left) return printf("nobody goes on although all agree and nobody left\n"), false;
  if (r.word != 0 || r.settled != (yes ? 1 : 0)) return printf("word %x, outcome %d\n", r.word, r.settled), false;
  return true;
}

int main(int argc, char** argv) {
  g_unmarked = argc > 1 && !strcmp(argv[1], "--leave-unmarked");
  unsigned long long runs = 0;
  const struct { unsigned nblk, looks, depth; } sizes[] = {{1, 0, 4}, {2, 0, 10}, {2, 1, 10}, {2, 2, 10}, {3, 0, 8}, {3, 1, 8}, {4, 0, 6}};
  for (auto s : sizes) {
    for (unsigned differs = 0; differs < (1u << s.nblk); ++differs) {
      std::vector<unsigned> taken, could;
      for (;;) {  // every order of the first `depth` turns
        if (!one(s.nblk, s.looks, differs, taken, could)) {
          printf("%u workgroups, %u looks, against %x\n", s.nblk, s.looks, differs);
          return 1;
        }
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
        taken.resize(at);
      }
    }
  }
  printf("ok: %llu runs\n", runs);
  return 0;
}

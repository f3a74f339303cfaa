// Tables that grow together (csrc/growths.h), with every launch failing in turn, and every release: a table has one array,
// with its keys in it, and the other one has been given back once.
// --forget: the tables keep their new arrays whatever fails.
#include <stdio.h>
#include <string.h>

#include <memory>

#include "growths.h"

using namespace pskv;

struct Array {
  bool keys = false;
  int released = 0;
};
struct Table {
  Array* slots;
  uint64_t cap;
};
typedef Growth<Table, Array> One;

struct Launches {
  int calls = 0, failing = -1, released = 0, failing_release = -1;
  bool forget = false;
  unsigned most = 0;
  int next() { return calls++ == failing ? 7 : 0; }
  int scatter(const One& g) {
    const int rc = next();
    if (!rc) g.t->slots->keys = true;
    return rc;
  }
  int stream(One* const* some, unsigned count, bool& begun) {
    most = count > most ? count : most;
    if (int rc = next()) return begun = forget, rc;
    begun = true;
    const int rc = next();
    for (unsigned i = 0; i < count; ++i) some[i]->t->slots->keys = true, some[i]->from->keys = false;
    return rc;
  }
  int release(Table*, Array* a) {
    ++a->released;
    return released++ == failing_release ? 9 : 0;
  }
};

struct Arrays {
  Array* made;
  int release_rc, allocate_rc;
  int release(Array* a) { return ++a->released, release_rc; }
  int allocate(uint64_t, Array** to) {
    if (!allocate_rc) *to = made;
    return allocate_rc;
  }
};

int main(int argc, char** argv) {
  const bool forget = argc > 1 && !strcmp(argv[1], "--forget");
  for (unsigned tables : {0u, 1u, 3u, 16u, 17u, 40u}) {
    for (unsigned kind = 0; kind < 3; ++kind) {  // which of them scatter: none, all, every third
      for (int fail = -1; fail < 90; ++fail) {
        std::vector<std::unique_ptr<Array>> arrays;
        std::vector<Table> all(tables);
        std::vector<One> todo;
        for (unsigned i = 0; i < tables; ++i) {
          for (int a = 0; a < 2; ++a) arrays.emplace_back(new Array());
          arrays[2 * i]->keys = true;
          const uint64_t factor = kind == 1 || (kind == 2 && i % 3 == 1) ? 16 : 4;
          all[i] = Table{arrays[2 * i + 1].get(), 100 * factor};
          todo.push_back(One{&all[i], arrays[2 * i].get(), 100, false});
        }
        Launches l;
        l.forget = forget;
        if (fail < 50) l.failing = fail; else l.failing_release = fail - 50;
        const int rc = move_growths(todo, 16u, (uint64_t)8, l);
        const bool failed = l.failing >= 0 && l.failing < l.calls;
        if (rc != (failed ? 7 : l.failing_release >= 0 && l.failing_release < l.released ? 9 : 0)) return printf("rc %d\n", rc), 1;
        if (l.most > 16) return printf("%u tables in a launch\n", l.most), 1;
        for (unsigned i = 0; i < tables; ++i) {
          Array *old = arrays[2 * i].get(), *fresh = arrays[2 * i + 1].get(), *mine = all[i].slots;
          if (mine != old && mine != fresh) return printf("no array\n"), 1;
          if (!mine->keys) return printf("table %u of %u, launch %d fails: no keys\n", i, tables, fail), 1;
          if (all[i].cap != (mine == old ? 100u : todo[i].t->cap) || (mine == fresh && all[i].cap == 100)) return printf("size\n"), 1;
          if (mine->released || (mine == old ? fresh : old)->released != 1) return printf("given back %d and %d times\n", old->released, fresh->released), 1;
          if (!failed && mine != fresh) return printf("not moved\n"), 1;
        }
      }
    }
  }
  // the array that a table moves to: its spare one, or a new one, and where there is none no trace of the spare
  for (int which = 0; which < 5; ++which) {
    Array old, made;
    Arrays ops{&made, which == 3 ? 5 : 0, which == 4 ? 6 : 0};
    Array *spare = which == 0 ? nullptr : &old, *fresh = nullptr;
    uint64_t cap = spare ? (which == 1 ? 512 : 128) : 0, want = 256;
    const int rc = next_array(spare, cap, want, fresh, ops);
    const bool large = which == 1, failed = which >= 3;
    if (rc != (which == 3 ? 5 : which == 4 ? 6 : 0) || spare || cap) return printf("spare left: %d\n", which), 1;
    if (old.released != (which >= 2 ? 1 : 0)) return printf("spare given back %d times\n", old.released), 1;
    if (!failed && (fresh != (large ? &old : &made) || want != (large ? 512u : 256u))) return printf("array %d\n", which), 1;
    if (failed && fresh) return printf("an array in spite of everything\n"), 1;
  }
  printf("ok\n");
  return 0;
}

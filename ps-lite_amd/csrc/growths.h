// Slot arrays that are to move, all tables' of a request with as few launches as there can be. (No GPU code: the host's tests
// run it over tables of their own.)
#ifndef PSKV_GROWTHS_H_
#define PSKV_GROWTHS_H_
#include <stdint.h>

#include <vector>

namespace pskv {

// A table that has been given its new array (slots, cap) already, and the one that its keys are in.
template <typename Table, typename Slots>
struct Growth {
  Table* t;
  Slots* from;
  uint64_t cap;  // of `from`
  bool moved;
};

// Moves them. A table whose move could not be queued keeps its old array, whichever one of the others failed: its new array
// has nothing in it. Returns the first error. Ops:
//   int scatter(const Growth&)                           one that becomes more than `most_factor` times as large
//   int stream(Growth* const*, unsigned count, bool& begun)   up to `most_tables` others. It is two launches, of which the
//                        first (`begun`) leaves in the old arrays nothing but keys for the second: should that one alone
//                        fail, no array has all keys, and the tables keep the new ones, which have most
//   int release(Table*, Slots*)                          an array that the table does not have any more
template <typename Ops, typename Table, typename Slots>
int move_growths(std::vector<Growth<Table, Slots>>& todo, unsigned most_tables, uint64_t most_factor, Ops& ops) {
  int rc = 0;
  std::vector<Growth<Table, Slots>*> some;
  auto stream = [&] {
    if (some.empty() || rc) return;
    bool begun = false;
    rc = ops.stream(some.data(), (unsigned)some.size(), begun);
    for (auto* g : some) g->moved = !rc || begun;
    some.clear();
  };
  for (auto& g : todo) {
    if (rc) break;
    if (g.t->cap / g.cap > most_factor) {
      rc = ops.scatter(g);
      g.moved = !rc;
      continue;
    }
    some.push_back(&g);
    if (some.size() == most_tables) stream();
  }
  stream();
  for (auto& g : todo) {
    Slots* gone = g.from;
    if (!g.moved) {
      gone = g.t->slots;
      g.t->slots = g.from;
      g.t->cap = g.cap;
    }
    const int r = ops.release(g.t, gone);
    if (!rc) rc = r;
  }
  return rc;
}

// The array that a table which needs `want` slots moves to: the spare one (`spare_cap` slots, or null) where that is large
// enough, and `want` is its size then, or else a new one, and the spare goes. The table has no spare after it. Ops:
//   int release(Slots*)     int allocate(uint64_t slots, Slots** fresh)
template <typename Ops, typename Slots>
int next_array(Slots*& spare, uint64_t& spare_cap, uint64_t& want, Slots*& fresh, Ops& ops) {
  Slots* const was = spare;
  const uint64_t cap = spare_cap;
  spare = nullptr;
  spare_cap = 0;
  if (was && cap >= want) {
    fresh = was;
    want = cap;
    return 0;
  }
  const int rc = was ? ops.release(was) : 0;
  return rc ? rc : ops.allocate(want, &fresh);
}

}  // namespace pskv
#endif  // PSKV_GROWTHS_H_

// Checks of the parameter ring's bookkeeping (csrc/slot_ring.hpp), host only.
// Prints "done" and exits 0; a failed check names its line and exits 1.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "slot_ring.hpp"

#define CHECK(x)                                       \
  do {                                                 \
    if (!(x)) {                                        \
      std::printf("line %d: %s\n", __LINE__, #x);      \
      std::exit(1);                                    \
    }                                                  \
  } while (0)

int main() {
  std::vector<int> waited;
  auto wait = [&](int first) { waited.push_back(first); };
  {  // single slots: as many queued as there are slots before the first wait
    g4::SlotRing r(64);
    for (int i = 0; i < 64; ++i) {
      CHECK(r.take(1, wait) == i);
      r.queued(i);
    }
    CHECK(waited.empty());
    CHECK(r.take(1, wait) == 0);
    CHECK(waited == std::vector<int>{0});
    // the run just given out is held: the ring comes round to it and refuses
    for (int i = 1; i < 64; ++i) {
      CHECK(r.take(1, wait) == i);
      r.queued(i);
    }
    CHECK(r.take(1, wait) == -1);
    CHECK(waited.size() == 64);
    r.queued(0);
    CHECK(r.take(1, wait) == 0);
  }
  waited.clear();
  {  // runs: no split over the end, one wait per run, the rest of it free then
    g4::SlotRing r(10);
    CHECK(r.take(4, wait) == 0);
    r.queued(0);
    CHECK(r.take(4, wait) == 4);
    r.queued(4);
    CHECK(r.take(3, wait) == 0);  // two left at the end: from the start again
    CHECK(waited == std::vector<int>{0});
    r.queued(0);
    CHECK(r.take(1, wait) == 3);  // freed with its run
    CHECK(waited.size() == 1);
    r.drop(3);
    CHECK(r.take(2, wait) == 4);
    CHECK((waited == std::vector<int>{0, 4}));
    CHECK(r.take(5, wait) == -1);  // from the start again: run 0 is queued, 4 held
    CHECK(waited.size() == 2);     // a refusal waits for nothing
    CHECK(r.take(4, wait) == 6);
  }
  {  // sizes that never fit
    g4::SlotRing r(4);
    CHECK(r.take(0, wait) == -1);
    CHECK(r.take(5, wait) == -1);
    CHECK(r.take(4, wait) == 0);
    CHECK(r.take(1, wait) == -1);
  }
  {  // a wait that fails leaves the run to be waited for again
    g4::SlotRing r(2);
    CHECK(r.take(2, wait) == 0);
    r.queued(0);
    bool thrown = false;
    try {
      r.take(1, [](int) { throw 1; });
    } catch (int) {
      thrown = true;
    }
    CHECK(thrown);
    waited.clear();
    CHECK(r.take(2, wait) == 0);
    CHECK(waited == std::vector<int>{0});
  }
  std::puts("done");
  return 0;
}

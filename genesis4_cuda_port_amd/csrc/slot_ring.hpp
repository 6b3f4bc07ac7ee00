// slot_ring.hpp - bookkeeping of a ring of equal slots, taken as runs of
// consecutive ones (host only; the memory and the events are the owner's).
#pragma once

#include <vector>

namespace g4 {

// A run is held from take() until queued() or drop(): held slots are never
// given out again.  After queued() the work that reads the run is on its way,
// and take() waits for it before it gives any of the run's slots out anew.
class SlotRing {
 public:
  explicit SlotRing(int slots) : slot_(static_cast<size_t>(slots)) {}

  // First slot of a run of n, which is then held, or -1 (and nothing changed)
  // where a held run is in the way.  wait(first) returns when the work of the
  // queued run that starts at `first` is done.
  template <class Wait>
  int take(int n, Wait&& wait) {
    const int size = static_cast<int>(slot_.size());
    if (n < 1 || n > size) return -1;
    const int at = next_ + n > size ? 0 : next_;
    for (int k = at; k < at + n; ++k)
      if (slot_[k].state == Held) return -1;
    for (int k = at; k < at + n; ++k)
      if (slot_[k].state == Queued) {
        const int first = slot_[k].first;
        wait(first);
        mark(first, Free);
      }
    for (int k = at; k < at + n; ++k) slot_[k] = Slot{Held, at, n};
    next_ = (at + n) % size;
    return at;
  }
  void queued(int first) { mark(first, Queued); }
  void drop(int first) { mark(first, Free); }

 private:
  enum State { Free, Held, Queued };
  struct Slot {
    State state = Free;
    int first = 0, len = 0;  // of its run
  };
  void mark(int first, State s) {
    const int len = slot_[first].len;
    for (int k = first; k < first + len; ++k) slot_[k].state = s;
  }
  std::vector<Slot> slot_;
  int next_ = 0;
};

}  // namespace g4

// When a staging slot may be written again.
#pragma once

namespace huvi {

// Held while a call queues the work that reads a slot.  Whichever way the call
// returns, the slot is then busy until the event that record() leaves behind that
// work, or, where no event could be recorded, the work has been waited for.
template <class Slot, class Record, class Wait>
struct SlotMark {
  Slot* slot;
  Record record;  // whether the event was recorded
  Wait wait;
  SlotMark(Slot* s, Record r, Wait w) : slot(s), record(r), wait(w) {}
  SlotMark(const SlotMark&) = delete;
  ~SlotMark() {
    slot->busy = record();
    if (!slot->busy) wait();
  }
};

}  // namespace huvi

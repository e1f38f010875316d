// A host's wait for a word in host memory that a kernel on some stream sets.
// Plain C++: the same code runs in the CPU tests.
#pragma once

namespace rbdi {

// Reads of the word before the first pause, and pauses (yields of the thread)
// before the stream is asked about: a kernel that is merely behind is met by
// the reads, and only one that is late by some hundred microseconds costs calls
// into the runtime.
constexpr int kSlotReads = 1 << 12;
constexpr int kSlotPauses = 1 << 10;

// Until arrived() is true, and then 0.  pending(&err) says whether the work
// that sets the word may still be running; once it is not, the word is read one
// last time, and if it has not arrived the wait ends with err, or with `lost`
// where there was no error.
template <class Arrived, class Pause, class Pending>
int wait_for_word(Arrived&& arrived, Pause&& pause, Pending&& pending, int lost) {
  for (int reads = 0; reads < kSlotReads; ++reads)
    if (arrived()) return 0;
  for (;;) {
    for (int pauses = 0; pauses < kSlotPauses; ++pauses) {
      if (arrived()) return 0;
      pause();
    }
    int err = 0;
    if (pending(&err)) continue;
    if (arrived()) return 0;
    return err ? err : lost;
  }
}

}  // namespace rbdi

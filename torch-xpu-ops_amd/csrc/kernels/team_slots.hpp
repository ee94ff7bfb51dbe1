// Which slot of library-owned exchange memory a team launch uses: every stream has its own (no HIP
// types in here).
#pragma once
#include <stdint.h>

#include <atomic>

namespace rownorm {

// Calls on one stream run one after the other, so a slot that belongs to a stream never serves two
// running calls.  (Slots handed out by a call counter do as soon as two streams are queued deep
// enough: calls with equal counters modulo the slots then overwrite each other's words, and every
// workgroup of both waits out its bound.)  A slot is taken by the first such call of a stream and
// kept; a stream that comes when all N are taken gets none, and its calls take the launches that
// exchange nothing.  A handle that the runtime uses again for a later stream finds the slot of the
// earlier one.
template <int N>
class StreamSlots {
 public:
  // The slot of the stream with this key (not 0), or -1.
  int of(uintptr_t key) {
    for (int i = 0; i < N; ++i) {
      uintptr_t k = key_[i].load(std::memory_order_relaxed);
      if (k == 0 && key_[i].compare_exchange_strong(k, key, std::memory_order_relaxed)) return i;
      if (k == key) return i;  // (also when another thread has just entered it)
    }
    return -1;
  }

 private:
  std::atomic<uintptr_t> key_[N] = {};
};

}  // namespace rownorm

// Which slot of library-owned exchange memory a team launch uses: every stream has its own; and the order
// of the team launches of different streams (no HIP types in here).
#pragma once
#include <stdint.h>

#include <atomic>
#include <mutex>

#include "plan.hpp"

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

// Ids of team calls: kTeamCallIds of them in turn, then the same again.  A word that an earlier call left in a slot
// carries that call's id, so a slot must not meet an id a second time before it is cleared: of() says when, with the
// first call after the ids have come round.
template <int N>
class TeamIds {
 public:
  // The id of call number n (over all slots) in `slot`; *clear: the slot's memory must be zeroed first.  (One
  // thread at a time for a slot.)
  unsigned int of(uint64_t n, int slot, bool* clear) {
    const uint64_t turn = n / kTeamCallIds;
    *clear = turn_[slot] != turn;
    turn_[slot] = turn;
    return (unsigned int)(n % kTeamCallIds) + 1;
  }

 private:
  uint64_t turn_[N] = {};
};

// One team launch at a time on a device.  The workgroups of a team wait for one another, so a launch must be able
// to have all of them resident.  Two such launches can take that from each other whatever their teams' sizes: the
// XCDs dispatch by themselves, each holds workgroups of the one where the other's are missing, and workgroups that
// need a whole compute unit find none where small ones have half of each; every wait of both then runs out (seen about
// once in 250 rounds of three streams that mix the two kinds: a second each).  Kernels that wait for nobody end by
// themselves and need no order.
//
// A launch on another stream than the last one waits on the device for an event behind the last one.  While streams
// take turns every launch records that event; kQuietCalls launches on one stream end that, so a program on one stream
// pays for no event (recording costs a launch some microseconds).  The first launch elsewhere then puts the event behind
// whatever the earlier stream has been given since -- unless that stream is under capture just now, where an event would
// become part of the graph: that call goes without teams.
//
// Runtime: Stream; bool capturing(Stream), void record(Stream) (the device's one event, behind the stream's work so
// far; no effect if the stream is gone, whose work was over or is not waited for), void wait(Stream).
template <class Runtime>
class TeamOrder {
 public:
  using Stream = typename Runtime::Stream;
  static constexpr int kQuietCalls = 256;

  // Before a team launch on a stream (`key`: as for StreamSlots; per_thread: its handle means another stream in another
  // thread, so its event cannot be left for later).  False: launch no team.  True: leave() must follow the launch, on
  // the same thread; other threads' team launches on the device are held up until then.
  bool enter(Runtime& rt, uintptr_t key, Stream stream, bool per_thread) {
    mutex_.lock();
    const bool other = last_key_ != 0 && last_key_ != key;
    if (other && !recorded_) {
      if (rt.capturing(last_)) {
        mutex_.unlock();
        return false;
      }
      rt.record(last_);
    }
    // (a per-thread key can come back in a new thread: its launches always wait for the one before)
    if (other || (per_thread && recorded_)) rt.wait(stream);
    if (other) turns_ = kQuietCalls;
    last_key_ = key;
    last_ = stream;
    per_thread_ = per_thread;
    return true;
  }
  void leave(Runtime& rt) {
    recorded_ = turns_ > 0 || per_thread_;
    if (turns_ > 0) --turns_;
    if (recorded_) rt.record(last_);
    mutex_.unlock();
  }

 private:
  std::mutex mutex_;
  uintptr_t last_key_ = 0;
  Stream last_{};
  bool recorded_ = false, per_thread_ = false;
  int turns_ = 0;  // launches that still record the event
};

}  // namespace rownorm

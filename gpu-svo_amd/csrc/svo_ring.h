// svo_ring.h -- the host's side of the pinned ring: waits for what the device
// puts there, and how the pieces of a read-out reach the caller's memory.  What
// is done to the device comes in as callables.
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <thread>
#include <vector>

namespace svo {

// The pauses of a thread that waits for the device or for another thread.  For
// SPIN it polls (or yields): a lookup is answered within 100 us and a piece of a
// read-out arrives 10 us after the one before.  What takes longer stands behind
// other work, a build's emission on the same hardware queue for instance, and
// may take milliseconds: then it sleeps for an eighth of the time waited so far,
// a millisecond at most.
class Backoff {
  using Clock = std::chrono::steady_clock;

 public:
  static constexpr Clock::duration SPIN = std::chrono::microseconds(200),
                                   NAP_MAX = std::chrono::milliseconds(1);
  // Sleeps once SPIN is over; returns whether it is.
  bool nap() {
    const Clock::duration waited = Clock::now() - start_;
    if (waited <= SPIN) return false;
    std::this_thread::sleep_for(std::min(waited / 8, NAP_MAX));
    return true;
  }
  void pause() {
    if (!nap()) std::this_thread::yield();
  }

 private:
  Clock::time_point start_ = Clock::now();
};

// Waits until n flags hold `number`; false when busy() says that the device has
// ended its work and one of them does not.  It is asked every ASK polls, about
// 15 us, or after each sleep.  (Asking costs a lookup 4 us and saves a
// synchronization of the device that follows as much: the runtime then has the
// marker of the kernel's end already.)
template <class Busy>
bool wait_flags(const uint32_t* flags, uint32_t n, uint32_t number, Busy busy) {
  constexpr uint32_t ASK = 4096;
  Backoff wait;
  for (uint32_t b = 0, polls = 0; b < n;) {
    if (__atomic_load_n(flags + b, __ATOMIC_ACQUIRE) == number) {
      ++b;
    } else if (++polls >= ASK) {
      polls = wait.nap() ? ASK : 0;
      if (!busy() && __atomic_load_n(flags + b, __ATOMIC_ACQUIRE) != number) return false;
    }
  }
  return true;
}

// Copies `bytes` bytes to dst through the `slots` pieces of `piece` bytes at
// `ring` (at most 64).  launch(at, n, slot) has the device put bytes
// [at, at + n), at most the whole ring, into the ring from slot `slot` on, and
// returns a status; wait(slot) waits until the last launch's piece for a slot
// is there, and returns one.  start(work) returns a thread that runs work(), or
// throws.  Up to `helpers` threads and the caller's empty the slots; where none
// can be started the caller's does all.  Returns the first status that is not
// 0 with all helpers ended.
template <class Launch, class Wait, class Start>
int empty_ring(char* dst, size_t bytes, const char* ring, size_t piece, size_t slots,
               size_t helpers, Launch launch, Wait wait, Start start) {
  const size_t n = (bytes + piece - 1) / piece;
  std::atomic<size_t> arrived{0}, claimed{0};
  std::atomic<bool> stop{false};
  std::atomic<size_t> emptied[64] = {};  // pieces copied out of each slot
  auto is_free = [&](size_t i) {         // the slot of piece i
    return emptied[i % slots].load(std::memory_order_acquire) >= i / slots;
  };
  auto take = [&](size_t i) {
    std::memcpy(dst + i * piece, ring + i % slots * piece, std::min(piece, bytes - i * piece));
    emptied[i % slots].store(i / slots + 1, std::memory_order_release);
  };
  auto work = [&] {
    for (size_t i; (i = claimed.fetch_add(1)) < n;) {
      Backoff wait;
      while (arrived.load(std::memory_order_acquire) <= i) {
        if (stop.load()) return;
        wait.pause();
      }
      take(i);
    }
  };
  std::vector<std::thread> threads;
  try {
    const size_t want = std::min(helpers, n / 2);
    threads.reserve(want);
    for (size_t k = 0; k < want; ++k) threads.emplace_back(start(work));
  } catch (...) {  // no more threads: those that started, or this one, do it
  }
  int st = 0;
  size_t sent = 0;
  for (size_t i = 0; i < n; ++i) {
    // as many pieces as have free slots, half a ring at a time
    if (sent <= i || (sent < n && sent - i <= slots / 2)) {
      size_t end = sent;
      while (end < n && is_free(end)) ++end;
      if (end - sent >= std::min(slots / 2, n - sent) || sent <= i) {
        Backoff wait;
        while (end <= i) {  // the slot of piece i is being emptied
          if (is_free(end)) ++end;
          else wait.pause();
        }
        st = launch(sent * piece, std::min(bytes, end * piece) - sent * piece, sent % slots);
        if (st) break;
        sent = end;
      }
    }
    st = wait(i % slots);
    if (st) break;
    arrived.store(i + 1, std::memory_order_release);
    if (threads.empty()) take(claimed.fetch_add(1));
  }
  if (st) stop.store(true);
  else work();
  for (auto& t : threads) t.join();
  return st;
}

}  // namespace svo

// svo_ring.h -- the host's side of the pinned ring: how the pieces of a
// read-out that the device puts there reach the caller's memory.  What is done
// to the device comes in as callables.
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>
#include <vector>

namespace svo {

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
      while (arrived.load(std::memory_order_acquire) <= i) {
        if (stop.load()) return;
        std::this_thread::yield();
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
        while (end <= i) {  // the slot of piece i is being emptied
          if (is_free(end)) ++end;
          else std::this_thread::yield();
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

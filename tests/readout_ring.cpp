// The read-out's host loop (empty_ring) on a device that a thread stands for.
//   readout_ring BYTES HELPERS DELAY_US FAIL_AT
// HELPERS threads can be started, the next start throws; the device takes
// DELAY_US a piece; launch or wait number FAIL_AT (0: none) returns an error.
// Prints the status, then "same" when the bytes came out as they went in.
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <deque>
#include <mutex>
#include <system_error>

#include "svo_ring.h"

int main(int argc, char** argv) {
  if (argc != 5) return 2;
  const size_t bytes = strtoull(argv[1], nullptr, 10), helpers = strtoull(argv[2], nullptr, 10);
  const auto delay = std::chrono::microseconds(atoi(argv[3]));
  const int fail_at = atoi(argv[4]);
  constexpr size_t PIECE = 512 << 10, SLOTS = 16;
  std::vector<char> src(bytes), dst(bytes + 64, 0x55), ring(PIECE * SLOTS);
  uint32_t x = 1;
  for (char& c : src) c = (char)((x = x * 1664525u + 1013904223u) >> 24);

  struct Launch {
    size_t at, n, slot;
  };
  std::mutex mu;
  std::condition_variable cv;
  std::deque<Launch> queue;
  bool end = false;
  std::atomic<uint32_t> put[SLOTS] = {};  // pieces that the device has put into each slot
  uint32_t due[SLOTS] = {};               // and those it was asked for
  std::thread device([&] {
    for (;;) {
      std::unique_lock<std::mutex> lk(mu);
      cv.wait(lk, [&] { return end || !queue.empty(); });
      if (queue.empty()) return;
      Launch l = queue.front();
      queue.pop_front();
      lk.unlock();
      for (size_t a = 0; a < l.n; a += PIECE, l.slot = (l.slot + 1) % SLOTS) {
        if (delay.count()) std::this_thread::sleep_for(delay);
        std::memcpy(&ring[l.slot * PIECE], &src[l.at + a], std::min(PIECE, l.n - a));
        put[l.slot].fetch_add(1, std::memory_order_release);
      }
    }
  });
  int calls = 0;
  size_t started = 0;
  const int st = svo::empty_ring(
      dst.data(), bytes, ring.data(), PIECE, SLOTS, 3,
      [&](size_t at, size_t n, size_t slot) {
        if (++calls == fail_at) return -4;
        for (size_t i = 0; i * PIECE < n; ++i) ++due[(slot + i) % SLOTS];
        std::lock_guard<std::mutex> lk(mu);
        queue.push_back({at, n, slot});
        cv.notify_one();
        return 0;
      },
      [&](size_t slot) {
        if (++calls == fail_at) return -4;
        while (put[slot].load(std::memory_order_acquire) != due[slot]) std::this_thread::yield();
        return 0;
      },
      [&](auto& work) {
        if (started == helpers)
          throw std::system_error(std::make_error_code(std::errc::resource_unavailable_try_again));
        ++started;
        return std::thread(work);
      });
  {
    std::lock_guard<std::mutex> lk(mu);
    end = true;
    cv.notify_one();
  }
  device.join();
  bool same = std::memcmp(src.data(), dst.data(), bytes) == 0;
  for (size_t i = bytes; i < dst.size(); ++i) same = same && dst[i] == 0x55;
  printf("%d %s\n", st, same ? "same" : "differ");
  return 0;
}

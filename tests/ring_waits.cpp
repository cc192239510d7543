// How long the waits for the ring keep cores busy, on a device that answers
// late.
//   ring_waits lookup MS   one wait whose flags are set after MS milliseconds
//   ring_waits read MS     a read-out with three helpers, its first piece late
//   ring_waits dead MS     flags that are never set; the device ends after MS
//   ring_waits last MS     flags that are set when the device ends, after MS
// Prints the result and the process's CPU milliseconds in the wait.
#include <cstdio>
#include <cstdlib>
#include <ctime>
#include <string>

#include "svo_ring.h"

static double cpu_ms() {
  timespec t;
  clock_gettime(CLOCK_PROCESS_CPUTIME_ID, &t);
  return 1e3 * (double)t.tv_sec + 1e-6 * (double)t.tv_nsec;
}

int main(int argc, char** argv) {
  if (argc != 3) return 2;
  const std::string mode = argv[1];
  const auto late = std::chrono::milliseconds(atoi(argv[2]));
  uint32_t flags[32] = {};
  std::atomic<bool> ended{false};
  std::thread device([&] {
    std::this_thread::sleep_for(late);
    if (mode != "dead")
      for (uint32_t& f : flags) __atomic_store_n(&f, 7u, __ATOMIC_RELEASE);
    ended.store(true);
  });
  const double c0 = cpu_ms();
  bool ok = true;
  auto wait = [&] { return svo::wait_flags(flags, 32, 7, [&] { return !ended.load(); }); };
  if (mode == "read") {
    constexpr size_t PIECE = 4096, SLOTS = 16;
    std::vector<char> dst(20 * PIECE), ring(SLOTS * PIECE, 1);
    ok = svo::empty_ring(
             dst.data(), dst.size(), ring.data(), PIECE, SLOTS, 3,
             [](size_t, size_t, size_t) { return 0; }, [&](size_t) { return wait() ? 0 : -4; },
             [](auto& work) { return std::thread(work); }) == 0;
  } else {
    ok = wait();
  }
  const double c1 = cpu_ms();
  device.join();
  printf("%d %.3f\n", ok ? 1 : 0, c1 - c0);
  return 0;
}

// The memory manager's worker threads on the host, with hip_stub.cpp
// standing in for the device: TryParallelFor never waits for another job,
// and a job that throws leaves the workers usable.  Built with
// AddressSanitizer by tests/test_transfer_host.py.  TEST INFRASTRUCTURE ONLY.
#include <stdio.h>
#include <stdlib.h>

#include <atomic>
#include <chrono>
#include <stdexcept>
#include <thread>

#include "../../imagevis3d_amd/csrc/memman.hpp"

using tvk::MemMan;

#define CHECK(c)                                                            \
  do {                                                                      \
    if (!(c)) {                                                             \
      fprintf(stderr, "%s:%d: check failed: %s\n", __FILE__, __LINE__, #c); \
      exit(1);                                                              \
    }                                                                       \
  } while (0)

static double now_ms() {
  return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

int main() {
  MemMan& mm = MemMan::ForDevice(0);
  {  // beside jobs of 300 ms, one after the other, a try returns at once
    std::atomic<bool> stop{false};
    std::thread jobs([&] {
      while (!stop)
        mm.ParallelFor(2, 2, [](size_t) { std::this_thread::sleep_for(std::chrono::milliseconds(300)); });
    });
    double longest = 0.0;
    for (const double t0 = now_ms(); now_ms() - t0 < 2500.0;) {
      const double t = now_ms();
      (void)mm.TryParallelFor(2, 2, [](size_t) {});
      longest = std::max(longest, now_ms() - t);
    }
    stop = true;
    jobs.join();
    printf("longest try %.1f ms\n", longest);
    CHECK(longest < 150.0);
    printf("OK try\n");
  }
  {  // from inside a job, on every thread of it
    std::atomic<int> ran{0}, refused{0};
    mm.ParallelFor(16, 4, [&](size_t) {
      if (!mm.TryParallelFor(2, 2, [&](size_t) { ++ran; })) ++refused;
    });
    CHECK(ran == 0 && refused == 16);
    printf("OK nested\n");
  }
  {  // a job that throws on the caller's thread: the next ones run
    const std::thread::id me = std::this_thread::get_id();
    for (int rep = 0; rep < 20; ++rep) {
      std::atomic<int> running{0};
      bool thrown = false;
      try {
        mm.ParallelFor(64, 4, [&](size_t) {
          ++running;
          std::this_thread::sleep_for(std::chrono::microseconds(200));
          --running;
          if (std::this_thread::get_id() == me) throw std::runtime_error("source");
        });
      } catch (const std::runtime_error&) {
        thrown = true;
      }
      CHECK(thrown && running == 0);  // no worker is inside the job any more
      std::atomic<int> hits{0};
      CHECK(mm.TryParallelFor(64, 4, [&](size_t) { ++hits; }) && hits == 64);
    }
    printf("OK throw\n");
  }
  printf("ALL OK\n");
  return 0;
}

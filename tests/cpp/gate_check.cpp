// Admission of resident launches (resident_gate.h) on a device of 256 units.
// Prints nothing and returns 0 when every pair is admitted together exactly
// where it should be.
#include <atomic>
#include <chrono>
#include <cstdio>
#include <thread>

#include "resident_gate.h"
using namespace femgpu;

// A launch of `groups` workgroups of which a unit holds `per`.
static ResFit fit(int groups, int per) {
  return {double(groups) / (256.0 * per), 1.0 / per, groups};
}

// Whether b is admitted beside a (each pair on a device of its own).
static bool together(ResFit a, ResFit b) {
  static int device = 0;
  const int d = device++;
  std::atomic<bool> in{false};
  std::thread t;
  bool both;
  {
    ResidentGate first(d, 256, a);
    t = std::thread([&] {
      ResidentGate second(d, 256, b);
      in = true;
    });
    for (int i = 0; i < 100 && !in; ++i) std::this_thread::sleep_for(std::chrono::milliseconds(2));
    both = in;
  }
  t.join();  // (at the latest now it is admitted)
  return both;
}

int main() {
  const struct { ResFit a, b; bool both; const char *what; } cases[] = {
      {fit(10, 1), fit(10, 1), true, "two small launches of whole units"},
      {fit(128, 1), fit(128, 1), true, "whole units, the device exactly"},
      {fit(128, 1), fit(136, 1), false, "whole units, more than the device"},
      {fit(200, 1), fit(200, 1), false, "whole units, much more"},
      {fit(200, 2), fit(48, 2), true, "half units, by shares"},
      {fit(200, 2), fit(56, 1), true, "mixed, by units"},
      {fit(256, 2), fit(8, 1), false, "no unit without a workgroup left for a whole one"},
      {fit(256, 2), fit(256, 2), false, "no room for the next half"},
      {fit(512, 2), fit(8, 2), false, "a full device"},
      {fit(256, 4), fit(256, 4), true, "quarters, by shares"},
  };
  int bad = 0;
  for (const auto &c : cases)
    for (int swap = 0; swap < 2; ++swap)
      if (together(swap ? c.b : c.a, swap ? c.a : c.b) != c.both) {
        std::printf("FAIL %s (%d): expected %d\n", c.what, swap, c.both);
        ++bad;
      }
  // A launch of the whole device comes to its turn while two threads keep small
  // launches coming, at least one of them running at any time.
  {
    const int d = 1000;
    std::atomic<bool> stop{false}, in{false};
    std::atomic<int> running{0};
    auto small = [&] {
      while (!stop) {
        ResidentGate g(d, 256, fit(10, 1));
        ++running;
        const auto t0 = std::chrono::steady_clock::now();
        // (until the other one runs too, or 50 ms)
        while (running < 2 && !stop && std::chrono::steady_clock::now() - t0 < std::chrono::milliseconds(50))
          std::this_thread::yield();
        std::this_thread::sleep_for(std::chrono::milliseconds(1));
        --running;
      }
    };
    std::thread a(small), b(small);
    std::this_thread::sleep_for(std::chrono::milliseconds(20));
    std::thread big([&] {
      ResidentGate g(d, 256, fit(256, 1));
      in = true;
    });
    for (int i = 0; i < 1000 && !in; ++i) std::this_thread::sleep_for(std::chrono::milliseconds(2));
    if (!in) {
      std::printf("FAIL a large launch is kept out\n");
      ++bad;
    }
    stop = true;
    a.join();
    b.join();
    big.join();
  }
  return bad != 0;
}

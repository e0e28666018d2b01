// resident_gate.h -- admission of resident launches to a device.
#pragma once

#include <algorithm>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <map>
#include <mutex>

namespace femgpu {

// A context's use of the forms that stay on the chip (femgpu_set_resident).
struct ResidentUse {
  int mode = 0;                 // FEMGPU_RESIDENT_*
  bool off = false;             // a launch did not complete: launches from then on
  int64_t completed = 0, given_up = 0;
  int64_t lose_from = -1;       // tests: launches from this one on lack a workgroup
  bool late = false;            // tests: one gives up at its end
  bool on() const { return mode != 1 && !off; }
  bool short_waits = false;     // tests: waits run out after 2 ms, nothing is lost
  bool impatient() const { return short_waits || lose_from >= 0; }
  bool lose() const { return lose_from >= 0 && completed >= lose_from; }
};

// The bound of a wait in such tests, 2 ms, as the word that the kernels read.
constexpr uint64_t TEST_WAIT_TICKS = 200000;
inline double test_wait() {
  double v;
  static_assert(sizeof v == sizeof TEST_WAIT_TICKS, "");
  std::memcpy(&v, &TEST_WAIT_TICKS, sizeof v);
  return v;
}

// Resident launches (resident.h) wait for each other's workgroups, so all
// workgroups of a launch must reach the device: alone they do when they fit
// it; beside others they do while the launches' shares and the largest
// workgroup together stay within it (then some compute unit always has room
// for the next workgroup).  A launch that would not fit waits here for the
// others to end.
class ResidentGate {
 public:
  ResidentGate(int device, double share, double block) : g_(gate(device)), share_(share) {
    std::unique_lock<std::mutex> lock(g_.mu);
    g_.cv.wait(lock, [&] {
      return g_.n == 0 || g_.load + share + std::max(g_.block, block) <= 1.0;
    });
    ++g_.n;
    g_.load += share;
    g_.block = std::max(g_.block, block);
  }
  ~ResidentGate() {
    {
      std::lock_guard<std::mutex> lock(g_.mu);
      g_.load -= share_;
      if (--g_.n == 0) g_.load = g_.block = 0.0;
    }
    g_.cv.notify_all();
  }

 private:
  struct Gate {
    std::mutex mu;
    std::condition_variable cv;
    int n = 0;
    double load = 0.0, block = 0.0;
  };
  static Gate &gate(int device) {
    static std::mutex mu;
    static std::map<int, Gate> gates;
    std::lock_guard<std::mutex> lock(mu);
    return gates[device];
  }
  Gate &g_;
  double share_;
};

}  // namespace femgpu

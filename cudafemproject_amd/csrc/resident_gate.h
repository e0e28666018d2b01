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
  int64_t completed = 0, given_up = 0;
  int skip = 0, back_off = 0;   // calls left in the launch form; their number last time
  int64_t lose_from = -1;       // tests: launches from this one on lack a workgroup
  bool late = false;            // tests: one gives up at its end
  // Whether a call should try the resident form (asked once per call).  A launch
  // that did not complete cost a wait of a second, most likely for another
  // process's workgroups: the next 64 calls go without, twice as many after
  // another in a row, at most 4096.
  bool on() {
    if (mode == 1) return false;
    if (skip == 0) return true;
    --skip;
    return false;
  }
  void ended(bool complete) {
    ++(complete ? completed : given_up);
    back_off = complete ? 0 : std::min(std::max(64, 2 * back_off), 4096);
    if (!complete) skip = back_off;
  }
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

// The part of the device that a resident launch takes, of one compute unit that
// a workgroup takes, and its workgroups.
struct ResFit {
  double share = 0.0, block = 0.0;
  int groups = 0;
};

// Resident launches (resident.h) wait for each other's workgroups, so all
// workgroups of a launch must reach the device: alone they do when they fit
// it; beside others they do while some compute unit always has room for the next
// workgroup.  It has while the launches' shares and the largest workgroup
// together stay within the device, and also while the launches have no more
// workgroups than the device has units (wherever they are, a unit without any is
// left for the next): where a unit holds one workgroup, only the second lets
// two small launches run together.  A launch that would not fit waits here for
// the others to end, and those that come after it wait behind it (a stream of
// small ones would keep a large one out for good).
class ResidentGate {
 public:
  ResidentGate(int device, int units, const ResFit &fit) : g_(gate(device)), fit_(fit) {
    std::unique_lock<std::mutex> lock(g_.mu);
    const uint64_t turn = g_.last++;
    g_.cv.wait(lock, [&] {
      return turn == g_.next &&
             (g_.n == 0 || g_.load + fit.share + std::max(g_.block, fit.block) <= 1.0 ||
              g_.groups + fit.groups <= units);
    });
    ++g_.next;
    ++g_.n;
    g_.load += fit.share;
    g_.groups += fit.groups;
    g_.block = std::max(g_.block, fit.block);
    lock.unlock();
    g_.cv.notify_all();  // (the next in turn may fit too)
  }
  ~ResidentGate() {
    {
      std::lock_guard<std::mutex> lock(g_.mu);
      g_.load -= fit_.share;
      g_.groups -= fit_.groups;
      if (--g_.n == 0) g_.load = g_.block = 0.0;
    }
    g_.cv.notify_all();
  }

 private:
  struct Gate {
    std::mutex mu;
    std::condition_variable cv;
    uint64_t last = 0, next = 0;  // turns given out and taken
    int n = 0, groups = 0;
    double load = 0.0, block = 0.0;
  };
  static Gate &gate(int device) {
    static std::mutex mu;
    static std::map<int, Gate> gates;
    std::lock_guard<std::mutex> lock(mu);
    return gates[device];
  }
  Gate &g_;
  const ResFit fit_;
};

}  // namespace femgpu

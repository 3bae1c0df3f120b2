// resident_gate.hpp -- the host's side of launches whose blocks all stay on the
// device and wait for each other.
#pragma once
#include <map>
#include <mutex>

namespace dmsc {

// One such grid at a time per device: a second one beside it could hold the
// compute units the first still waits for.  (Kernels that end by themselves
// only delay it.)  Held from the launch until the host has seen its end.
class ResidentGrid {
 public:
  explicit ResidentGrid(int device) : device_(device) {
    std::lock_guard<std::mutex> lk(lock());
    int& n = taken()[device_];
    held_ = n == 0;
    n = 1;
  }
  ~ResidentGrid() {
    if (!held_) return;
    std::lock_guard<std::mutex> lk(lock());
    taken()[device_] = 0;
  }
  ResidentGrid(const ResidentGrid&) = delete;
  ResidentGrid& operator=(const ResidentGrid&) = delete;
  bool held() const { return held_; }

 private:
  static std::mutex& lock() {
    static std::mutex m;
    return m;
  }
  static std::map<int, int>& taken() {
    static std::map<int, int> t;
    return t;
  }
  int device_;
  bool held_ = false;
};

// After a launch has given up (another process holds compute units it waits
// for) a context's next solves do without: one, then two, four, ... up to 64
// between two attempts, until a launch runs to its end again.  So a device that
// stays shared costs few waits, each as long as the poll bound lets it be.  A
// larger bound than the one that ran out is tried at once.
class ResidentBackoff {
 public:
  // Whether a solve that could take the launch should.
  bool due(int polls) {
    if (skip_ == 0 || polls > polls_) return true;
    skip_--;
    return false;
  }
  void stalled(int polls) {
    polls_ = polls;
    wait_ = wait_ == 0 ? 1 : wait_ < kMost ? 2 * wait_ : kMost;
    skip_ = wait_;
  }
  void completed() { wait_ = skip_ = 0; }

 private:
  static constexpr int kMost = 64;
  int polls_ = 0, wait_ = 0, skip_ = 0;
};

}  // namespace dmsc

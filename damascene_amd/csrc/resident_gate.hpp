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

}  // namespace dmsc

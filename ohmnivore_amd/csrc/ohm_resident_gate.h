// ohm_resident_gate.h — which resident solves (ohm_persist.hip) run side by
// side on a device, and when none is tried. Host code only.
#pragma once

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdint>
#include <mutex>

namespace ohm {

// The workgroups of a resident solve wait for each other, so those of all
// solves under way on a device must be on it at once: two threads' solves that
// each held the compute units the other waits for would both time out. A solve
// takes places, one per workgroup, before its launch and gives them back when
// it has been waited for; solves that fit together run together, the others
// take their turn in the order they asked. Places come in eights, because the
// device deals a launch's workgroups out to its eight dies in turn: a die holds
// every solve's share if the shares, rounded up, fit.
//
// Where another process holds compute units, a solve gives up after its time
// limit (0.2 s) and goes on in the pipeline. The next ones would do the same,
// so after a give-up none is tried for a second, after further ones for two,
// four, up to 32; one that finishes opens the gate again.
class ResidentGate {
 public:
  static int places(int workgroups, int capacity) {
    return std::min((workgroups + 7) / 8 * 8, capacity);
  }
  void enter(int places, int capacity) {
    std::unique_lock<std::mutex> lock(mu_);
    const int64_t ticket = next_++;
    cv_.wait(lock, [&] { return serving_ == ticket && taken_ + places <= capacity; });
    serving_++;
    taken_ += places;
    cv_.notify_all();  // the next in line may fit too
  }
  void leave(int places) {
    std::lock_guard<std::mutex> lock(mu_);
    taken_ -= places;
    cv_.notify_all();
  }
  bool open(int64_t now_ms = clock_ms()) const {
    return now_ms >= closed_until_.load(std::memory_order_relaxed);
  }
  // How a solve ended: given up at its time limit, or not.
  void report(bool gave_up, int64_t now_ms = clock_ms()) {
    std::lock_guard<std::mutex> lock(mu_);
    pause_ms_ = gave_up ? std::min<int64_t>(std::max<int64_t>(2 * pause_ms_, 1000), 32'000) : 0;
    closed_until_.store(gave_up ? now_ms + pause_ms_ : 0, std::memory_order_relaxed);
  }
  static int64_t clock_ms() {
    return std::chrono::duration_cast<std::chrono::milliseconds>(
               std::chrono::steady_clock::now().time_since_epoch())
        .count();
  }

 private:
  std::mutex mu_;
  std::condition_variable cv_;
  int64_t next_ = 0, serving_ = 0;  // tickets given out, and the one whose turn it is
  int taken_ = 0;
  int64_t pause_ms_ = 0;
  std::atomic<int64_t> closed_until_{0};
};

// The gate of a device.
inline ResidentGate &resident_gate(int device) {
  static ResidentGate gates[64];
  return gates[(unsigned)device % 64];
}

// A solve's places from its launch until it has been waited for.
class ResidentPass {
 public:
  ResidentPass(int device, int workgroups, int capacity)
      : gate_(resident_gate(device)), places_(ResidentGate::places(workgroups, capacity)) {
    gate_.enter(places_, capacity);
  }
  ~ResidentPass() { gate_.leave(places_); }
  ResidentPass(const ResidentPass &) = delete;
  ResidentPass &operator=(const ResidentPass &) = delete;

 private:
  ResidentGate &gate_;
  const int places_;
};

}  // namespace ohm

// hc_stage.h -- pinned host slots that read-backs stage through, shared by the
// contexts of a device.
//
// A read-back borrows slots and returns them; none belongs to a context.  Pinning two
// slots cost each context's first read-back 0.1 to 0.2 ms (a 24^3 box: fluid 0.13 ms
// without slots, 0.21 with its own), more than such a case's step, and a request loop
// opens a context per case.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>

namespace hcg {

struct StageSlot {
  void* p = nullptr;
  size_t cap = 0;
  hipEvent_t ev = nullptr;
};

// The free slots of one device: at most kMost of kMostBytes in all while contexts are
// open, two after the last one is closed (a program that opens one after the other).
class StagePool {
 public:
  // never destroyed: a context may be closed while the process ends
  static StagePool& of(int device) {
    static StagePool* const pools = new StagePool[kDevices];
    return pools[device % kDevices];
  }

  void open() {
    std::lock_guard<std::mutex> hold(mutex_);
    ++users_;
  }
  void close() {
    std::lock_guard<std::mutex> hold(mutex_);
    if (--users_ > 0) return;
    while (n_ > 2) drop_smallest();
  }

  // A slot of at least `bytes`, a new one if none is free; the device is current.
  bool take(size_t bytes, StageSlot& s) {
    {
      std::lock_guard<std::mutex> hold(mutex_);
      int best = -1;
      for (int k = 0; k < n_; ++k)
        if (free_[k].cap >= bytes && (best < 0 || free_[k].cap < free_[best].cap)) best = k;
      if (best >= 0) {
        s = remove(best);
        return true;
      }
    }
    s = StageSlot{};
    size_t cap = 65536;
    while (cap < bytes) cap *= 2;
    if (hipHostMalloc(&s.p, cap, hipHostMallocDefault) == hipSuccess) {
      s.cap = cap;
      if (hipEventCreateWithFlags(&s.ev, hipEventDisableTiming) == hipSuccess) return true;
      s.ev = nullptr;
    } else {
      s.p = nullptr;
    }
    (void)hipGetLastError();
    release(s);
    return false;
  }

  // back; nothing on the device writes to it any more
  void give(const StageSlot& s) {
    std::lock_guard<std::mutex> hold(mutex_);
    if (n_ == kMost) drop_smallest();
    free_[n_++] = s;
    bytes_ += s.cap;
    while (bytes_ > kMostBytes) drop_smallest();
  }

 private:
  static constexpr int kDevices = 64, kMost = 32;
  static constexpr size_t kMostBytes = size_t(8) << 20;

  static void release(const StageSlot& s) {
    if (s.ev) (void)hipEventDestroy(s.ev);
    if (s.p) (void)hipHostFree(s.p);
  }
  StageSlot remove(int k) {
    const StageSlot s = free_[k];
    free_[k] = free_[--n_];
    bytes_ -= s.cap;
    return s;
  }
  void drop_smallest() {
    int least = 0;
    for (int k = 1; k < n_; ++k)
      if (free_[k].cap < free_[least].cap) least = k;
    release(remove(least));
  }

  std::mutex mutex_;
  StageSlot free_[kMost];
  int n_ = 0, users_ = 0;
  size_t bytes_ = 0;
};

}  // namespace hcg

// What has to be done once for every device of a process, such as raising a kernel's limit of dynamic LDS: a function's
// attributes belong to the device that is current when they are set, so a process that drives a second device sets them
// there as well.  Host code only.
#pragma once

#include <atomic>
#include <mutex>

namespace sjhip {

class OncePerDevice {
 public:
  // The result of make() (0: done) on `device`; later calls for that device return 0 without it.  A failure is not kept: the
  // next call tries again.  Threads may call it at the same time.
  template <typename Make> int operator()(int device, Make make) {
    if (device < 0 || device >= kDevices) return make();
    if (done_[device].load(std::memory_order_acquire)) return 0;
    std::lock_guard<std::mutex> lock(mutex_);
    if (done_[device].load(std::memory_order_relaxed)) return 0;
    const int rc = make();
    if (rc == 0) done_[device].store(true, std::memory_order_release);
    return rc;
  }

 private:
  static constexpr int kDevices = 64;  // (beyond them make() runs on every call)
  std::atomic<bool> done_[kDevices] = {};
  std::mutex mutex_;
};

}  // namespace sjhip

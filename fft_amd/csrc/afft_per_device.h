// afft_per_device.h -- host code: something to be done once on each GPU of the
// process, whichever thread comes first.
#pragma once

#include <atomic>

namespace afgpu {

// once(dev, f): f() unless it has already succeeded (returned 0) for that
// device.  Threads that arrive together may each call f, which therefore has to
// be harmless when repeated; a failure is returned and tried again next time.
class PerDevice {
 public:
  template <typename F>
  auto once(int dev, F&& f) -> decltype(f()) {
    const unsigned long long bit = dev >= 0 && dev < 64 ? 1ull << dev : 0;
    if (done_.load(std::memory_order_acquire) & bit) return decltype(f())(0);
    const auto e = f();
    if (e == decltype(f())(0)) done_.fetch_or(bit, std::memory_order_release);
    return e;
  }

 private:
  std::atomic<unsigned long long> done_{0};
};

}  // namespace afgpu

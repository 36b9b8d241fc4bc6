// A set-up step that every device needs once (a kernel's LDS limit belongs to
// the device that is current when it is set). Host code without HIP.
#pragma once

#include <atomic>
#include <cstdint>

namespace la {

struct OncePerDevice {
  std::atomic<uint64_t> done{0};  // a bit per device; devices past 63 take the step every time

  // f() unless it has succeeded (returned 0) for this device. Threads that meet may both take it.
  template <typename F>
  auto run(int dev, F f) -> decltype(f()) {
    const uint64_t bit = dev >= 0 && dev < 64 ? 1ull << dev : 0;
    if (done.load(std::memory_order_acquire) & bit) return decltype(f()){};
    const auto e = f();
    if (e == decltype(f()){}) done.fetch_or(bit, std::memory_order_release);
    return e;
  }
};

}  // namespace la

// Host side: what a launch has to know about or set on the device that is current.
#pragma once
#include <hip/hip_runtime.h>
#include <atomic>

namespace kgc {

// An action that each device needs once (a kernel's attributes there): tried until it has succeeded on
// the device, from then on only looked up.
class OncePerDevice {
  static constexpr int N = 64;
  std::atomic<bool> done_[N] = {};

 public:
  template <typename F> bool operator()(int device, F&& act) {
    if (device < 0 || device >= N) return act();
    if (done_[device].load(std::memory_order_acquire)) return true;
    if (!act()) return false;
    done_[device].store(true, std::memory_order_release);
    return true;
  }
};

// A number that each device has.
class NumberPerDevice {
  static constexpr int N = 64;
  std::atomic<int> n_[N] = {};

 public:
  template <typename F> int operator()(int device, F&& ask) {
    if (device < 0 || device >= N) return ask();
    int n = n_[device].load(std::memory_order_relaxed);
    if (n == 0) n_[device].store(n = ask(), std::memory_order_relaxed);
    return n;
  }
};

inline int current_device() {
  int dev = -1;
  return hipGetDevice(&dev) == hipSuccess ? dev : -1;
}

// compute units of the current device (fewer than 256 where a GPU is partitioned)
inline int device_cus() {
  static NumberPerDevice cus;
  const int dev = current_device();
  return cus(dev, [&] {
    int n = 0;
    return hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0 ? n : 256;
  });
}

// dynamic LDS beyond 64 KB on the current device; false: refused, the caller takes its other route
template <typename K> bool allow_lds(OncePerDevice& once, K* kernel, size_t bytes) {
  return once(current_device(), [&] {
    const bool ok = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) == hipSuccess;
    if (!ok) (void)hipGetLastError();        // not the next launch's error
    return ok;
  });
}

}  // namespace kgc

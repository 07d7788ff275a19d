// Something done once per GPU, from whatever thread comes first.
#ifndef NATIVE_HIP_DEVICE_ONCE_H
#define NATIVE_HIP_DEVICE_ONCE_H

#include <atomic>
#include <cstdint>

namespace nh {

// Executors live on several threads and may drive several GPUs, and what a launch has to set beforehand (a kernel's LDS
// limit) belongs to the kernel on one GPU.  Threads that come first together each do it: it must bear that.
class DeviceOnce {
  public:
    // prepare() unless it has succeeded for `device` before; its result, whose zero means success.
    template <typename F> auto run(int device, F &&prepare) -> decltype(prepare()) {
        const uint64_t bit = device >= 0 && device < 64 ? (uint64_t)1 << device : 0;
        decltype(prepare()) result{};
        if ((done_.load(std::memory_order_acquire) & bit) != 0) return result;
        result = prepare();
        if (result == decltype(result){}) done_.fetch_or(bit, std::memory_order_release);
        return result;
    }

  private:
    std::atomic<uint64_t> done_{0};
};

}  // namespace nh
#endif

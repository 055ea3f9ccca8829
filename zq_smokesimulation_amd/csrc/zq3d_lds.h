// zq3d_lds.h -- dynamic LDS above the 64 KiB that a kernel gets without asking.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>

namespace zq3d {

// Raises one kernel's limit (one static object per kernel).  The attribute belongs to the device, so it is
// asked for once on each device that launches the kernel, and again after a refusal.  No stream operation:
// launches under capture may go through here.
class LdsLimit {
public:
    hipError_t raise(const void* kernel, int bytes) {
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return e;
        const unsigned long long bit = dev >= 0 && dev < 64 ? 1ull << dev : 0ull;
        if (done_.load(std::memory_order_acquire) & bit) return hipSuccess;
        e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
        if (e == hipSuccess) done_.fetch_or(bit, std::memory_order_release);
        return e;
    }

private:
    std::atomic<unsigned long long> done_{0};  // bit d: device d has the limit
};

}  // namespace zq3d

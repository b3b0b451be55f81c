// Dynamic LDS beyond the 64 KiB that a launch may ask for by itself.
#pragma once

#include <hip/hip_runtime_api.h>

#include <atomic>
#include <cstdint>

// One per kernel, static at its launch: the devices on which it has been marked.
struct LdsGrant {
    std::atomic<uint64_t> devices{0};
};

// Lets `kernel` be launched with up to `bytes` of dynamic LDS on the current device: 0 or a HIP error.  The attribute belongs to
// a kernel as loaded on one device, so it is set once per kernel and device (always with the same bytes).  Any number of threads
// may ask; two first callers set it twice.
inline int allow_lds(LdsGrant &grant, const void *kernel, size_t bytes) {
    int device = -1;
    const hipError_t known = hipGetDevice(&device);
    if (known != hipSuccess) return (int)known;
    if (device < 0 || device >= 64) return (int)hipErrorInvalidDevice;
    const uint64_t bit = 1ull << device;
    if (grant.devices.load(std::memory_order_acquire) & bit) return 0;
    const hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    if (e != hipSuccess) return (int)e;
    grant.devices.fetch_or(bit, std::memory_order_release);
    return 0;
}

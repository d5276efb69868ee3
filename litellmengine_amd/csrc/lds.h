// Kernels with more than 64 KB of dynamic LDS.
#pragma once
#include <hip/hip_runtime_api.h>
#include <stdint.h>
#include <atomic>

// A kernel's right to `bytes` of LDS, which the runtime grants per device: asked for at the first launch on each (`granted`,
// one for every kernel, has a bit for each device; asking costs the host about as much as a launch).
inline hipError_t lle_grant_lds(const void* kernel, int bytes, std::atomic<uint64_t>& granted) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const uint64_t bit = dev >= 0 && dev < 64 ? (uint64_t)1 << dev : 0;
    if (granted.load(std::memory_order_acquire) & bit) return hipSuccess;
    e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess)
        granted.fetch_or(bit, std::memory_order_release);
    else
        (void)hipGetLastError();  // (told here, not by the next launch)
    return e;
}

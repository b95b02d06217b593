// The limit of dynamic shared memory that a kernel may be launched with: kept by the runtime for each kernel and device, raised on the first
// launch that needs it.
#pragma once
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <cstddef>

// Raises `kernel`'s limit to `bytes` on the current device; `raised`, a static word of the launch's own, has a bit for each device on which that
// has been done (beyond 64 devices: at each launch).  Several threads may find it undone at once: each then does it.
inline hipError_t qe_raise_shared_limit(const void* kernel, size_t bytes, std::atomic<unsigned long>& raised) {
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    const unsigned long bit = device < 64 ? 1ul << device : 0;
    if (raised.load(std::memory_order_acquire) & bit) return hipSuccess;
    e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    if (e == hipSuccess) raised.fetch_or(bit, std::memory_order_release);
    return e;
}

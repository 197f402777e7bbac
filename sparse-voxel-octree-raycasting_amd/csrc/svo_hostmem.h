// svo_hostmem.h -- which host memory a kernel may write to.
#pragma once
#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <cstdint>

// The device address of `bytes` of pinned host memory at p, or null when one
// pinned allocation does not hold all of them, or it belongs to another
// device, or p is not word-aligned.  Both ends pinned is not enough: pinned
// memory is mapped at its host address, so between the ends of two allocations
// may lie memory the device cannot reach.
inline uint32_t* svo_host_writable(int device, void* p, size_t bytes)
{
    hipPointerAttribute_t a;
    hipDeviceptr_t base = nullptr;
    size_t size = 0;
    if (((uintptr_t)p & 3u) == 0 && hipPointerGetAttributes(&a, p) == hipSuccess && a.type == hipMemoryTypeHost &&
        a.device == device && a.devicePointer &&
        hipMemGetAddressRange(&base, &size, (hipDeviceptr_t)a.devicePointer) == hipSuccess) {
        const uintptr_t d = (uintptr_t)a.devicePointer, b = (uintptr_t)base;
        if (d >= b && d - b <= size && bytes <= size - (d - b)) return (uint32_t*)a.devicePointer;
    }
    (void)hipGetLastError();
    return nullptr;
}

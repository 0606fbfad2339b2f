// Caller memory that a kernel may read or write in place of a copy.  A range counts only where it lies
// in one allocation: two arrays with unmapped pages between them can hold its first and its last byte, and
// what the copies refuse must not become an access of a kernel.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <cstdint>

namespace rl {

inline bool in_one_allocation(const void* p, size_t bytes) {
    hipDeviceptr_t base = nullptr;
    size_t size = 0;
    if (hipMemGetAddressRange(&base, &size, const_cast<void*>(p)) != hipSuccess) {
        (void)hipGetLastError();   // memory that HIP does not know
        return false;
    }
    const uintptr_t first = reinterpret_cast<uintptr_t>(base), at = reinterpret_cast<uintptr_t>(p);
    return at >= first && at - first <= size && bytes <= size - (at - first);
}

inline bool memory_kind(const void* p, hipPointerAttribute_t* a) {
    if (hipPointerGetAttributes(a, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return true;
}

// The device's address of a page-locked host range, or null (pageable, device or managed memory).
inline void* mapped_host(const void* p, size_t bytes) {
    hipPointerAttribute_t a{};
    if (p == nullptr || bytes == 0 || !memory_kind(p, &a) || a.type != hipMemoryTypeHost || !in_one_allocation(p, bytes)) {
        return nullptr;
    }
    return a.devicePointer;
}

// Whether the range is memory of the given GPU.
inline bool own_device(int device, const void* p, size_t bytes) {
    hipPointerAttribute_t a{};
    return memory_kind(p, &a) && a.type == hipMemoryTypeDevice && a.device == device && in_one_allocation(p, bytes);
}

}  // namespace rl

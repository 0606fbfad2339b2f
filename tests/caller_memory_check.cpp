// rl_caller_memory.h on the CPU, over a HIP that knows two page-locked and two device allocations with a gap
// between them, and a page-locked one whose device address differs.  Exit status 1 names the first wrong answer.
#include <cstdio>

#include "rl_caller_memory.h"

namespace {

struct Allocation {
    uintptr_t first;
    size_t size;
    hipMemoryType type;
    int device;
    intptr_t mapped;   // device address - address
};

constexpr Allocation kKnown[] = {
    { 0x10000, 0x1000, hipMemoryTypeHost, 0, 0 },        { 0x14000, 0x1000, hipMemoryTypeHost, 0, 0 },
    { 0x20000, 0x1000, hipMemoryTypeDevice, 0, 0 },      { 0x24000, 0x1000, hipMemoryTypeDevice, 0, 0 },
    { 0x30000, 0x1000, hipMemoryTypeDevice, 1, 0 },      { 0x40000, 0x1000, hipMemoryTypeHost, 0, 0x500000 },
    { 0x50000, 0x1000, hipMemoryTypeManaged, 0, 0 },
};

const Allocation* find(const void* p) {
    const uintptr_t at = reinterpret_cast<uintptr_t>(p);
    for (const Allocation& a : kKnown) {
        if (at >= a.first && at < a.first + a.size) {
            return &a;
        }
    }
    return nullptr;
}

const void* ptr(uintptr_t at) { return reinterpret_cast<const void*>(at); }

int failures = 0;

void expect(bool ok, const char* what) {
    if (!ok) {
        std::printf("wrong: %s\n", what);
        failures++;
    }
}

}  // namespace

extern "C" {

hipError_t hipPointerGetAttributes(hipPointerAttribute_t* attributes, const void* p) {
    const Allocation* a = find(p);
    if (a == nullptr) {
        attributes->type = hipMemoryTypeUnregistered;
        return hipSuccess;
    }
    attributes->type = a->type;
    attributes->device = a->device;
    attributes->devicePointer = reinterpret_cast<void*>(reinterpret_cast<uintptr_t>(p) + a->mapped);
    return hipSuccess;
}

hipError_t hipMemGetAddressRange(hipDeviceptr_t* base, size_t* size, hipDeviceptr_t p) {
    const Allocation* a = find(p);
    if (a == nullptr) {
        return hipErrorNotFound;
    }
    *base = reinterpret_cast<hipDeviceptr_t>(a->first);
    *size = a->size;
    return hipSuccess;
}

hipError_t hipGetLastError(void) { return hipSuccess; }

}  // extern "C"

int main() {
    using rl::mapped_host;
    using rl::own_device;
    expect(mapped_host(ptr(0x10000), 0x1000) == ptr(0x10000), "whole page-locked array");
    expect(mapped_host(ptr(0x10ff8), 8) == ptr(0x10ff8), "its end");
    expect(mapped_host(ptr(0x40010), 16) == ptr(0x540010), "its device address");
    expect(mapped_host(ptr(0x10ff8), 9) == nullptr, "one byte too many");
    expect(mapped_host(ptr(0x10800), 0x4000) == nullptr, "from one page-locked array into another");
    expect(mapped_host(ptr(0x20000), 8) == nullptr, "device memory");
    expect(mapped_host(ptr(0x50000), 8) == nullptr, "managed memory");
    expect(mapped_host(ptr(0x90000), 8) == nullptr, "pageable memory");
    expect(mapped_host(ptr(0x10000), 0) == nullptr, "no bytes");
    expect(mapped_host(nullptr, 8) == nullptr, "null");
    expect(own_device(0, ptr(0x20008), 0xff8), "device array");
    expect(!own_device(0, ptr(0x20008), 0xff9), "one byte too many of it");
    expect(!own_device(0, ptr(0x20800), 0x4000), "from one device array into another");
    expect(!own_device(0, ptr(0x30000), 8), "another GPU's memory");
    expect(!own_device(0, ptr(0x10000), 8), "page-locked memory as device memory");
    expect(!own_device(0, ptr(0x90000), 8), "pageable memory as device memory");
    return failures == 0 ? 0 : 1;
}

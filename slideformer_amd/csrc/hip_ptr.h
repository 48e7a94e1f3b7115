// slideformer_amd: what kind of memory an address is, as the HIP runtime knows it.
//
// hipPointerGetAttributes is a lookup in the runtime's allocation table (~0.06 us
// on MI355X).  Device, managed and unified memory may be read and written by
// kernels in place; page-locked host memory (hipHostMalloc, torch pin_memory)
// is what the copy engines move directly; pageable memory is unknown to the
// runtime (unregistered, or an error on a host without a device).
#ifndef SLIDEFORMER_AMD_HIP_PTR_H
#define SLIDEFORMER_AMD_HIP_PTR_H

#include <hip/hip_runtime.h>

#include <cstring>

namespace la_ptr {

// The runtime's memory type of `ptr`, or hipMemoryTypeUnregistered when it
// does not know the address (the query's own failure is cleared, so that it
// is not reported by a later call).
inline hipMemoryType memory_type(const void* ptr)
{
    hipPointerAttribute_t a;
    std::memset(&a, 0, sizeof(a));
    if (hipPointerGetAttributes(&a, ptr) != hipSuccess) {
        (void)hipGetLastError();
        return hipMemoryTypeUnregistered;
    }
    return a.type;
}

// Memory the kernels may touch: device, managed or unified.
inline bool device_accessible(const void* ptr)
{
    const hipMemoryType t = memory_type(ptr);
    return t == hipMemoryTypeDevice || t == hipMemoryTypeManaged || t == hipMemoryTypeUnified;
}

// Page-locked host memory, which the copy engines read and write directly.
inline bool page_locked(const void* ptr) { return memory_type(ptr) == hipMemoryTypeHost; }

// Whether kernels on `device` may read and write all of [ptr, ptr + bytes) in
// host memory, at the same address: one page-locked allocation of that device,
// mapped at its host address, and coherent (the kernels' accesses then bypass
// the L2: nothing stale is read, and results are in host memory once the launch
// is complete).  On this runtime plain, mapped and coherent allocations and
// registrations are; any other flag (portable, write-combined, non-coherent)
// can make the memory coarse-grained.
inline bool kernel_reaches_host(const void* ptr, uint64_t bytes, int device)
{
    hipPointerAttribute_t a;
    std::memset(&a, 0, sizeof(a));
    unsigned flags = 0;
    void* start = nullptr;
    size_t size = 0;
    const hipDeviceptr_t p = const_cast<void*>(ptr);
    if (hipPointerGetAttributes(&a, ptr) != hipSuccess || a.type != hipMemoryTypeHost ||
        hipHostGetFlags(&flags, p) != hipSuccess ||
        hipPointerGetAttribute(&start, HIP_POINTER_ATTRIBUTE_RANGE_START_ADDR, p) != hipSuccess ||
        hipPointerGetAttribute(&size, HIP_POINTER_ATTRIBUTE_RANGE_SIZE, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    const uint64_t offset = static_cast<uint64_t>(static_cast<const char*>(ptr) - static_cast<const char*>(start));
    return a.device == device && a.devicePointer == ptr && !(flags & ~(hipHostMallocMapped | hipHostMallocCoherent)) &&
           offset <= size && bytes <= size - offset;
}

}  // namespace la_ptr

#endif  // SLIDEFORMER_AMD_HIP_PTR_H

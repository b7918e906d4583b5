// alloc.h -- device and page-locked allocations that may fail.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

namespace srm {

// Allocations whose failure the caller handles.  The runtime keeps an error until it is
// read, so a failed allocation's would be taken for the next launch's: it is read here
inline hipError_t device_alloc(void **p, size_t bytes)
{
    const hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess) {
        *p = nullptr;
        (void)hipGetLastError();
    }
    return e;
}
inline hipError_t host_alloc(void **p, size_t bytes)
{
    const hipError_t e = hipHostMalloc(p, bytes, hipHostMallocDefault);
    if (e != hipSuccess) {
        *p = nullptr;
        (void)hipGetLastError();
    }
    return e;
}
// no device has as much: the failure that the testing hooks ask for
constexpr size_t NO_DEVICE_HAS = (size_t)1 << 60;
bool filter_alloc_fails();   // srm_debug_fail_filter_allocs

}  // namespace srm

// The HIP runtime's entry points as a host program sees them, without a device: memory is the host's, copies are made at
// once, launches are handed to a hook, copies can be made to fail, a stream and an event are of the device that was current
// when they were made. Linked into a program of its own, before libamdhip64.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>

namespace fake {
struct Config {
    dim3 grid, block;
    size_t lds;
};
inline std::mutex mu;
inline std::map<const void *, int> attribute;  // a kernel's dynamic LDS limit, as last set
inline std::function<void(const void *kernel, dim3 grid, dim3 block, size_t lds)> launched;
inline thread_local Config config;
inline thread_local int device = 0;
inline std::map<const void *, size_t> pinned;  // host memory of hipHostMalloc
inline int async_live = 0, copies = 0, fail_at = -1;
inline size_t largest_copy = 0;
struct Handle {
    int device;
};
} // namespace fake

extern "C" {
hipError_t hipFuncSetAttribute(const void *f, hipFuncAttribute attr, int value) {
    std::lock_guard<std::mutex> g(fake::mu);
    if (attr == hipFuncAttributeMaxDynamicSharedMemorySize) fake::attribute[f] = value;
    return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t) {
    fake::config = {grid, block, lds};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *s) {
    *grid = fake::config.grid;
    *block = fake::config.block;
    *lds = fake::config.lds;
    *s = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **, size_t lds, hipStream_t) {
    if (fake::launched) fake::launched(f, grid, block, lds);
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "a failed call"; }

hipError_t hipGetDevice(int *d) { return *d = fake::device, hipSuccess; }
hipError_t hipSetDevice(int d) { return fake::device = d, hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    *s = (hipStream_t) new fake::Handle{fake::device};
    return hipSuccess;
}
hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t *d) { return *d = ((fake::Handle *)s)->device, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { return delete (fake::Handle *)s, hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    *e = (hipEvent_t) new fake::Handle{fake::device};
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    return ((fake::Handle *)e)->device == ((fake::Handle *)s)->device ? hipSuccess : hipErrorInvalidHandle;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { return delete (fake::Handle *)e, hipSuccess; }

hipError_t hipMalloc(void **p, size_t n) { return *p = std::malloc(n), hipSuccess; }
hipError_t hipFree(void *p) { return std::free(p), hipSuccess; }
hipError_t hipMallocAsync(void **p, size_t n, hipStream_t) {
    fake::async_live++;
    return *p = std::malloc(n), hipSuccess;
}
hipError_t hipFreeAsync(void *p, hipStream_t) {
    fake::async_live--;
    return std::free(p), hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    *p = std::malloc(n);
    std::lock_guard<std::mutex> g(fake::mu);
    fake::pinned[*p] = n;
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    std::lock_guard<std::mutex> g(fake::mu);
    fake::pinned.erase(p);
    return std::free(p), hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
    std::lock_guard<std::mutex> g(fake::mu);
    std::memset((void *)a, 0, sizeof *a);
    a->type = hipMemoryTypeUnregistered;
    for (auto &m : fake::pinned)
        if (p >= m.first && p < (const char *)m.first + m.second) a->type = hipMemoryTypeHost;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    {
        std::lock_guard<std::mutex> g(fake::mu);
        if (fake::copies++ == fake::fail_at) return hipErrorUnknown;
        if (n > fake::largest_copy) fake::largest_copy = n;
    }
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemset(void *d, int v, size_t n) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { return std::memset(d, v, n), hipSuccess; }

// (the device code is not there to be registered)
void **__hipRegisterFatBinary(const void *) { return nullptr; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, dim3 *, dim3 *, int *) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
}

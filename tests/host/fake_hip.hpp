// The HIP runtime's entry points as a host program sees them, without a device: memory is the host's, copies are made at
// once, launches are handed to a hook, any call can be made to fail. Link it into a program of its own, before libamdhip64.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>

namespace fake {
inline std::mutex mu;
inline std::map<const void *, int> attribute;  // a kernel's dynamic LDS limit, as last set
inline std::function<void(const void *kernel, dim3 grid, dim3 block, size_t lds)> launched;
struct Config {
    dim3 grid, block;
    size_t lds;
};
inline thread_local Config config;
} // namespace fake

extern "C" hipError_t hipFuncSetAttribute(const void *f, hipFuncAttribute attr, int value) {
    std::lock_guard<std::mutex> g(fake::mu);
    if (attr == hipFuncAttributeMaxDynamicSharedMemorySize) fake::attribute[f] = value;
    return hipSuccess;
}
extern "C" hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t) {
    fake::config = {grid, block, lds};
    return hipSuccess;
}
extern "C" hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *s) {
    *grid = fake::config.grid;
    *block = fake::config.block;
    *lds = fake::config.lds;
    *s = nullptr;
    return hipSuccess;
}
extern "C" hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **, size_t lds, hipStream_t) {
    if (fake::launched) fake::launched(f, grid, block, lds);
    return hipSuccess;
}
extern "C" hipError_t hipGetLastError() { return hipSuccess; }
// (the device code is not there to be registered)
extern "C" void **__hipRegisterFatBinary(const void *) { return nullptr; }
extern "C" void __hipUnregisterFatBinary(void **) {}
extern "C" void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, dim3 *, dim3 *,
                                      int *) {}
extern "C" void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}

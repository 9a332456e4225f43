// A HIP runtime without a device, for tests of the library's host code: device
// memory is host memory (filled with a pattern), kernels do not run, and any
// allocation or call can be made to fail.  An executable that includes it and
// is linked with -rdynamic takes these functions in place of the runtime's.
#pragma once
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace fake {
inline int fail_alloc = -1;          // allocations until one fails (-1: none does)
inline bool failed = false;          // that allocation was asked for
inline int allocations = 0;          // device and pinned, so far
inline bool sticky = false;          // a failed call is what hipGetLastError reports next
inline hipError_t last = hipSuccess;
inline int device = -1;              // of the last hipSetDevice
inline std::map<const void*, std::string>& names() {   // kernels by the address of their host stub
    static std::map<const void*, std::string> n;
    return n;
}
// called for every launch: kernel's name and arguments, as hipLaunchKernel has them
inline hipError_t (*on_launch)(const std::string&, void**) = nullptr;

inline hipError_t alloc(void** p, size_t n) {
    if (fail_alloc >= 0 && fail_alloc-- == 0) {
        failed = true;
        if (sticky) last = hipErrorOutOfMemory;
        return hipErrorOutOfMemory;
    }
    ++allocations;
    *p = std::malloc(n + 64);
    std::memset(*p, 0xab, n + 64);
    return hipSuccess;
}
}  // namespace fake

extern "C" {
void** __hipRegisterFatBinary(const void*) {
    static void* h = nullptr;
    return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    fake::names()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* t) {
    *g = *b = dim3{1, 1, 1};
    *s = 0;
    *t = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t) {
    const hipError_t e = fake::on_launch ? fake::on_launch(fake::names()[f], args) : hipSuccess;
    if (e != hipSuccess) fake::last = e;
    return e;
}
hipError_t hipMalloc(void** p, size_t n) { return fake::alloc(p, n); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return fake::alloc(p, n); }
hipError_t hipFree(void* p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) {
    *d = h;
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) {
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n) {
    *n = 2;
    return hipSuccess;
}
hipError_t hipSetDevice(int d) {
    fake::device = d;
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    std::memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 4;
    return hipSuccess;
}
hipError_t hipGetLastError(void) {
    const hipError_t e = fake::last;
    fake::last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "fake error"; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = nullptr;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
    *e = nullptr;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 0;
    return hipSuccess;
}
}

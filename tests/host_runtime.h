// host_runtime.h -- the HIP runtime's memory and stream calls on host memory,
// for tests of the library's host code without a GPU: an executable that
// includes this and links libcamr_hydro.so has the library call these.
// Kernels do not run.  fake::cap bounds the "device" memory, fake::fail_at
// makes the n-th hipMalloc from now on fail (1 = the next), fake::lose_freed the
// one after every hipFree (as if another program had taken what was freed).
#pragma once

#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>

namespace fake {
inline size_t cap = size_t(1) << 40, used = 0, peak = 0;
inline long fail_at = 0, mallocs = 0, launches = 0;
inline bool lose_freed = false;
inline std::map<void *, size_t> live;
inline hipError_t last = hipSuccess;
} // namespace fake

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
    ++fake::mallocs;
    if ((fake::fail_at > 0 && --fake::fail_at == 0) || fake::used + n > fake::cap) {
        *p = nullptr;
        return fake::last = hipErrorOutOfMemory;
    }
    *p = calloc(n ? n : 1, 1);
    fake::live[*p] = n;
    fake::used += n;
    if (fake::used > fake::peak) fake::peak = fake::used;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    auto it = fake::live.find(p);
    if (it == fake::live.end()) return p ? hipErrorInvalidValue : hipSuccess;
    fake::used -= it->second;
    fake::live.erase(it);
    free(p);
    if (fake::lose_freed) fake::fail_at = 1;
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *f, size_t *t) {
    *f = fake::cap - fake::used;
    *t = fake::cap;
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    *p = calloc(n ? n : 1, 1);
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n) {
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipGetLastError(void) {
    const hipError_t e = fake::last;
    fake::last = hipSuccess;
    return e;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    *s = (hipStream_t)malloc(1);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    free((void *)s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) {
    *e = (hipEvent_t)malloc(1);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
    free((void *)e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *m, hipStream_t *s) {
    *g = *b = dim3(1);
    *m = 0;
    *s = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) {
    ++fake::launches;
    return hipSuccess;
}
} // extern "C"

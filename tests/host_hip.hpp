// Stands in for the HIP runtime's memory, stream and event calls in host-only
// test programs that link libzkp.so: "device" memory is host memory, zeroed, with
// a limit; kernels do not run (an MSM's result is infinity). Include it first.
#pragma once
#include <hip/hip_runtime.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <mutex>

namespace host_hip {
inline size_t limit = (size_t)1 << 40, used = 0, allocations = 0, frees = 0;
inline std::map<void*, size_t> live;
inline std::mutex mu;
}  // namespace host_hip

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    std::lock_guard<std::mutex> lk(host_hip::mu);
    if (host_hip::used + n > host_hip::limit) return hipErrorOutOfMemory;
    *p = calloc(1, n);
    host_hip::live[*p] = n;
    host_hip::used += n;
    host_hip::allocations++;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    std::lock_guard<std::mutex> lk(host_hip::mu);
    auto it = host_hip::live.find(p);
    if (it == host_hip::live.end()) abort();
    host_hip::used -= it->second;
    host_hip::live.erase(it);
    host_hip::frees++;
    free(p);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
    std::lock_guard<std::mutex> lk(host_hip::mu);
    *f = host_hip::limit - host_hip::used;
    *t = host_hip::limit;
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return (*p = calloc(1, n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) {
    static char sym[1 << 20];
    *p = sym;
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)malloc(1); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { free((void*)s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)malloc(1); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { free((void*)e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0; return hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*) { return hipSuccess; }
}

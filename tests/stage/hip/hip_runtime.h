// The part of the HIP runtime that upf_stage.h calls, on host memory, for
// stage_check.cpp: copies happen at once, and allocations fail on request.
#ifndef STAGE_HIP_RUNTIME_H_
#define STAGE_HIP_RUNTIME_H_

#include <cstdlib>
#include <cstring>

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
typedef void* hipStream_t;
typedef int* hipEvent_t;
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;

inline bool no_pinned = false, no_events = false;
inline int pinned_copies = 0, plain_copies = 0;
inline char *pinned = nullptr, *pinned_end = nullptr;

inline hipError_t last_error = hipSuccess;

inline hipError_t hipGetLastError() { const hipError_t e = last_error; last_error = hipSuccess; return e; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    if (no_pinned) return last_error = hipErrorOutOfMemory;
    *p = pinned = static_cast<char*>(std::malloc(n));
    pinned_end = pinned + n;
    return hipSuccess;
}
inline hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    static int event;
    if (no_events) return last_error = hipErrorOutOfMemory;
    *e = &event;
    return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { return e ? hipSuccess : hipErrorOutOfMemory; }
inline hipError_t hipEventSynchronize(hipEvent_t e) { return e ? hipSuccess : hipErrorOutOfMemory; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) {
    const char* host = static_cast<const char*>(k == hipMemcpyHostToDevice ? s : d);
    __atomic_fetch_add(pinned && host >= pinned && host < pinned_end ? &pinned_copies : &plain_copies, 1, __ATOMIC_RELAXED);
    std::memcpy(d, s, n);
    return hipSuccess;
}

#endif

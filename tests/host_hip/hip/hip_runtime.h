// The part of the HIP runtime's interface that glac_amd/csrc/transfer.hpp calls, on host memory alone, for
// tests/transfer_check.cpp: copies are done at once and written down.
#pragma once
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <mutex>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
enum hipMemoryType {
    hipMemoryTypeUnregistered = 0,
    hipMemoryTypeHost = 1,
    hipMemoryTypeDevice = 2,
    hipMemoryTypeManaged = 3
};
struct hipPointerAttribute_t {
    hipMemoryType type;
};
using hipStream_t = void *;
using hipEvent_t = void *;
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;

struct Runtime {
    struct Copy {
        const char *dst, *src;
        size_t bytes;
    };
    static constexpr int kMost = 4096;
    std::mutex lock;
    Copy copies[kMost];
    int n = 0, syncs = 0;
    const char *slices = nullptr;  // what hipHostMalloc gave
    size_t slice_bytes = 0;
    const char *known[8];  // the first bytes of arrays that the runtime knows
    int n_known = 0;
    hipMemoryType known_type = hipMemoryTypeHost;
    bool no_pinned = false, unknown_is_error = false;
    hipError_t last = hipSuccess;
};
inline Runtime rt;

inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipGetLastError()
{
    const hipError_t e = rt.last;
    rt.last = hipSuccess;
    return e;
}
inline hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes, hipMemcpyKind, hipStream_t)
{
    std::memcpy(dst, src, bytes);
    std::lock_guard<std::mutex> hold(rt.lock);
    if (rt.n < Runtime::kMost) rt.copies[rt.n++] = {(const char *)dst, (const char *)src, bytes};
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t)
{
    rt.syncs++;
    return hipSuccess;
}
inline hipError_t hipHostMalloc(void **p, size_t bytes, unsigned)
{
    if (rt.no_pinned) return rt.last = hipErrorOutOfMemory;
    *p = std::malloc(bytes);
    rt.slices = (const char *)*p;
    rt.slice_bytes = bytes;
    return hipSuccess;
}
inline hipError_t hipHostFree(void *p)
{
    std::free(p);
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    *e = &rt;
    return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{
    for (int k = 0; k < rt.n_known; k++)
        if (p == rt.known[k]) {
            a->type = rt.known_type;
            return hipSuccess;
        }
    if (rt.unknown_is_error) return rt.last = hipErrorInvalidValue;
    a->type = hipMemoryTypeUnregistered;
    return hipSuccess;
}

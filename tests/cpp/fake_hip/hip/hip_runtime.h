// A stand-in for the HIP runtime that the library's host code sees when it is compiled for the
// CPU tests: device memory is addresses and sizes only. Allocations take the lowest free
// address, as long as `budget` bytes last, and carry a number of their own; streams can be
// put in error; every call is counted.
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <map>
#include <set>

#define __host__
#define __device__
#define __global__
#define __forceinline__ inline

enum hipError_t {
    hipSuccess = 0,
    hipErrorInvalidValue = 1,
    hipErrorOutOfMemory = 2,
    hipErrorInvalidDevice = 101,
    hipErrorIllegalAddress = 700
};
struct FakeStream {
    bool bad = false;
};
struct FakeEvent {};
typedef FakeStream* hipStream_t;
typedef FakeEvent* hipEvent_t;
typedef void* hipDeviceptr_t;
enum { hipStreamNonBlocking = 1, hipHostMallocDefault = 0 };
enum hipPointer_attribute { HIP_POINTER_ATTRIBUTE_BUFFER_ID = 7 };

namespace fake {
struct Allocation {
    size_t bytes;
    unsigned long long id;
};
inline std::map<uintptr_t, Allocation> device, pinned;   // by address
inline std::set<FakeStream*> streams;
inline std::set<FakeEvent*> events;
inline unsigned long long next_id = 1;
inline size_t budget = (size_t)1 << 40, pinned_budget = (size_t)1 << 40;
inline int mallocs = 0, frees = 0, bad_frees = 0;
inline size_t used(const std::map<uintptr_t, Allocation>& m)
{
    size_t n = 0;
    for (const auto& a : m) n += a.second.bytes;
    return n;
}
inline hipError_t take(std::map<uintptr_t, Allocation>& m, uintptr_t at, size_t limit, void** p, size_t bytes)
{
    if (used(m) + bytes > limit) return hipErrorOutOfMemory;
    for (const auto& a : m) {   // the lowest gap, at steps of 4 KB
        if (at + bytes <= a.first) break;
        at = (a.first + a.second.bytes + 4095) / 4096 * 4096;
    }
    m[at] = Allocation{bytes, next_id++};
    *p = (void*)at;
    return hipSuccess;
}
// hipDeviceReset: memory, streams and events are gone
inline void reset()
{
    device.clear();
    pinned.clear();
    streams.clear();
    events.clear();
}
}  // namespace fake

inline hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
inline hipError_t hipSetDevice(int d) { return d == 0 ? hipSuccess : hipErrorInvalidDevice; }
inline hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipMalloc(void** p, size_t bytes)
{
    ++fake::mallocs;
    return fake::take(fake::device, (uintptr_t)1 << 32, fake::budget, p, bytes);
}
inline hipError_t hipFree(void* p)
{
    ++fake::frees;
    if (fake::device.erase((uintptr_t)p)) return hipSuccess;
    ++fake::bad_frees;
    return hipErrorInvalidValue;
}
inline hipError_t hipHostMalloc(void** p, size_t bytes, unsigned)
{
    return fake::take(fake::pinned, (uintptr_t)1 << 50, fake::pinned_budget, p, bytes);
}
inline hipError_t hipHostFree(void* p)
{
    if (fake::pinned.erase((uintptr_t)p)) return hipSuccess;
    ++fake::bad_frees;
    return hipErrorInvalidValue;
}
inline hipError_t hipPointerGetAttribute(void* out, hipPointer_attribute, void* p)
{
    for (const auto* m : {&fake::device, &fake::pinned}) {
        const auto it = m->find((uintptr_t)p);
        if (it == m->end()) continue;
        *(unsigned long long*)out = it->second.id;
        return hipSuccess;
    }
    return hipErrorInvalidValue;
}
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
inline hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
inline hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned)
{
    fake::streams.insert(*s = new FakeStream());
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s)
{
    if (s && !fake::streams.count(s)) return hipErrorInvalidValue;
    return s && s->bad ? hipErrorIllegalAddress : hipSuccess;
}
inline hipError_t hipStreamDestroy(hipStream_t s)
{
    if (!fake::streams.erase(s)) {
        ++fake::bad_frees;
        return hipErrorInvalidValue;
    }
    delete s;
    return hipSuccess;
}
inline hipError_t hipEventCreate(hipEvent_t* e)
{
    fake::events.insert(*e = new FakeEvent());
    return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e)
{
    if (!fake::events.erase(e)) {
        ++fake::bad_frees;
        return hipErrorInvalidValue;
    }
    delete e;
    return hipSuccess;
}
// device intrinsics that the shared headers name; never called
inline int __builtin_amdgcn_update_dpp(int, int v, int, int, int, bool) { return v; }
inline int __builtin_amdgcn_readlane(int v, int) { return v; }

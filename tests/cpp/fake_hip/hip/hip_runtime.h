// A stand-in for the few HIP calls of lt_hostio.cpp, for host checks of its error paths: device memory is host memory with
// a limit, pinned memory can be refused, copies are done when their stream or event is waited for, and a copy
// can be made to fail.
#pragma once

#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

typedef int hipError_t;
constexpr hipError_t hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999;
struct ihipStream_t;
struct ihipEvent_t;
typedef ihipStream_t* hipStream_t;
typedef ihipEvent_t* hipEvent_t;
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
constexpr unsigned hipStreamNonBlocking = 1, hipEventDisableTiming = 2, hipHostMallocDefault = 0;

namespace fake {
struct Copy {
    void* dst;
    const void* src;
    size_t bytes;
};
struct State {
    std::mutex mu;
    size_t limit = ~(size_t)0, used = 0;
    bool no_pinned = false;
    int copies_until_failure = -1;  // < 0: none fails
    std::map<void*, size_t> device, pinned;
    std::map<hipStream_t, std::vector<Copy>> queued;
    std::map<hipEvent_t, hipStream_t> recorded;
};
inline State& state()
{
    static State s;
    return s;
}
inline size_t pending()
{
    std::lock_guard<std::mutex> lock(state().mu);
    size_t n = 0;
    for (auto& q : state().queued) n += q.second.size();
    return n;
}
inline void drain(hipStream_t s)
{
    for (const Copy& c : state().queued[s]) std::memcpy(c.dst, c.src, c.bytes);
    state().queued[s].clear();
}
}  // namespace fake

inline hipError_t hipMalloc(void** p, size_t n)
{
    std::lock_guard<std::mutex> lock(fake::state().mu);
    if (fake::state().used + n > fake::state().limit) return hipErrorOutOfMemory;
    *p = std::malloc(n ? n : 1);
    fake::state().device[*p] = n;
    fake::state().used += n;
    return hipSuccess;
}
inline hipError_t hipFree(void* p)
{
    std::lock_guard<std::mutex> lock(fake::state().mu);
    if (!p) return hipSuccess;
    auto it = fake::state().device.find(p);
    if (it == fake::state().device.end()) std::abort();
    fake::state().used -= it->second;
    fake::state().device.erase(it);
    std::free(p);
    return hipSuccess;
}
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    std::lock_guard<std::mutex> lock(fake::state().mu);
    if (fake::state().no_pinned) return hipErrorOutOfMemory;
    *p = std::malloc(n);
    fake::state().pinned[*p] = n;
    return hipSuccess;
}
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int* d)
{
    *d = 0;
    return hipSuccess;
}
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned)
{
    *s = (hipStream_t)std::malloc(1);
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
    *e = (hipEvent_t)std::malloc(1);
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t s)
{
    std::lock_guard<std::mutex> lock(fake::state().mu);
    if (fake::state().copies_until_failure >= 0 && fake::state().copies_until_failure-- == 0) return hipErrorUnknown;
    fake::state().queued[s].push_back({dst, src, n});
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    std::lock_guard<std::mutex> lock(fake::state().mu);
    fake::state().recorded[e] = s;
    return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e)
{
    std::lock_guard<std::mutex> lock(fake::state().mu);
    fake::drain(fake::state().recorded[e]);  // (what was queued after the record is done too: no harm to these checks)
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s)
{
    std::lock_guard<std::mutex> lock(fake::state().mu);
    fake::drain(s);
    return hipSuccess;
}

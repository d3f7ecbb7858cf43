// lt_hostio.cpp -- copies of the synchronous host-array calls.
//
// The caller's arrays are pageable, and often fresh: their pages are first touched by the copy. The runtime's own copy
// of 90 MB of such planes took 6.6 ms, 37 times the kernel before it. Here the device writes pieces into a pinned area
// and four threads move them on, page faults included, while the next pieces arrive (2.3 ms); up to one piece a single
// thread does the same without starting others. With one image of the inputs in pinned memory, one copy of the results
// and buffers that stay, a likelihood evaluation on 512 x 512 pixels takes 80-89 us (335 with its own allocations and
// nine copies), 20000 point gradients of 503 halos 145-148 (192). Where the area cannot be had the calls copy from and to
// pageable memory. What stays is bounded (64 MB of scratch, 16 MB pinned, the
// planes of the largest map call) and given back when an allocation would fail.
#include "lt_hostio.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>
#include <vector>

#include "lt_internal.h"

namespace lt {

static HostState g_host[kMaxDevices];

HostState& host_state(int dev) { return g_host[dev]; }

int host_ready(HostState& h)
{
    if (!h.stream) LT_HIP_TRY(hipStreamCreateWithFlags(&h.stream, hipStreamNonBlocking));
    if (!h.pinned && hipHostMalloc((void**)&h.pinned, kHostPinned, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        h.pinned = nullptr;
    }
    return LT_OK;
}

char* host_image(HostState& h, size_t bytes, std::vector<char>& own)
{
    if (h.pinned && bytes <= kHostPinned) return h.pinned;
    own.resize(bytes);
    return own.data();
}

static void give_back(HostState& h)
{
    if (h.stream) (void)hipStreamSynchronize(h.stream);
    for (void** p : {&h.halos, &h.planes, &h.scratch}) {
        if (*p) (void)hipFree(*p);
        *p = nullptr;
    }
    h.halos_bytes = h.planes_bytes = h.scratch_bytes = 0;
}

// a kept buffer of at least `need` bytes; what it held is lost
static hipError_t grow(void** buf, size_t* have, size_t need, size_t slack)
{
    if (need <= *have) return hipSuccess;
    hipError_t e = *buf ? hipFree(*buf) : hipSuccess;
    *buf = nullptr;
    *have = 0;
    if (e == hipSuccess) e = hipMalloc(buf, need + slack);
    if (e == hipSuccess) *have = need + slack;
    else *buf = nullptr;
    return e;
}

static int no_memory(size_t bytes)
{
    (void)hipGetLastError();
    return set_error(LT_ERR_NOMEM, "device allocation of " + std::to_string(bytes) + " bytes failed");
}

int host_room(HostState& h, size_t halos, size_t planes)
{
    for (int again = 0; again < 2; ++again) {
        if (again) give_back(h);
        if (grow(&h.halos, &h.halos_bytes, halos, again ? 0 : halos / 4) == hipSuccess &&
            grow(&h.planes, &h.planes_bytes, planes, again ? 0 : planes / 4) == hipSuccess)
            return LT_OK;
    }
    return no_memory(halos + planes);
}

hipError_t device_alloc(void** p, size_t bytes)
{
    hipError_t e = hipMalloc(p, bytes);
    int dev = 0;
    if (e == hipSuccess || hipGetDevice(&dev) != hipSuccess || dev >= kMaxDevices) return e;
    HostState& h = g_host[dev];
    std::unique_lock<std::mutex> lock(h.mu, std::try_to_lock);
    if (!lock) return e;
    (void)hipGetLastError();
    give_back(h);
    return hipMalloc(p, bytes);
}

int HostScratch::take(HostState& h, size_t bytes)
{
    own = bytes > kHostKept * 4 / 5;
    for (int again = 0; again < 2; ++again) {
        if (again) give_back(h);
        if (own ? hipMalloc((void**)&p, bytes) == hipSuccess
                : grow(&h.scratch, &h.scratch_bytes, bytes, again ? 0 : bytes / 4) == hipSuccess) {
            if (!own) p = (char*)h.scratch;
            return LT_OK;
        }
    }
    p = nullptr;
    own = false;
    return no_memory(bytes);
}

HostScratch::~HostScratch()
{
    if (own) (void)hipFree(p);
}

// One thread's share of a large copy: pieces in turn through its two parts of the pinned area, one arriving while
// the other is moved on.
static void copy_share(HostState& h, int dev, int w, const std::vector<HostCopy>& pieces, std::atomic<size_t>& next,
                       std::atomic<int>& error)
{
    hipError_t e = hipSetDevice(dev);
    if (e == hipSuccess && !h.copy_stream[w]) e = hipStreamCreateWithFlags(&h.copy_stream[w], hipStreamNonBlocking);
    for (int k = 0; k < 2; ++k)
        if (e == hipSuccess && !h.copied[w][k]) e = hipEventCreateWithFlags(&h.copied[w][k], hipEventDisableTiming);
    const HostCopy* pending[2] = {nullptr, nullptr};
    for (int k = 0; e == hipSuccess; k ^= 1) {
        char* const at = h.pinned + (size_t)(2 * w + k) * kHostPiece;
        const size_t i = error.load() ? pieces.size() : next.fetch_add(1);
        if (i < pieces.size()) {  // (the part's own last piece was moved on a turn ago)
            e = hipMemcpyAsync(at, pieces[i].dev, pieces[i].bytes, hipMemcpyDeviceToHost, h.copy_stream[w]);
            if (e == hipSuccess) e = hipEventRecord(h.copied[w][k], h.copy_stream[w]);
            if (e != hipSuccess) break;
            pending[k] = &pieces[i];
        }
        if (const HostCopy* c = pending[k ^ 1]) {
            e = hipEventSynchronize(h.copied[w][k ^ 1]);
            if (e == hipSuccess) std::memcpy(c->host, h.pinned + (size_t)(2 * w + (k ^ 1)) * kHostPiece, c->bytes);
            pending[k ^ 1] = nullptr;
        } else if (!pending[k]) {
            break;
        }
    }
    if (e != hipSuccess) {
        if (h.copy_stream[w]) (void)hipStreamSynchronize(h.copy_stream[w]);
        int none = 0;
        error.compare_exchange_strong(none, (int)e);
    }
}

// The copies queued on h.stream, all of them or up to the first that fails.
static hipError_t queue_small(HostState& h, const HostCopy* copies, int n)
{
    if (!h.pinned) {
        for (int i = 0; i < n; ++i)
            if (copies[i].bytes) {
                const hipError_t e = hipMemcpyAsync(copies[i].host, copies[i].dev, copies[i].bytes, hipMemcpyDeviceToHost, h.stream);
                if (e != hipSuccess) return e;
            }
        return hipSuccess;
    }
    // through the start of the pinned area, neighbours on the device in one copy
    size_t at = 0;
    for (int i = 0; i < n;) {
        size_t bytes = copies[i].bytes;
        int k = i + 1;
        for (; k < n && (const char*)copies[k].dev == (const char*)copies[i].dev + bytes; ++k) bytes += copies[k].bytes;
        if (bytes) {
            const hipError_t e = hipMemcpyAsync(h.pinned + at, copies[i].dev, bytes, hipMemcpyDeviceToHost, h.stream);
            if (e != hipSuccess) return e;
        }
        at += bytes;
        i = k;
    }
    return hipSuccess;
}

int host_download(HostState& h, const HostCopy* copies, int n)
{
    size_t total = 0;
    for (int i = 0; i < n; ++i) total += copies[i].bytes;
    if (!h.pinned || total <= kHostPiece) {
        const hipError_t e = queue_small(h, copies, n);
        // also after an error: the call's upload may still read the pinned area, the copies still write it
        const hipError_t es = hipStreamSynchronize(h.stream);
        if (e != hipSuccess || es != hipSuccess) return hip_error(e != hipSuccess ? e : es, "copy to the host");
        if (!h.pinned) return LT_OK;
        size_t at = 0;
        for (int i = 0; i < n; ++i) {
            if (copies[i].bytes) std::memcpy(copies[i].host, h.pinned + at, copies[i].bytes);
            at += copies[i].bytes;
        }
        return LT_OK;
    }
    // (the upload too is done before the pinned area is written, and before anything below may throw)
    LT_HIP_TRY(hipStreamSynchronize(h.stream));
    std::vector<HostCopy> pieces;
    for (int i = 0; i < n; ++i)
        for (size_t o = 0; o < copies[i].bytes; o += kHostPiece)
            pieces.push_back({(char*)copies[i].host + o, (const char*)copies[i].dev + o, std::min(kHostPiece, copies[i].bytes - o)});
    int dev = 0;
    LT_HIP_TRY(hipGetDevice(&dev));
    std::atomic<size_t> next{0};
    std::atomic<int> error{0};
    std::vector<std::thread> others;
    others.reserve(kHostThreads);
    try {
        for (int w = 1; w < std::min<int>(kHostThreads, (int)pieces.size()); ++w)
            others.emplace_back([&, w] { copy_share(h, dev, w, pieces, next, error); });
    } catch (...) {  // no more threads, or no memory for one: those there are take all
    }
    copy_share(h, dev, 0, pieces, next, error);
    for (std::thread& t : others) t.join();
    if (error.load()) return hip_error((hipError_t)error.load(), "copy to the host");
    return LT_OK;
}

}  // namespace lt

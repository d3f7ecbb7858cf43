// lt_hostio.h -- what the synchronous host-array calls keep per device between calls (a stream, device buffers, a
// pinned area) and their copies between the caller's arrays and the device.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>
#include <vector>

namespace lt {

constexpr size_t kHostPiece = 1 << 21;             // bytes of a piece of a copy
constexpr int kHostThreads = 4;                    // threads of a large copy to the host, two pieces of the pinned area each
constexpr size_t kHostPinned = 2 * kHostThreads * kHostPiece;
constexpr size_t kHostKept = 64 << 20;             // device bytes that a call's scratch may keep

// One per device; a call holds `mu` from its first use to its end.
struct HostState {
    std::mutex mu;
    hipStream_t stream = nullptr;
    char* pinned = nullptr;         // kHostPinned bytes, or NULL where they cannot be had
    void* halos = nullptr;          // grow-only buffers of the map calls
    size_t halos_bytes = 0;
    void* planes = nullptr;
    size_t planes_bytes = 0;
    void* scratch = nullptr;        // at most kHostKept bytes, see HostScratch
    size_t scratch_bytes = 0;
    hipStream_t copy_stream[kHostThreads] = {};
    hipEvent_t copied[kHostThreads][2] = {};
};

constexpr int kMaxDevices = 64;
HostState& host_state(int dev);
// the stream and the pinned area of the current device's state, made on the first call; without the area the calls
// copy from and to pageable memory
int host_ready(HostState& h);
// where a call forms the image of its inputs: the pinned area, or `own` where that is too small or missing
char* host_image(HostState& h, size_t bytes, std::vector<char>& own);
// the map calls' buffers, of at least these sizes; what they held is lost. Gives back everything kept rather than fail.
int host_room(HostState& h, size_t halos, size_t planes);

// hipMalloc that gives back the kept buffers of the device, if no call is using them, rather than fail.
hipError_t device_alloc(void** p, size_t bytes);

// Device memory of one call: the kept buffer, or an allocation of its own that goes with it.
struct HostScratch {
    char* p = nullptr;
    bool own = false;
    int take(HostState& h, size_t bytes);
    ~HostScratch();
};

// A copy device -> host. Small ones go through the start of the pinned area.
struct HostCopy {
    void* host;
    const void* dev;
    size_t bytes;
};

// All the copies device -> host, after the work queued on h.stream; returns when they are done.
int host_download(HostState& h, const HostCopy* copies, int n);

}  // namespace lt

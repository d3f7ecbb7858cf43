// hostio_check.cpp -- the kept buffers and copies of the host-array calls (lt_hostio.cpp) under conditions that a GPU box does
// not bring about at will, on the stand-in runtime of fake_hip: device memory that runs out.
#include <cstdio>
#include <string>
#include <vector>

#include "lt_hostio.h"
#include "lt_internal.h"

namespace lt {
static std::string g_error;
int set_error(int code, const std::string& msg)
{
    g_error = msg;
    return code;
}
int hip_error(hipError_t, const char* where) { return set_error(LT_ERR_HIP, where); }
}  // namespace lt

using namespace lt;

static int failures = 0;
static void expect(bool ok, const char* what)
{
    std::printf("%s: %s\n", ok ? "ok" : "FAILED", what);
    failures += !ok;
}

// Every buffer that is kept goes back before an allocation of a host call fails, whichever needs the memory.
static void check_room()
{
    HostState& h = host_state(0);
    const size_t mb = 1 << 20;
    expect(host_ready(h) == LT_OK, "stream and pinned area");
    fake::state().limit = 100 * mb;
    {
        HostScratch s;
        expect(s.take(h, 40 * mb) == LT_OK && !s.own, "40 MB of scratch are kept (50 with the slack)");
    }
    expect(host_room(h, mb, 60 * mb) == LT_OK && h.scratch_bytes == 0, "planes of 60 MB take the scratch's place");
    expect(h.planes_bytes >= 60 * mb && h.halos_bytes >= mb && h.halos && h.planes, "both of the map's buffers are there");
    {
        HostScratch s;
        expect(s.take(h, 45 * mb) == LT_OK && !s.own && h.planes_bytes == 0, "kept scratch takes the planes' place");
    }
    expect(host_room(h, mb, 98 * mb) == LT_OK, "planes without slack where they fit so");
    {
        HostScratch s;
        expect(s.take(h, 90 * mb) == LT_OK && s.own && h.planes_bytes == 0, "a call's own scratch takes their place");
    }
    expect(fake::state().used == 0, "its own scratch went with it");
    expect(host_room(h, mb, 70 * mb) == LT_OK, "planes again");
    void* p = nullptr;
    expect(device_alloc(&p, 80 * mb) == hipSuccess && h.planes_bytes == 0, "other allocations take their place too");
    expect(host_room(h, mb, 30 * mb) == LT_ERR_NOMEM && !h.planes && !h.planes_bytes, "what does not fit fails");
    (void)hipFree(p);
    expect(host_room(h, mb, 30 * mb) == LT_OK, "and fits later");
}

int main(int argc, char** argv)
{
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "room") check_room();
    else return 2;
    std::puts(failures ? "FAILED" : "OK");
    return failures != 0;
}

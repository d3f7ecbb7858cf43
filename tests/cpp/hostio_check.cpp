// hostio_check.cpp -- the kept buffers and copies of the host-array calls (lt_hostio.cpp) under conditions that a GPU box does
// not bring about at will, on the stand-in runtime of fake_hip: device memory that runs out, pinned memory that is refused, copies and
// allocations that fail under way.
#include <cstdio>
#include <cstdlib>
#include <new>
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

// the allocation of this thread that fails, counted from now (< 0: none)
static thread_local int g_fail_new = -1;

void* operator new(size_t n)
{
    if (g_fail_new >= 0 && g_fail_new-- == 0) throw std::bad_alloc();
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

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

// Planes on the device copied to host arrays as a map call does; true when they arrive whole.
static bool download(HostState& h, const std::vector<size_t>& sizes)
{
    std::vector<std::vector<char>> from, to;
    std::vector<HostCopy> copies;
    for (size_t n : sizes) {
        from.emplace_back(n);
        for (size_t i = 0; i < n; ++i) from.back()[i] = (char)(i * 31 + i / 4097 + sizes.size());
        to.emplace_back(n, (char)0x55);
    }
    for (size_t k = 0; k < sizes.size(); ++k) copies.push_back({to[k].data(), from[k].data(), sizes[k]});
    return host_download(h, copies.data(), (int)copies.size()) == LT_OK && from == to && fake::pending() == 0;
}

// Without the pinned area the calls go on.
static void check_pinned()
{
    HostState& h = host_state(0);
    fake::state().no_pinned = true;
    expect(host_ready(h) == LT_OK && !h.pinned, "no pinned area, and no error");
    std::vector<char> own;
    char* const image = host_image(h, 5000, own);
    expect(image && own.size() == 5000 && image == own.data(), "the image is the call's own");
    expect(download(h, {1000, 24, 3 * kHostPiece + 17}), "planes arrive without it");
    fake::state().no_pinned = false;
    expect(host_ready(h) == LT_OK && h.pinned, "it is asked for again by the next call");
    std::vector<char> none;
    expect(host_image(h, 5000, none) == h.pinned && none.empty(), "the image lies in it");
    expect(host_image(h, kHostPinned + 1, none) == none.data() && none.size() == kHostPinned + 1, "unless it is too large");
    expect(download(h, {1000, 24}) && download(h, {0, 3 * kHostPiece + 17, 9 * kHostPiece, 5}), "planes arrive through it");
}

// After a failure nothing is queued that would still read or write the pinned area or the caller's arrays.
static void check_errors()
{
    HostState& h = host_state(0);
    expect(host_ready(h) == LT_OK, "stream and pinned area");
    std::vector<char> in(1000, 1), dev(1000), a(5 * kHostPiece + 3), b(100), out(a.size()), out2(b.size());
    const HostCopy small[3] = {{out2.data(), b.data(), 40}, {out2.data() + 50, b.data() + 50, 40}, {out.data(), a.data(), 1000}};
    const HostCopy large[2] = {{out.data(), a.data(), a.size()}, {out2.data(), b.data(), b.size()}};
    bool quiet = true;
    int failed = 0;
    for (int pinned = 1; pinned >= 0; --pinned) {
        char* const area = h.pinned;
        if (!pinned) h.pinned = nullptr;
        for (int k = 0; k < 8; ++k)
            for (int which = 0; which < 2; ++which) {
                quiet &= hipMemcpyAsync(dev.data(), in.data(), in.size(), hipMemcpyHostToDevice, h.stream) == hipSuccess;  // the call's upload
                fake::state().copies_until_failure = k;
                failed += host_download(h, which ? large : small, which ? 2 : 3) != LT_OK;
                fake::state().copies_until_failure = -1;
                quiet &= fake::pending() == 0;
            }
        h.pinned = area;
    }
    expect(failed == 3 + 7 + 3 + 2, "a failing copy is reported");
    expect(quiet, "and nothing is left queued");
    expect(download(h, {9 * kHostPiece, 5}), "the next copy is whole");
    int thrown = 0, whole = 0;
    for (int k = 0; k < 40; ++k) {  // out of host memory: at the list of pieces, or at a thread's start
        g_fail_new = k;
        bool ok = false;
        try {
            ok = host_download(h, large, 2) == LT_OK;
        } catch (const std::bad_alloc&) {
            ++thrown;
        }
        g_fail_new = -1;
        whole += ok && out == a;
        quiet &= fake::pending() == 0;
    }
    expect(thrown >= 1 && thrown + whole == 40 && quiet, "out of memory the threads that did start take all");
}

int main(int argc, char** argv)
{
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "room") check_room();
    else if (what == "pinned") check_pinned();
    else if (what == "errors") check_errors();
    else return 2;
    std::puts(failures ? "FAILED" : "OK");
    return failures != 0;
}

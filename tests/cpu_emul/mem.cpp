// Device buffers and the block cache (rtg_mem.hip) on a stand-in for the HIP
// runtime: host blocks of a bounded "device", with the runtime's rules that
// the library relies on (a failed call's error is stored until it is read).
#include <cstdlib>
#include <map>
#include <memory>

#include "../../raytrace_amd/csrc/rtg_mem.hip"

namespace {
size_t g_room = 0, g_used = 0;  // bytes of the device, and in use
std::map<void *, size_t> g_live;
hipError_t g_stored = hipSuccess;
int g_mallocs = 0, g_frees = 0;
int g_device = 0, g_waited = -1;  // the thread's device, and the one last waited for
bool g_capturing = false;         // waits are refused, as while a stream captures
rtg::BlockCache *g_cache = nullptr;

hipError_t answer(hipError_t e) {
    if (e != hipSuccess) g_stored = e;
    return e;
}
}  // namespace

extern "C" {

hipError_t hipMalloc(void **p, size_t n) {
    if (g_used + n > g_room) return answer(hipErrorOutOfMemory);
    *p = malloc(16);
    g_live[*p] = n;
    g_used += n;
    ++g_mallocs;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    const auto it = g_live.find(p);
    if (it == g_live.end()) return answer(hipErrorInvalidValue);
    g_used -= it->second;
    g_live.erase(it);
    free(p);
    ++g_frees;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
    *d = g_device;
    return hipSuccess;
}
hipError_t hipSetDevice(int d) {
    g_device = d;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize(void) {
    if (g_capturing) return answer(hipErrorStreamCaptureUnsupported);
    g_waited = g_device;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    return g_capturing ? answer(hipErrorStreamCaptureUnsupported) : hipSuccess;
}
hipError_t hipGetLastError(void) {
    const hipError_t e = g_stored;
    g_stored = hipSuccess;
    return e;
}

}  // extern "C"

rtg::BlockCache *rtg::block_cache() { return g_cache; }

namespace {
// A fresh device of `room` bytes and an empty cache for the life of one case.
struct Case {
    rtg::BlockCache cache;
    explicit Case(size_t room) {
        g_room = room, g_used = 0, g_stored = hipSuccess, g_mallocs = g_frees = 0;
        g_device = cache.device = 0, g_waited = -1, g_capturing = false;
        g_cache = &cache;
    }
    ~Case() {
        cache.clear();
        g_cache = nullptr;
    }
};
constexpr size_t kMB = size_t(1) << 20;
}  // namespace

extern "C" {

// A kept block makes room for an allocation that would fail without it: the
// allocation succeeds and leaves no stored error behind (bit 0: its status,
// bit 1: the stored error); one that fails all the same leaves none either.
int mem_no_stored_error(int fits) {
    Case c(100 * kMB);
    { rtg::SceneBuf a; (void)a.alloc(60 * kMB); }  // into the cache
    rtg::DevBuf b;
    const int st = b.alloc((fits ? 90 : 110) * kMB);
    return (st == (fits ? RTG_OK : RTG_E_NOMEM) ? 0 : 1) | (hipGetLastError() == hipSuccess ? 0 : 2);
}

// A block that a refused wait could not show to be unused goes to hipFree, and
// the refusal leaves no stored error: how = 0 a buffer allocated anew, 1 a
// build's temporary, 2 (control) the same buffer after a wait that succeeded.
int mem_refused_wait(int how) {
    Case c(100 * kMB);
    {
        rtg::SceneBuf a;
        (void)a.alloc(kMB);
        g_capturing = how != 2;
        if (how == 1) {
            const rtg::SyncOnExit<1> idle{nullptr, {&a}};
        } else {
            (void)a.alloc(2 * kMB);
        }
    }
    g_capturing = false;
    // how 0: the first block freed, the second kept; 1: freed; 2: both kept
    const bool frees = g_frees == (how == 2 ? 0 : 1);
    return (frees ? 0 : 1) | (hipGetLastError() == hipSuccess ? 0 : 2);
}

// The wait is for the cache's device, also on a thread whose device is another.
int mem_waits_for_its_device(int thread_device) {
    Case c(100 * kMB);
    c.cache.device = 3;
    rtg::SceneBuf a;
    (void)a.alloc(kMB);
    g_device = thread_device;
    (void)a.alloc(2 * kMB);
    return (g_waited == 3 ? 0 : 1) | (g_device == thread_device ? 0 : 2);
}

// A program that moves on to other sizes: 512 MB of kept blocks that nobody
// takes any more, then `n` rounds of a buffer of `bytes` that comes and goes.
// Returns the rounds that had to allocate; -1 when more than 512 MB stay kept.
int mem_moves_on(int n, unsigned long long bytes) {
    Case c(~size_t(0) / 2);
    {
        rtg::SceneBuf old[128];
        for (rtg::SceneBuf &b : old) (void)b.alloc(4 * kMB);
    }
    const int before = g_mallocs;
    for (int k = 0; k < n; ++k) {
        rtg::SceneBuf b;
        (void)b.alloc((size_t)bytes);
    }
    return g_used > 512 * kMB ? -1 : g_mallocs - before;
}

// Blocks kept after `n` buffers of 16 bytes each are released.
int mem_small_blocks_kept(int n) {
    Case c(~size_t(0) / 2);
    {
        std::unique_ptr<rtg::SceneBuf[]> b(new rtg::SceneBuf[n]);
        for (int k = 0; k < n; ++k) (void)b[k].alloc(16);
    }
    return (int)g_live.size();
}

}  // extern "C"

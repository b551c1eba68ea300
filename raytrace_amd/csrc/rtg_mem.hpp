// rtg_mem.hpp — device memory of the library: buffers, and the cache of the
// blocks of destroyed scenes and finished builds.  Host code only, without
// kernels, so that it also runs against a stand-in for the runtime
// (tests/cpu_emul/mem.cpp).
#pragma once
#include <hip/hip_runtime.h>

#include <list>
#include <map>
#include <mutex>
#include <utility>

#include "../../include/rtg.h"

namespace rtg {

// Device allocation owned by a scene or the render arena.
struct DevBuf {
    void *p = nullptr;
    size_t bytes = 0;
    size_t cap = 0;       // size of the block behind it
    bool reuse = false;   // its block comes from the arena's BlockCache
    bool idle = true;     // and returns to it: false once a wait for its users failed
    int alloc(size_t n);  // RTG_OK / RTG_E_NOMEM
    void release();
    void swap(DevBuf &o) {
        std::swap(p, o.p), std::swap(bytes, o.bytes), std::swap(cap, o.cap), std::swap(reuse, o.reuse);
        std::swap(idle, o.idle);
    }
    ~DevBuf() { release(); }
    DevBuf() = default;
    DevBuf(const DevBuf &) = delete;
    DevBuf &operator=(const DevBuf &) = delete;
    template <class T>
    T *as() const { return static_cast<T *>(p); }
};

// A scene's arrays and a build's temporaries: nothing on the GPU may still use
// the block when it is released (hipFree would wait for the device; a cached
// block is handed out again at once).  Where the wait before that failed,
// `idle` is cleared, and the block goes to hipFree.
struct SceneBuf : DevBuf {
    SceneBuf() { reuse = true; }
};

// Device blocks of destroyed scenes and finished builds, kept for the next
// ones: a scene takes some 40 allocations, and each hipFree waits for the
// device.  At most kMost bytes are kept, each block counted in whole pages, as
// the runtime hands them out; a block that does not fit displaces the ones kept
// longest, so that sizes nobody asks for any more make way.  rtg_shutdown frees
// them, and so does an allocation of the library that fails.
class BlockCache {
public:
    int device = -1;  // of its blocks
    static constexpr size_t kMost = size_t(512) << 20, kPage = 4096;
    void *take(size_t n, size_t &cap);  // a kept block of n to 5/4 n bytes, or null
    bool keep(void *p, size_t cap);     // false: not kept (the caller frees it)
    void clear();
    ~BlockCache() { clear(); }

private:
    struct Block {
        void *p;
        size_t cap;
    };
    using Blocks = std::list<Block>;
    static size_t charge(size_t cap) { return (cap + kPage - 1) / kPage * kPage; }
    void drop(std::multimap<size_t, Blocks::iterator>::iterator it);  // forget it
    std::mutex m;
    Blocks blocks;  // the one kept longest first
    std::multimap<size_t, Blocks::iterator> by_size;
    size_t total = 0;
};

// The arena's cache; null before rtg_init and after rtg_shutdown.
BlockCache *block_cache();
// Wait for everything enqueued on the arena's device, whichever device is the
// calling thread's.  false: the wait failed (a stream captures, a device error).
bool device_idle();

// Waits for the stream before the buffers of a build are released, on every
// path; declared after them.
template <size_t N>
struct SyncOnExit {
    hipStream_t stream;
    SceneBuf *bufs[N];
    ~SyncOnExit() {
        if (hipStreamSynchronize(stream) == hipSuccess) return;
        (void)hipGetLastError();
        for (SceneBuf *b : bufs) b->idle = false;
    }
};

int ensure(DevBuf &b, size_t bytes);

}  // namespace rtg

// rtg_mem.hip — device buffers and the block cache (rtg_mem.hpp).
#include "rtg_mem.hpp"

namespace rtg {

void BlockCache::drop(std::multimap<size_t, Blocks::iterator>::iterator it) {
    total -= charge(it->first);
    blocks.erase(it->second);
    by_size.erase(it);
}
void *BlockCache::take(size_t n, size_t &cap) {
    std::lock_guard<std::mutex> l(m);
    const auto it = by_size.lower_bound(n);
    if (it == by_size.end() || it->first > n + n / 4) return nullptr;
    void *const p = it->second->p;
    cap = it->first;
    drop(it);
    return p;
}
bool BlockCache::keep(void *p, size_t cap) try {
    if (charge(cap) > kMost) return false;
    std::lock_guard<std::mutex> l(m);
    Blocks one{Block{p, cap}};
    const auto at = by_size.emplace(cap, one.begin());  // before anything is displaced: it may throw
    while (total + charge(cap) > kMost) {
        const Blocks::iterator old = blocks.begin();
        auto it = by_size.lower_bound(old->cap);
        while (it->second != old) ++it;  // (blocks of one size: the oldest is the first)
        (void)hipFree(old->p);
        drop(it);
    }
    blocks.splice(blocks.end(), one);
    total += charge(at->first);
    return true;
} catch (...) {  // no memory for the entry
    return false;
}
void BlockCache::clear() {
    std::lock_guard<std::mutex> l(m);
    for (const Block &b : blocks) (void)hipFree(b.p);
    blocks.clear();
    by_size.clear();
    total = 0;
}

int DevBuf::alloc(size_t n) {
    if (p != nullptr && reuse && !device_idle()) idle = false;  // renders may still read the old block
    release();
    if (n == 0) n = 16;
    BlockCache *const cache = block_cache();
    cap = n;
    if (reuse && cache) p = cache->take(n, cap);
    // The runtime stores a failed call's error until it is read, and the check
    // after a kernel launch reads it: each failure here is answered here.
    if (p == nullptr && hipMalloc(&p, n) != hipSuccess) {
        (void)hipGetLastError();
        if (cache) cache->clear();  // kept blocks make room
        if (hipMalloc(&p, n) != hipSuccess) {
            (void)hipGetLastError();
            p = nullptr;
            return RTG_E_NOMEM;
        }
    }
    bytes = n;
    idle = true;
    return RTG_OK;
}
void DevBuf::release() {
    BlockCache *const cache = reuse && idle ? block_cache() : nullptr;
    if (p != nullptr && !(cache && cache->keep(p, cap))) (void)hipFree(p);
    p = nullptr;
    bytes = cap = 0;
}
bool device_idle() {
    const BlockCache *const cache = block_cache();
    int cur = -1;
    if (cache == nullptr || hipGetDevice(&cur) != hipSuccess) return false;
    const bool other = cur != cache->device;
    const bool ok = (!other || hipSetDevice(cache->device) == hipSuccess) && hipDeviceSynchronize() == hipSuccess;
    if (other) (void)hipSetDevice(cur);
    if (!ok) (void)hipGetLastError();  // answered here, not by the next launch's check
    return ok;
}

int ensure(DevBuf &b, size_t n) {
    if (b.p != nullptr && b.bytes >= n) return RTG_OK;
    return b.alloc(n);
}

}  // namespace rtg

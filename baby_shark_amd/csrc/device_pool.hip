// A small per-device pool of released device blocks: the triangle soups that
// callers gave back (bs_device_free) and the large working buffers of calls
// that need them only while they run.  Giving a block of gigabytes back to
// the driver costs far more than the kernels that fill it: the driver clears
// freed memory in the background and the next large hipMalloc waits for it
// (dual contouring of 571 k leaves, a 1.4 GB soup, back to back: 39 ms a call
// with hipMalloc and hipFree, 3.6 ms with the pool).
//
// Blocks are handed out whole to requests of at least half their size.  At
// most BLOCKS blocks and BLOCK_BYTES bytes per device stay parked, the oldest
// leaving first; bs_release_cached_memory empties the pool, and so does any
// allocation of the library that runs out of memory, before it tries again.
#include <mutex>
#include <unordered_map>
#include <vector>

#include "common.hpp"

namespace bs {

namespace {

constexpr size_t BLOCKS = 16;
constexpr uint64_t BLOCK_BYTES = 8ull << 30;

struct DeviceBlock {
    void* p;
    uint64_t bytes;
    int device;
};

struct BlockPool {
    std::mutex mu;
    std::unordered_map<void*, DeviceBlock> live;  // blocks in use
    std::vector<DeviceBlock> idle;                // released blocks, oldest first
};

BlockPool& block_pool() {
    static BlockPool* p = new BlockPool();  // never destroyed: device memory may outlive static teardown
    return *p;
}

struct CurrentDevice {
    int prev = -1;
    explicit CurrentDevice(int dev) {
        (void)hipGetDevice(&prev);
        if (prev != dev) (void)hipSetDevice(dev);
    }
    ~CurrentDevice() {
        if (prev >= 0) (void)hipSetDevice(prev);
    }
};

void free_blocks(const std::vector<DeviceBlock>& blocks) {
    for (const DeviceBlock& b : blocks) {
        CurrentDevice g(b.device);
        (void)hipFree(b.p);
    }
}

// bs_refuse_allocations: requests of this thread so far, and the ones to refuse
thread_local uint64_t t_requests = 0, t_refuse_from = 0, t_refuse_to = 0;

hipError_t malloc_or_empty_pools(void** p, uint64_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        release_cached_memory();
        e = hipMalloc(p, bytes);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        *p = nullptr;
    }
    return e;
}

}  // namespace

bool allocation_refused() {
    ++t_requests;
    return t_requests >= t_refuse_from && t_requests < t_refuse_to;
}

uint64_t refuse_allocations(uint64_t first, uint64_t count) {
    const uint64_t seen = t_requests;
    t_requests = 0;
    t_refuse_from = first;
    t_refuse_to = first ? first + count : 0;
    return seen;
}

hipError_t device_malloc(void** p, uint64_t bytes) {
    *p = nullptr;
    return allocation_refused() ? hipErrorOutOfMemory : malloc_or_empty_pools(p, bytes);
}

void* alloc_block(uint64_t bytes) {
    if (!bytes) bytes = 256;
    if (allocation_refused()) BS_HIP(hipErrorOutOfMemory);
    int dev = -1;
    BS_HIP(hipGetDevice(&dev));
    BlockPool& P = block_pool();
    {
        std::lock_guard<std::mutex> lk(P.mu);
        int best = -1;
        for (int i = 0; i < (int)P.idle.size(); ++i) {  // the smallest that holds it and isn't twice too large
            const DeviceBlock& b = P.idle[i];
            if (b.device == dev && b.bytes >= bytes && b.bytes / 2 <= bytes && (best < 0 || b.bytes < P.idle[best].bytes))
                best = i;
        }
        if (best >= 0) {
            const DeviceBlock b = P.idle[best];
            P.live.emplace(b.p, b);
            P.idle.erase(P.idle.begin() + best);
            return b.p;
        }
    }
    void* p = nullptr;
    BS_HIP(malloc_or_empty_pools(&p, bytes));
    try {
        std::lock_guard<std::mutex> lk(P.mu);
        P.live.emplace(p, DeviceBlock{p, bytes, dev});
    } catch (...) {
        (void)hipFree(p);
        throw;
    }
    return p;
}

void free_block(void* p, bool wait) {
    if (!p) return;
    BlockPool& P = block_pool();
    DeviceBlock b{};
    {
        std::lock_guard<std::mutex> lk(P.mu);
        auto it = P.live.find(p);
        if (it != P.live.end()) {
            b = it->second;
            P.live.erase(it);
        } else {
            for (const DeviceBlock& parked : P.idle)
                if (parked.p == p) return;  // given back before: the pool's, and not the driver's to free
        }
    }
    if (!b.p) {  // not one of the pool's
        (void)hipFree(p);
        return;
    }
    std::vector<DeviceBlock> evict;
    bool parked = false;
    bool park = b.bytes <= BLOCK_BYTES;
    if (park && wait) {
        CurrentDevice g(b.device);
        park = hipDeviceSynchronize() == hipSuccess;
    }
    if (park) {
        try {
            evict.reserve(BLOCKS + 2);  // no more than that is parked on a device
            std::lock_guard<std::mutex> lk(P.mu);
            P.idle.push_back(b);
            parked = true;
            uint64_t bytes = 0;
            size_t count = 0;
            for (size_t i = P.idle.size(); i-- > 0;) {  // keep the newest within the limits
                if (P.idle[i].device != b.device) continue;
                if (count + 1 > BLOCKS || bytes + P.idle[i].bytes > BLOCK_BYTES) {
                    evict.push_back(P.idle[i]);
                    P.idle.erase(P.idle.begin() + i);
                } else {
                    bytes += P.idle[i].bytes;
                    ++count;
                }
            }
        } catch (const std::bad_alloc&) {  // the host is out of memory: the block goes back to the driver
        }
    }
    if (!parked) {
        CurrentDevice g(b.device);
        (void)hipFree(b.p);
    }
    free_blocks(evict);
}

void release_cached_memory() {
    release_cached_leaves();
    BlockPool& P = block_pool();
    std::vector<DeviceBlock> all;
    {
        std::lock_guard<std::mutex> lk(P.mu);
        all.swap(P.idle);
    }
    free_blocks(all);
}

}  // namespace bs

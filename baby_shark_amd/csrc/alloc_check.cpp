// The scratch arena and the block pool (common.hpp, device_pool.hip) on the CPU
// alone, over a HIP runtime of a few functions in host memory whose allocations
// can be made to fail (`make -C baby_shark_amd/csrc alloc_check`).  Exit status 0
// when every check holds.
#include <cstdio>
#include <cstdlib>
#include <set>

#include "common.hpp"

namespace {

std::set<void*> g_live;       // blocks of the runtime below
int g_fail_from = 0;          // this allocation (1: the next) and every later one fails; 0: none
int g_bad = 0;

#define CHECK(c)                                                                       \
    do {                                                                               \
        if (!(c)) {                                                                    \
            std::fprintf(stderr, "%s:%d: check failed: %s\n", __FILE__, __LINE__, #c); \
            ++g_bad;                                                                   \
        }                                                                              \
    } while (0)

}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) {
    if (g_fail_from == 1) return hipErrorOutOfMemory;
    if (g_fail_from > 1) --g_fail_from;
    *p = std::malloc(bytes);
    g_live.insert(*p);
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    if (p && !g_live.erase(p)) return hipErrorInvalidValue;
    std::free(p);
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
}

namespace bs {
void release_cached_leaves() {}
void set_last_error(const std::string&) {}
}  // namespace bs

using namespace bs;

static bool throws(Scratch& s, int slot, size_t bytes) {
    try {
        s.get(slot, bytes);
    } catch (const Error&) {
        return true;
    }
    return false;
}

// A buffer that could not grow is gone, and a later request of any size gets
// memory of its own or fails.
static void check_scratch() {
    Scratch s;
    CHECK(s.get(S_SUBS, 4096) != nullptr);
    g_fail_from = 1;
    CHECK(throws(s, S_SUBS, 1 << 20));
    CHECK(throws(s, S_SUBS, 1024));
    g_fail_from = 0;
    CHECK(s.get(S_SUBS, 1024) != nullptr);
    s.release();
    CHECK(g_live.empty());
}

// A request that the driver refuses empties the pool and tries once more; one
// that fails leaves nothing behind.
static void check_pool() {
    void* a = alloc_block(1 << 20);
    free_block(a);
    CHECK(g_live.size() == 1);
    CHECK(alloc_block(1 << 19) == a);  // of half its size
    free_block(a);
    g_fail_from = 1;
    bool failed = false;
    try {
        alloc_block(1 << 22);
    } catch (const Error&) {
        failed = true;
    }
    CHECK(failed);
    CHECK(g_live.empty());
    g_fail_from = 0;
    a = alloc_block(100);
    free_block(a, false);
    release_cached_memory();
    CHECK(g_live.empty());
}

// A block given back twice: the second time it is the pool's, which keeps it.
static void check_second_release() {
    void* a = alloc_block(1 << 20);
    free_block(a);
    free_block(a);
    CHECK(g_live.count(a) == 1);
    void* b = alloc_block(1 << 20);
    CHECK(g_live.count(b) == 1);
    free_block(b);
    release_cached_memory();
    CHECK(g_live.empty());
}

int main() {
    check_scratch();
    check_pool();
    check_second_release();
    if (g_bad) return 1;
    std::puts("allocation checks passed");
    return 0;
}

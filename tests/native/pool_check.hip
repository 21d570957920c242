// Host-side check of the buffers a context keeps (DevPool, drr_internal.h), with a
// stand-in for the device's memory of a given size.  Prints "ok" or the line of
// the first expectation that does not hold.
#include <hip/hip_runtime.h>
#include <stdio.h>
#include <stdlib.h>

#include <map>

namespace {
size_t g_free = 0;  // what the stand-in device has left
std::map<void *, size_t> g_live;

hipError_t fake_malloc(void **p, size_t n) {
    if (n > g_free) {
        *p = nullptr;
        return hipErrorOutOfMemory;
    }
    g_free -= n;
    *p = malloc(1);
    g_live[*p] = n;
    return hipSuccess;
}
hipError_t fake_free(void *p) {
    if (!p) return hipSuccess;
    g_free += g_live.at(p);
    g_live.erase(p);
    free(p);
    return hipSuccess;
}
size_t held() {
    size_t n = 0;
    for (auto &b : g_live) n += b.second;
    return n;
}
}  // namespace
#define hipMalloc fake_malloc
#define hipFree fake_free
#define hipGetLastError() hipSuccess
#include "../../deepdrr_amd/csrc/drr_internal.h"

#define EXPECT(x)                                    \
    do {                                             \
        if (!(x)) {                                  \
            printf("line %d: %s\n", __LINE__, #x);   \
            return 1;                                \
        }                                            \
    } while (0)

int main() {
    const size_t MB = (size_t)1 << 20;
    {
        g_free = 8192 * MB;
        auto pool = std::make_shared<DevPool>();
        PoolBuf a, b;
        // a volume's cells: the same size again takes the same buffer
        EXPECT(a.take(pool, 300 * MB) == hipSuccess);
        void *const first = a.as<char>();
        a.reset();
        EXPECT(held() == 300 * MB);
        EXPECT(a.take(pool, 300 * MB) == hipSuccess && a.as<char>() == first && held() == 300 * MB);
        // a smaller volume does not sit in it, and what no one takes is given back
        a.reset();
        EXPECT(a.take(pool, 200 * MB) == hipSuccess && held() == 200 * MB);
        // at most one is kept, and none of more than 2 GB
        EXPECT(b.take(pool, 100 * MB) == hipSuccess);
        a.reset();
        b.reset();
        EXPECT(held() <= 200 * MB);
        EXPECT(a.take(pool, 3000 * MB) == hipSuccess);
        a.reset();
        EXPECT(held() <= 200 * MB);
        // small ones: any that fits and is not over twice as large, 64 MB of them at most
        EXPECT(a.take(pool, 3 * MB) == hipSuccess);
        void *const small = a.as<char>();
        a.reset();
        EXPECT(b.take(pool, 2 * MB) == hipSuccess && b.as<char>() == small);
        b.reset();
        PoolBuf many[100];
        for (auto &m : many) EXPECT(m.take(pool, 8 * MB) == hipSuccess);
        for (auto &m : many) m.reset();
        EXPECT(held() <= 200 * MB + 64 * MB);
        for (auto &m : many) EXPECT(m.take(pool, 100) == hipSuccess);
        for (auto &m : many) m.reset();
        // a buffer whose work is not known to have ended is not handed on
        EXPECT(a.take(pool, 5000) == hipSuccess);
        void *const busy = a.as<char>();
        a.discard();
        EXPECT(!g_live.count(busy) && !a.as<char>());
        a.discard();  // nothing left to do
        pool.reset();
        EXPECT(g_live.empty());
    }
    {
        // when memory runs out every context's are given back, for any allocation
        g_free = 1000 * MB;
        auto one = std::make_shared<DevPool>(), two = std::make_shared<DevPool>();
        PoolBuf a, b;
        EXPECT(a.take(one, 600 * MB) == hipSuccess);
        a.reset();
        EXPECT(b.take(two, 700 * MB) == hipSuccess && held() == 700 * MB);
        b.reset();
        void *p = nullptr;
        EXPECT(drr_device_malloc(&p, 900 * MB) == hipSuccess && held() == 900 * MB);
        EXPECT(b.take(two, 700 * MB) == hipErrorOutOfMemory && !b.as<char>());
        EXPECT(drr_device_malloc(&p, 200 * MB) == hipErrorOutOfMemory);
        // a pool outlives its context in what it lent
        g_free = 1000 * MB;
        EXPECT(b.take(two, 30 * MB) == hipSuccess);
        two.reset();
        b.reset();
        EXPECT(held() == 900 * MB);
        one.reset();
        EXPECT(held() == 900 * MB);
    }
    printf("ok\n");
    return 0;
}

// The device and pinned-memory pools.  Calls of equal size reuse their
// workspaces; a hipFree would wait for the device.
#include "pool.hpp"

#include "common.hpp"

#include <memory>

namespace idrs {
namespace {

// The idle buffers of a device stay within a quarter of its memory.  The
// pools live until the process ends.
std::mutex g_pools_mu;
std::map<int, BufferPool *> g_pools;

BufferPool &device_pool(int dev) {
    std::lock_guard<std::mutex> g(g_pools_mu);
    BufferPool *&p = g_pools[dev];
    if (!p) {
        size_t left = 0, total = 0;
        const size_t cap = hipMemGetInfo(&left, &total) == hipSuccess ? total / 4 : size_t(1) << 30;
        p = new BufferPool({[](size_t bytes) {
                                void *q = nullptr;
                                if (hipMalloc(&q, bytes) == hipSuccess) return q;
                                (void)hipGetLastError();
                                return (void *)nullptr;
                            },
                            [](void *q) { (void)hipFree(q); }},
                           cap);
    }
    return *p;
}

size_t pool_round(size_t bytes) {
    bytes = (bytes + 255) & ~(size_t)255;
    return bytes ? bytes : 256;
}

std::mutex g_pinned_mu;
std::multimap<std::pair<size_t, unsigned>, void *> g_pinned;

}  // namespace

hipError_t dev_malloc_bytes(void **p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipErrorOutOfMemory) return e;
    (void)hipGetLastError();
    int dev = 0;
    if ((e = hipGetDevice(&dev)) != hipSuccess) return e;
    *p = device_pool(dev).allocate(bytes);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}

size_t pool_release() {
    std::vector<BufferPool *> all;
    {
        std::lock_guard<std::mutex> g(g_pools_mu);
        for (auto &e : g_pools) all.push_back(e.second);
    }
    size_t freed = 0;
    for (BufferPool *p : all) freed += p->trim();
    return freed;
}

void *pool_try_alloc(size_t bytes) {
    int dev = 0;
    HIP_TRY(hipGetDevice(&dev));
    return device_pool(dev).take(pool_round(bytes));
}

void *pool_alloc(size_t bytes) {
    void *p = pool_try_alloc(bytes);
    if (!p) {
        set_last_error("no device memory for %zu bytes", bytes);
        throw HipError{hipErrorOutOfMemory};
    }
    return p;
}

void pool_free(void *p, size_t bytes) {
    if (!p) return;
    int dev = 0;
    if (hipPointerAttribute_t at{}; hipPointerGetAttributes(&at, p) == hipSuccess) dev = at.device;
    device_pool(dev).give(p, pool_round(bytes));
}

void *pinned_take(size_t bytes, unsigned flags) {
    bytes = pool_round(bytes);
    {
        std::lock_guard<std::mutex> g(g_pinned_mu);
        auto it = g_pinned.find({bytes, flags});
        if (it != g_pinned.end()) {
            void *p = it->second;
            g_pinned.erase(it);
            return p;
        }
    }
    void *p = nullptr;
    HIP_TRY(hipHostMalloc(&p, bytes, flags));
    return p;
}

void pinned_give(void *p, size_t bytes, unsigned flags) {
    if (!p) return;
    std::lock_guard<std::mutex> g(g_pinned_mu);
    g_pinned.emplace(std::make_pair(pool_round(bytes), flags), p);
}

}  // namespace idrs

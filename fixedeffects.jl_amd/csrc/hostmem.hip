// hostmem.hip -- see hostmem.h.
#include "hostmem.h"

#include <map>
#include <mutex>
#include <vector>

namespace fehip {

namespace {

// Size classes: powers of two up to 64 KB, then steps of an eighth of the
// power of two below, so a block is at most 1/8 larger than asked for and
// handles of nearly the same size share blocks.
size_t size_class(size_t b) {
    if (b <= 256) return 256;
    size_t p = 256;
    while (p * 2 <= b) p *= 2;
    if (p == b) return b;
    if (b <= 65536) return 2 * p;
    const size_t step = p / 8;
    return (b + step - 1) / step * step;
}

struct Pool {
    std::mutex mu;
    std::multimap<size_t, void *> blocks;
    size_t held = 0;
};

// one per device, never destroyed (handles may be closed at process exit)
Pool &pool_of(int device) {
    static std::mutex mu;
    static std::map<int, Pool *> *pools = new std::map<int, Pool *>();
    std::lock_guard<std::mutex> lk(mu);
    Pool *&p = (*pools)[device];
    if (!p) p = new Pool();
    return *p;
}

}  // namespace

hipError_t pool_get(size_t bytes, void **ptr, size_t *size, int *device) {
    *ptr = nullptr;
    hipError_t e = hipGetDevice(device);
    if (e != hipSuccess) return e;
    *size = size_class(bytes);
    Pool &p = pool_of(*device);
    {
        std::lock_guard<std::mutex> lk(p.mu);
        auto it = p.blocks.find(*size);
        if (it != p.blocks.end()) {
            *ptr = it->second;
            p.held -= *size;
            p.blocks.erase(it);
            return hipSuccess;
        }
    }
    e = hipMalloc(ptr, *size);
    if (e == hipSuccess) return e;
    (void)hipGetLastError();
    std::vector<void *> out;
    {
        std::lock_guard<std::mutex> lk(p.mu);
        for (auto &b : p.blocks) out.push_back(b.second);
        p.blocks.clear();
        p.held = 0;
    }
    for (void *q : out) (void)hipFree(q);
    *ptr = nullptr;
    return hipMalloc(ptr, *size);
}

void pool_put(void *ptr, size_t size, int device) {
    Pool &p = pool_of(device);
    {
        std::lock_guard<std::mutex> lk(p.mu);
        if (p.held + size <= kPoolBytes) {
            p.blocks.emplace(size, ptr);
            p.held += size;
            return;
        }
    }
    (void)hipFree(ptr);
}

}  // namespace fehip

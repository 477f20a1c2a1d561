// hostmem.hip -- see hostmem.h.
#include "hostmem.h"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

namespace fehip {

namespace {

// Size classes: powers of two up to 64 KB, then steps of an eighth of the
// power of two below, so a block is at most 1/8 larger than asked for and
// handles of nearly the same size share blocks; from 1 GiB on, steps of 2 MiB
// (what the device maps), so a handle that fills the device gives little away.
size_t size_class(size_t b) {
    if (b >= size_t(1) << 30) return (b + (size_t(2) << 20) - 1) >> 21 << 21;
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
    size_t total = 0;  // blocks in use and held

    // hipMalloc and hipFree, counted (mu is not held)
    hipError_t take(void **ptr, size_t size, size_t limit) {
        {
            std::lock_guard<std::mutex> lk(mu);
            if (size > limit || total > limit - size) return hipErrorOutOfMemory;
            total += size;
        }
        const hipError_t e = hipMalloc(ptr, size);
        if (e == hipSuccess) return e;
        (void)hipGetLastError();
        *ptr = nullptr;
        std::lock_guard<std::mutex> lk(mu);
        total -= size;
        return e;
    }
    void drop(void *ptr, size_t size) {
        (void)hipFree(ptr);
        std::lock_guard<std::mutex> lk(mu);
        total -= size;
    }
    bool over(size_t limit) {
        std::lock_guard<std::mutex> lk(mu);
        return total > limit;
    }
    void trim() {
        std::multimap<size_t, void *> out;
        {
            std::lock_guard<std::mutex> lk(mu);
            out.swap(blocks);
            held = 0;
        }
        for (auto &b : out) drop(b.second, b.first);
    }
};

std::atomic<size_t> g_limit{SIZE_MAX};  // FEHIP_DEVICE_MB, in bytes

// one per device, never destroyed (handles may be closed at process exit)
struct Pools {
    std::mutex mu;
    std::map<int, Pool *> by_device;
};
Pools &pools() {
    static Pools *p = new Pools();
    return *p;
}
Pool &pool_of(int device) {
    Pools &ps = pools();
    std::lock_guard<std::mutex> lk(ps.mu);
    Pool *&p = ps.by_device[device];
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
    const size_t limit = g_limit.load(std::memory_order_relaxed);
    if (limit != SIZE_MAX && p.over(limit)) p.trim();
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
    e = p.take(ptr, *size, limit);
    if (e == hipSuccess) return e;
    p.trim();
    return p.take(ptr, *size, limit);
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
    p.drop(ptr, size);
}

void pool_read_limit() {
    const char *env = getenv("FEHIP_DEVICE_MB");
    g_limit.store(env && *env ? (size_t)std::max(0ll, atoll(env)) << 20 : SIZE_MAX, std::memory_order_relaxed);
}

void pool_trim() {
    std::vector<Pool *> all;
    {
        std::lock_guard<std::mutex> lk(pools().mu);
        for (auto &p : pools().by_device) all.push_back(p.second);
    }
    for (Pool *p : all) p->trim();
}

// ---------------------------------------------------------------------------
// copies of pageable host memory
//
// The runtime's own copy of pageable memory goes through one thread: 80 MB
// arrive on the device at 29 GB/s and leave it at 17.  Here a few threads
// take chunks of the array in turn; each fills (or empties) pinned buffers of
// its own and queues the copies on the caller's stream, so the host's reads,
// the link and the page faults of fresh output arrays overlap.  Refs are
// narrowed to the 4 bytes the device keeps on the way, which halves their
// traffic on the link, and range-checked.
// ---------------------------------------------------------------------------
namespace {

constexpr int kThreads = 7;                        // with the calling one
constexpr size_t kChunk = size_t(2) << 20;         // bytes of one pinned buffer
// Smaller copies take the runtime's own path.  Measured, staged against
// runtime: to the device 8 MB 383 / 234 us, 16 MB 548 / 453, 80 MB 2110 / 2779
// (as refs, narrowed to 40 MB: 1447); from the device 2 MB 118 / 148 us, 8 MB
// 363 / 481, 80 MB 2015 / 4698.
constexpr size_t kInBytes = size_t(32) << 20;
constexpr size_t kOutBytes = size_t(2) << 20;

struct Staging {
    std::mutex use;  // one staged copy at a time; others take the runtime's path
    unsigned char *buf = nullptr;  // kThreads x 2 x kChunk, pinned
    std::map<int, std::vector<hipEvent_t>> events;  // per device, one per buffer
    // threads
    std::mutex mu;
    std::condition_variable work, done;
    const std::function<void(int)> *job = nullptr;
    uint64_t round = 0;
    int left = 0, nthreads = 0;
    bool ready = false, failed = false;

    bool init(int device) {
        if (failed) return false;
        if (!buf && hipHostMalloc((void **)&buf, kThreads * 2 * kChunk, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            buf = nullptr;
            failed = true;
            return false;
        }
        std::vector<hipEvent_t> &ev = events[device];
        while (ev.size() < 2 * kThreads) {
            hipEvent_t e = nullptr;
            if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                failed = true;
                return false;
            }
            ev.push_back(e);
        }
        if (!ready) {
            ready = true;
            const int want = std::min<int>(kThreads - 1, (int)std::max(2u, std::thread::hardware_concurrency()) / 2);
            for (int i = 0; i < want; i++) {
                try {
                    std::thread([this, i] { loop(i + 1); }).detach();
                } catch (...) {
                    break;  // fewer threads do the same work
                }
                nthreads++;
            }
        }
        return true;
    }

    void loop(int id) {
        uint64_t seen = 0;
        for (;;) {
            const std::function<void(int)> *f;
            {
                std::unique_lock<std::mutex> lk(mu);
                work.wait(lk, [&] { return round != seen; });
                seen = round;
                f = job;
            }
            (*f)(id);
            std::lock_guard<std::mutex> lk(mu);
            if (--left == 0) done.notify_one();
        }
    }

    // f(id) on every thread, 0 the caller
    void run(const std::function<void(int)> &f) {
        {
            std::lock_guard<std::mutex> lk(mu);
            job = &f;
            left = nthreads;
            round++;
        }
        work.notify_all();
        f(0);
        std::unique_lock<std::mutex> lk(mu);
        done.wait(lk, [&] { return left == 0; });
    }
};

Staging &staging() {
    static Staging *s = new Staging();  // its threads live as long as the process
    return *s;
}

// fill(dst, first, count): write elements [first, first + count) into a pinned
// buffer.  n elements of out_size bytes each on the device.  False: not taken.
template <typename F>
bool staged_in(void *dst, int64_t n, size_t out_size, hipStream_t st, F &&fill, hipError_t *err) {
    Staging &s = staging();
    std::unique_lock<std::mutex> lk(s.use, std::try_to_lock);
    int dev = 0;
    if (!lk.owns_lock() || hipGetDevice(&dev) != hipSuccess || !s.init(dev)) return false;
    // chunks small enough that every thread gets some of a small copy
    const int64_t most = (int64_t)(kChunk / out_size);
    const int64_t per = std::min<int64_t>(most, std::max<int64_t>(most / 4, (n + 2 * kThreads - 1) / (2 * kThreads)));
    std::atomic<int64_t> next{0};
    std::atomic<int> bad{(int)hipSuccess};
    hipEvent_t *ev = s.events[dev].data();
    const std::function<void(int)> f = [&](int id) {
        if (id && hipSetDevice(dev) != hipSuccess) return;
        bool used[2] = {false, false};
        for (int slot = 0;; slot ^= 1) {
            const int64_t a = next.fetch_add(per);
            if (a >= n || bad.load() != (int)hipSuccess) break;
            const int64_t c = std::min(per, n - a);
            unsigned char *b = s.buf + (size_t)(2 * id + slot) * kChunk;
            hipError_t e = used[slot] ? hipEventSynchronize(ev[2 * id + slot]) : hipSuccess;
            if (e == hipSuccess) {
                fill(b, a, c);
                e = hipMemcpyAsync((unsigned char *)dst + (size_t)a * out_size, b, (size_t)c * out_size,
                                   hipMemcpyHostToDevice, st);
            }
            if (e == hipSuccess) e = hipEventRecord(ev[2 * id + slot], st);
            used[slot] = true;
            if (e != hipSuccess) {
                bad.store((int)e);
                break;
            }
        }
        // the buffers are the next copy's too
        for (int slot = 0; slot < 2; slot++)
            if (used[slot]) (void)hipEventSynchronize(ev[2 * id + slot]);
    };
    s.run(f);
    *err = (hipError_t)bad.load();
    return true;
}

}  // namespace

hipError_t copy_in(void *dst, const void *src, size_t bytes, hipStream_t st) {
    hipError_t e = hipSuccess;
    if (bytes >= kInBytes && staged_in(dst, (int64_t)bytes, 1, st,
                  [&](void *b, int64_t a, int64_t c) { std::memcpy(b, (const unsigned char *)src + a, (size_t)c); }, &e))
        return e;
    return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st);
}

bool copy_in_refs(int32_t *dst, const int64_t *src, int64_t n, int64_t nlev, bool *bad, hipStream_t st,
                  hipError_t *err) {
    if ((size_t)n * sizeof(int64_t) < kInBytes) return false;
    std::atomic<bool> out{false};
    if (!staged_in(dst, n, sizeof(int32_t), st,
                   [&](void *buf, int64_t a, int64_t c) {
                       int32_t *b = (int32_t *)buf;
                       bool any = false;
                       for (int64_t i = 0; i < c; i++) {
                           const int64_t v = src[a + i];
                           any |= (uint64_t)(v - 1) >= (uint64_t)nlev;
                           b[i] = (int32_t)(v - 1);
                       }
                       if (any) out.store(true);
                   },
                   err))
        return false;
    *bad = out.load();
    return true;
}

hipError_t copy_out(void *dst, const void *src, size_t bytes, hipStream_t st) {
    Staging &s = staging();
    std::unique_lock<std::mutex> lk(s.use, std::defer_lock);
    int dev = 0;
    if (bytes < kOutBytes || !lk.try_lock() || hipGetDevice(&dev) != hipSuccess || !s.init(dev)) {
        const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st);
        return e == hipSuccess ? hipStreamSynchronize(st) : e;
    }
    const size_t per = std::min(kChunk, std::max(kChunk / 4, (bytes + 2 * kThreads - 1) / (2 * kThreads)));
    std::atomic<size_t> next{0};
    std::atomic<int> bad{(int)hipSuccess};
    hipEvent_t *ev = s.events[dev].data();
    const std::function<void(int)> f = [&](int id) {
        if (id && hipSetDevice(dev) != hipSuccess) return;
        size_t at[2], len[2] = {0, 0};
        auto issue = [&](int slot) {
            len[slot] = 0;
            const size_t a = next.fetch_add(per);
            if (a >= bytes || bad.load() != (int)hipSuccess) return;
            at[slot] = a;
            const size_t c = std::min(per, bytes - a);
            hipError_t e = hipMemcpyAsync(s.buf + (size_t)(2 * id + slot) * kChunk, (const unsigned char *)src + a, c,
                                          hipMemcpyDeviceToHost, st);
            if (e == hipSuccess) e = hipEventRecord(ev[2 * id + slot], st);
            if (e != hipSuccess) bad.store((int)e);
            else len[slot] = c;
        };
        issue(0);
        for (int slot = 0; len[slot]; slot ^= 1) {
            issue(slot ^ 1);
            const hipError_t e = hipEventSynchronize(ev[2 * id + slot]);
            if (e != hipSuccess) {
                bad.store((int)e);
                break;
            }
            std::memcpy((unsigned char *)dst + at[slot], s.buf + (size_t)(2 * id + slot) * kChunk, len[slot]);
            len[slot] = 0;
        }
        // (a buffer still in flight after an error)
        for (int slot = 0; slot < 2; slot++)
            if (len[slot]) (void)hipEventSynchronize(ev[2 * id + slot]);
    };
    s.run(f);
    return (hipError_t)bad.load();
}

}  // namespace fehip

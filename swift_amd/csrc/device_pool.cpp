// device_pool.cpp -- see device_pool.hpp.
#include <algorithm>
#include <list>
#include <mutex>
#include <unordered_map>
#include <utility>

#include "device_pool.hpp"

namespace swift {

namespace {

struct Block {
    void *ptr;
    size_t size;
    int dev;
    uint64_t freed;  // the pool's count of frees when it was kept
    bool leaving;    // in pool_free, on its way to the kept ones
    bool idle;       // the device was waited for after its owner let it go
};

struct Pool {
    std::mutex mu;
    std::unordered_map<void *, Block> live;  // allocated here, in use
    std::list<Block> kept;                   // oldest first
    std::unordered_map<int, size_t> bytes;   // kept, by device
    // by device: what was kept by this count of frees was waited for
    std::unordered_map<int, uint64_t> waited;
    uint64_t frees = 0;
};
Pool &pool() {
    static Pool *p = new Pool;  // lives until the process ends
    return *p;
}

// sizes in steps of an eighth of their power of two, so that calls of slightly
// different sizes share blocks
size_t block_size(size_t bytes) {
    size_t step = 256;
    while (step * 16 <= bytes) step <<= 1;
    return (bytes + step - 1) / step * step;
}

// False once the caller has given the block's pointer to hipFree itself: its
// address is then unmapped or another allocation's.
bool mapped(const Block &b) {
    hipDeviceptr_t base = nullptr;
    size_t size = 0;
    if (hipMemGetAddressRange(&base, &size, (hipDeviceptr_t)b.ptr) == hipSuccess)
        return base == (hipDeviceptr_t)b.ptr && size >= b.size;
    (void)hipGetLastError();
    return false;
}

// Takes the kept blocks that `which` names out of the pool, to be given back
// without its lock: hipFree waits for the device, and other threads allocate.
template <class Which> std::list<Block> take(Pool &p, Which which) {
    std::list<Block> out;
    for (auto it = p.kept.begin(); it != p.kept.end();) {
        auto at = it++;
        if (!which(*at)) continue;
        p.bytes[at->dev] -= at->size;
        out.splice(out.end(), p.kept, at);
    }
    return out;
}

// (hipFree's device is the block's own, whichever is current; what it refuses,
// in a thread that captures a stream, is kept)
void give_back(Pool &p, std::list<Block> blocks) {
    for (auto it = blocks.begin(); it != blocks.end();) {
        auto at = it++;
        if (!mapped(*at) || hipFree(at->ptr) == hipSuccess) blocks.erase(at);
        else (void)hipGetLastError();
    }
    std::lock_guard<std::mutex> lk(p.mu);
    for (const Block &b : blocks) p.bytes[b.dev] += b.size;
    p.kept.splice(p.kept.begin(), blocks);
}

// Waits for the device as hipFree does, by a hipFree (1.3 us with the
// allocation): hipDeviceSynchronize would end every stream capture in progress,
// also those under which another thread may allocate and free.  What was kept
// before is idle then.
bool wait_idle(Pool &p, int dev) {
    uint64_t before;
    {
        std::lock_guard<std::mutex> lk(p.mu);
        before = p.frees;
    }
    void *one = nullptr;
    if (hipMalloc(&one, 1) != hipSuccess || hipFree(one) != hipSuccess) return false;
    std::lock_guard<std::mutex> lk(p.mu);
    try {
        uint64_t &w = p.waited[dev];
        w = std::max(w, before);
    } catch (...) {  // no memory for the pool's own tables: nothing is marked
    }
    return true;
}

}  // namespace

// The kept block of this size let go last (the likeliest to be in the caches),
// of those known to be idle; *wait: there are only others.
static void *from_kept(Pool &p, int dev, size_t size, bool *wait) {
    std::lock_guard<std::mutex> lk(p.mu);
    *wait = false;
    for (auto it = p.kept.end(); it != p.kept.begin();) {
        --it;
        if (it->dev != dev || it->size != size) continue;
        const bool there = mapped(*it);
        if (there && !it->idle && it->freed > p.waited[dev]) {
            *wait = true;
            continue;
        }
        void *ptr = it->ptr;
        if (there) p.live[ptr] = *it;
        p.bytes[dev] -= size;
        it = p.kept.erase(it);
        if (there) return ptr;
    }
    return nullptr;
}

static hipError_t alloc_from_pool(void **ptr, size_t bytes, bool may_wait) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (bytes > kPoolBlock && (e = hipMalloc(ptr, bytes)) != hipErrorOutOfMemory) return e;
    Pool &p = pool();
    const size_t size = bytes > kPoolBlock ? bytes : block_size(bytes ? bytes : 1);
    if (bytes <= kPoolBlock) {
        bool wait;
        void *got = from_kept(p, dev, size, &wait);
        if (!got && wait && may_wait && wait_idle(p, dev)) got = from_kept(p, dev, size, &wait);
        if (got) {
            *ptr = got;
            return hipSuccess;
        }
        (void)hipGetLastError();
        e = hipSuccess;
    }
    if (e == hipSuccess) e = hipMalloc(ptr, size);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        if (pool_trim() == hipSuccess) e = hipMalloc(ptr, size);
    }
    if (e == hipSuccess && size <= kPoolBlock) {
        std::lock_guard<std::mutex> lk(p.mu);
        try {
            p.live[*ptr] = Block{*ptr, size, dev, 0, false, false};
        } catch (...) {  // not entered: pool_free hands it to hipFree
        }
    }
    return e;
}

hipError_t pool_alloc(void **ptr, size_t bytes, bool may_wait) {
    hipError_t e;
    try {
        e = alloc_from_pool(ptr, bytes, may_wait);
    } catch (...) {  // no memory for the pool's own tables
        e = hipMalloc(ptr, bytes ? bytes : 1);
    }
    if (e != hipSuccess) (void)hipGetLastError();  // reported here, not by the next launch
    return e;
}

hipError_t pool_trim() {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    Pool &p = pool();
    std::unique_lock<std::mutex> lk(p.mu);
    std::list<Block> out = take(p, [&](const Block &b) { return b.dev == dev; });
    lk.unlock();
    give_back(p, std::move(out));
    return hipSuccess;
}

hipError_t device_malloc(void **ptr, size_t bytes) {
    hipError_t e = hipMalloc(ptr, bytes);
    if (e == hipErrorOutOfMemory && pool_trim() == hipSuccess) e = hipMalloc(ptr, bytes);
    if (e != hipSuccess) (void)hipGetLastError();  // reported here, not by the next launch
    return e;
}

hipError_t pool_free(void *ptr, bool wait) {
    if (!ptr) return hipSuccess;
    Pool &p = pool();
    Block b{};
    {
        std::lock_guard<std::mutex> lk(p.mu);
        auto it = p.live.find(ptr);
        if (it == p.live.end()) {
            // freed before: hipFree would unmap what the next owner is handed
            for (const Block &k : p.kept)
                if (k.ptr == ptr) return hipErrorInvalidValue;
        } else if (it->second.leaving) {
            return hipErrorInvalidValue;
        } else {
            it->second.leaving = true;
            b = it->second;
        }
    }
    if (!b.ptr) return hipFree(ptr);
    int dev = 0;
    const bool keep = hipGetDevice(&dev) == hipSuccess && dev == b.dev && mapped(b) &&
                      (!wait || wait_idle(p, dev));
    if (!keep) (void)hipGetLastError();
    std::unique_lock<std::mutex> lk(p.mu);
    p.live.erase(ptr);
    b.freed = ++p.frees;
    b.leaving = false;
    b.idle = wait;
    bool kept = false;
    if (keep) {
        try {
            size_t &held = p.bytes[dev];
            p.kept.push_back(b);
            held += b.size;
            kept = true;
        } catch (...) {  // no memory for the pool's own tables
        }
    }
    if (!kept) {
        lk.unlock();
        return hipFree(ptr);
    }
    std::list<Block> out = take(p, [&](const Block &k) {
        return k.freed + kPoolAge < p.frees || (k.dev == dev && p.bytes[dev] > kPoolBytes);
    });
    lk.unlock();
    if (!out.empty()) give_back(p, std::move(out));
    return hipSuccess;
}

}  // namespace swift

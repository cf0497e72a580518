// Kept blocks of device memory (asx_pool.hpp).
#include "asx_pool.hpp"

#include <stdint.h>

#include <algorithm>
#include <mutex>
#include <unordered_map>
#include <vector>

namespace asx {

namespace {

struct Block {
    void *p;
    size_t bytes;
    int dev;
    uint64_t id;
};
struct Pinned {
    void *p;
    uint64_t id;
};

struct Pool {
    std::mutex lock;
    std::unordered_map<const void *, Block> live;
    std::vector<Block> kept;  // oldest first
    std::vector<Pinned> pinned;
};

// Never destroyed: at process exit the HIP runtime may be gone before static objects are.
Pool &pool()
{
    static Pool *p = new Pool;
    return *p;
}

// HIP's number of the allocation at p; every allocation has another one, also at the address of an earlier one (0: there is
// none).  hipDeviceReset takes all memory of the device, and what lies at a kept address afterwards, if anything, is
// somebody else's: a block counts as the pool's only while its number is the one it was allocated with.
uint64_t allocation_id(const void *p)
{
    uint64_t id = 0;
    if (hipPointerGetAttribute(&id, HIP_POINTER_ATTRIBUTE_BUFFER_ID, const_cast<void *>(p)) == hipSuccess) return id;
    (void)hipGetLastError();  // or the next launch would seem to have failed
    return 0;
}

hipError_t device_free(const Block &b)
{
    if (allocation_id(b.p) != b.id) return hipErrorInvalidValue;
    return hipFree(b.p);
}

// Sizes in eighths of a power of two: requests that differ a little meet each other's blocks.
size_t rounded(size_t bytes)
{
    size_t step = 65536;
    while (step * 16 <= bytes) step *= 2;
    return (std::max<size_t>(bytes, 1) + step - 1) / step * step;
}

class OnDevice {
public:
    explicit OnDevice(int dev)
    {
        (void)hipGetDevice(&was_);
        if (was_ != dev) (void)hipSetDevice(dev), moved_ = true;
    }
    ~OnDevice()
    {
        if (moved_) (void)hipSetDevice(was_);
    }

private:
    int was_ = 0;
    bool moved_ = false;
};

// Takes blocks of `dev` out of the kept ones (all of them, or the oldest beyond the bounds).
std::vector<Block> surplus(Pool &P, int dev, bool all)
{
    std::vector<Block> out;
    size_t bytes = 0, blocks = 0;
    for (const Block &b : P.kept)
        if (b.dev == dev) bytes += b.bytes, ++blocks;
    for (size_t i = 0; i < P.kept.size();) {
        const Block b = P.kept[i];
        if (b.dev != dev || !(all || bytes > kPoolMaxBytes || blocks > kPoolMaxBlocks)) {
            ++i;
            continue;
        }
        bytes -= b.bytes;
        --blocks;
        out.push_back(b);
        P.kept.erase(P.kept.begin() + (std::ptrdiff_t)i);
    }
    return out;
}

}  // namespace

hipError_t pool_malloc_bytes(void **p, size_t bytes, bool brief)
{
    *p = nullptr;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const size_t want = rounded(bytes);
    Pool &P = pool();
    const size_t most = brief ? 4 * want : want + want / 4;
    for (;;) {
        Block b;
        {
            std::lock_guard<std::mutex> g(P.lock);
            size_t best = P.kept.size();
            for (size_t i = 0; i < P.kept.size(); ++i) {
                const Block &k = P.kept[i];
                if (k.dev == dev && k.bytes >= want && k.bytes <= most && (best == P.kept.size() || k.bytes < P.kept[best].bytes)) best = i;
            }
            if (best == P.kept.size()) break;
            b = P.kept[best];
            P.kept.erase(P.kept.begin() + (std::ptrdiff_t)best);
        }
        if (allocation_id(b.p) != b.id) continue;  // lost in a reset of the device
        std::lock_guard<std::mutex> g(P.lock);
        P.live[b.p] = b;
        *p = b.p;
        return hipSuccess;
    }
    size_t got = want;
    e = hipMalloc(p, got);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        pool_release();
        e = hipMalloc(p, got);
        if (e == hipErrorOutOfMemory && bytes > 0 && bytes < want) {
            (void)hipGetLastError();
            got = bytes;
            e = hipMalloc(p, got);
        }
    }
    if (e != hipSuccess) {
        *p = nullptr;
        return e;
    }
    const uint64_t id = allocation_id(*p);
    std::lock_guard<std::mutex> g(P.lock);
    P.live[*p] = Block{*p, got, dev, id};
    return hipSuccess;
}

void pool_free(void *p, bool idle)
{
    if (!p) return;
    if (!idle) {
        (void)pool_return(p);
        return;
    }
    Pool &P = pool();
    std::vector<Block> out;
    {
        std::lock_guard<std::mutex> g(P.lock);
        const auto it = P.live.find(p);
        if (it == P.live.end()) return;  // not a block of this pool
        const Block b = it->second;
        P.live.erase(it);
        if (b.bytes > kPoolMaxBlockBytes) {
            out.push_back(b);
        } else {
            P.kept.push_back(b);
            out = surplus(P, b.dev, false);
        }
    }
    for (const Block &b : out) {
        OnDevice on(b.dev);
        (void)device_free(b);
    }
}

// hipFree waits for every stream of the device, and is allowed where hipDeviceSynchronize is refused and costs the capture:
// while a stream is captured in relaxed mode, or by another thread in thread-local mode.  1.4 us for a block of this size on
// an idle device, hipDeviceSynchronize 0.2.
bool pool_wait(const void *p)
{
    if (!p) return true;
    Pool &P = pool();
    int dev;
    {
        std::lock_guard<std::mutex> g(P.lock);
        const auto it = P.live.find(p);
        if (it == P.live.end()) return true;
        dev = it->second.dev;
    }
    OnDevice on(dev);
    void *token = nullptr;
    return hipMalloc(&token, 64) == hipSuccess && hipFree(token) == hipSuccess;
}

hipError_t pool_return(void *p)
{
    if (!p) return hipSuccess;
    Pool &P = pool();
    Block b;
    {
        std::lock_guard<std::mutex> g(P.lock);
        const auto it = P.live.find(p);
        if (it == P.live.end()) return hipErrorInvalidValue;
        b = it->second;
        P.live.erase(it);
    }
    OnDevice on(b.dev);
    return device_free(b);
}

size_t pool_kept_bytes()
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    Pool &P = pool();
    std::lock_guard<std::mutex> g(P.lock);
    size_t bytes = 0;
    for (const Block &b : P.kept)
        if (b.dev == dev) bytes += b.bytes;
    return bytes;
}

void pool_release()
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return;
    Pool &P = pool();
    std::vector<Block> out;
    {
        std::lock_guard<std::mutex> g(P.lock);
        out = surplus(P, dev, true);
    }
    for (const Block &b : out) (void)device_free(b);
}

void *pinned_take()
{
    Pool &P = pool();
    for (;;) {
        Pinned k;
        {
            std::lock_guard<std::mutex> g(P.lock);
            if (P.pinned.empty()) break;
            k = P.pinned.back();
            P.pinned.pop_back();
        }
        if (allocation_id(k.p) == k.id) return k.p;
    }
    void *p = nullptr;
    // portable: readable and writable from every device
    return hipHostMalloc(&p, kPinnedBytes, hipHostMallocPortable) == hipSuccess ? p : nullptr;
}

void pinned_give(void *p, bool idle)
{
    if (!p) return;
    Pool &P = pool();
    if (idle) {
        const uint64_t id = allocation_id(p);
        std::lock_guard<std::mutex> g(P.lock);
        if (P.pinned.size() < 16) {
            P.pinned.push_back(Pinned{p, id});
            return;
        }
    }
    (void)hipHostFree(p);
}

}  // namespace asx

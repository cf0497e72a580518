// Device memory of the library: what plans keep and what builders and conversions need for the
// length of a call.  A hipMalloc takes about 0.1 ms and a hipFree, which waits for the device, 0.3 ms:
// six of each made up three quarters of a transpose of 3.6 M elements.  Freed blocks are therefore
// kept and handed out again, per device, up to kPoolMaxBytes and kPoolMaxBlocks; they go back to the
// device when an allocation fails, when a handle of the generic API is destroyed and when the caller
// asks (asx_release_cached_memory).  All functions may be called from any thread.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace asx {

constexpr size_t kPoolMaxBytes = (size_t)1 << 30;      // kept per device, all blocks together
constexpr size_t kPoolMaxBlockBytes = (size_t)1 << 29; // larger blocks are not kept
constexpr size_t kPoolMaxBlocks = 64;

// Memory of the current device, at least `bytes`.  `brief`: given back by the end of the call, so a
// kept block of up to four times the size will do; else at most a quarter more.
hipError_t pool_malloc_bytes(void **p, size_t bytes, bool brief);
template <typename P>
hipError_t pool_malloc(P **p, size_t bytes, bool brief)
{
    void *q = nullptr;
    const hipError_t e = pool_malloc_bytes(&q, bytes, brief);
    *p = static_cast<P *>(q);
    return e;
}
// Nothing on the device may still use the block: the caller has synchronised the streams that did,
// or calls pool_wait first.  Null is allowed.
void pool_free(void *p);
// Waits until everything queued on the device that owns p has run (as hipFree does).
void pool_wait(const void *p);
// Back to the device at once (waits as hipFree does).
hipError_t pool_return(void *p);
// Bytes kept on the current device; gives all of them back.
size_t pool_kept_bytes();
void pool_release();

// A few kilobytes of page-locked host memory that kernels and copies of one call write and the host
// reads after it has synchronised the stream; null if there is none to be had.
constexpr size_t kPinnedBytes = 8192;
void *pinned_take();
void pinned_give(void *p);

// Scratch of one call on one stream, handed back when the scope ends: after a wait for the stream
// unless the call has already waited (`idle`).
class Scratch {
public:
    explicit Scratch(hipStream_t s) : s_(s) {}
    ~Scratch()
    {
        if (n_ == 0 && !pinned_) return;
        if (!idle) (void)hipStreamSynchronize(s_);
        for (int i = 0; i < n_; ++i) pool_free(p_[i]);
        pinned_give(pinned_);
    }
    Scratch(const Scratch &) = delete;
    Scratch &operator=(const Scratch &) = delete;
    template <typename P>
    hipError_t take(P **p, size_t bytes)
    {
        if (n_ == kMost) return hipErrorOutOfMemory;
        const hipError_t e = pool_malloc(p, bytes, true);
        if (e == hipSuccess) p_[n_++] = *p;
        return e;
    }
    void *pinned() { return pinned_ ? pinned_ : (pinned_ = pinned_take()); }
    bool idle = false;

private:
    static constexpr int kMost = 8;
    hipStream_t s_;
    void *p_[kMost] = {};
    int n_ = 0;
    void *pinned_ = nullptr;
};

}  // namespace asx

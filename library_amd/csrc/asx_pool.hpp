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
// idle: nothing on the device uses the block any more - the caller has synchronised the streams that did, or pool_wait
// says so - and it may be kept.  Otherwise it goes back through hipFree, which waits by itself, and is never handed out
// again.  Null is allowed.
void pool_free(void *p, bool idle);
// Waits until everything queued on the device that owns p has run (as hipFree does); false where that was refused, for
// instance while a stream is being captured.
bool pool_wait(const void *p);
// Back to the device at once (waits as hipFree does).
hipError_t pool_return(void *p);
// Bytes kept on the current device; gives all of them back.
size_t pool_kept_bytes();
void pool_release();

// A few kilobytes of page-locked host memory that kernels and copies of one call write and the host
// reads after it has synchronised the stream; null if there is none to be had.
constexpr size_t kPinnedBytes = 8192;
void *pinned_take();
void pinned_give(void *p, bool idle);  // idle: as for pool_free

// Scratch of one call on one stream, handed back when the scope ends: after a wait for the stream
// unless the call has already waited (`idle`).  What a refused wait leaves in doubt is not kept.
class Scratch {
public:
    explicit Scratch(hipStream_t s) : s_(s) {}
    ~Scratch()
    {
        if (n_ == 0 && !pinned_) return;
        settle();
        for (int i = 0; i < n_; ++i) pool_free(p_[i], idle);
        pinned_give(pinned_, idle);
    }
    // waits unless the call has; whether nothing queued on the stream is left that could use the scratch
    bool settle()
    {
        if (!idle) idle = hipStreamSynchronize(s_) == hipSuccess;
        return idle;
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

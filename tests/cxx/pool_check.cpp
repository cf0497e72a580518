// The pool of device memory on a HIP that is played here: memory is the host's, streams are always done, and what waits is
// refused while `capturing`; while it is `relaxed`, only a wait for the device as such is, and the capture is lost by it.
// reset() takes every block, as hipDeviceReset does; the next allocations lie at the same addresses.  Usage: pool_check CASE; exit status 0 where the case holds.
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <map>

#include "../../library_amd/csrc/asx_pool.hpp"

namespace {
bool capturing = false, relaxed = false, lost = false;
std::map<void *, uint64_t> device_blocks, host_blocks;  // address: number of the allocation
std::multimap<size_t, void *> lost_blocks;               // by size
std::map<void *, size_t> sizes;
uint64_t allocations = 0;

void *allocate(size_t n, std::map<void *, uint64_t> &blocks)
{
    const auto it = lost_blocks.find(n);
    void *p = it == lost_blocks.end() ? malloc(n) : it->second;
    if (it != lost_blocks.end()) lost_blocks.erase(it);
    sizes[p] = n;
    blocks[p] = ++allocations;
    return p;
}
void reset()
{
    for (auto *blocks : {&device_blocks, &host_blocks}) {
        for (const auto &b : *blocks) lost_blocks.emplace(sizes[b.first], b.first);
        blocks->clear();
    }
}
}  // namespace

extern "C" {
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n)
{
    if (capturing) return *p = nullptr, hipErrorStreamCaptureUnsupported;
    *p = allocate(n, device_blocks);
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    if (capturing) return hipErrorStreamCaptureUnsupported;
    if (!device_blocks.erase(p)) return hipErrorInvalidValue;
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    *p = allocate(n, host_blocks);
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    if (capturing) return hipErrorStreamCaptureUnsupported;
    if (!host_blocks.erase(p)) return hipErrorInvalidValue;
    free(p);
    return hipSuccess;
}
hipError_t hipPointerGetAttribute(void *data, hipPointer_attribute what, hipDeviceptr_t p)
{
    if (what != HIP_POINTER_ATTRIBUTE_BUFFER_ID) return hipErrorInvalidValue;
    for (const auto *blocks : {&device_blocks, &host_blocks})
        if (blocks->count(p)) return memcpy(data, &blocks->at(p), sizeof(uint64_t)), hipSuccess;
    return hipErrorInvalidValue;
}
hipError_t hipDeviceSynchronize()
{
    lost |= relaxed;
    return capturing || relaxed ? hipErrorStreamCaptureUnsupported : hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return capturing ? hipErrorStreamCaptureUnsupported : hipSuccess; }
}

#define CHECK(x)                                               \
    do {                                                       \
        if (!(x)) {                                            \
            printf("%s:%d: %s\n", __FILE__, __LINE__, #x);     \
            exit(1);                                           \
        }                                                      \
    } while (0)

using namespace asx;

static void *block(size_t n, bool brief = false)
{
    void *p = nullptr;
    CHECK(pool_malloc(&p, n, brief) == hipSuccess && p);
    return p;
}

// what is given back after a wait is handed out again
static void kept()
{
    void *a = block(100000);
    CHECK(pool_wait(a));
    pool_free(a, true);
    CHECK(pool_kept_bytes() >= 100000 && block(100000) == a);
}

// what a refused wait leaves in doubt is not
static void refused_wait_of_a_plan()
{
    void *a = block(100000), *b = block(300000);
    capturing = true;
    const bool idle = pool_wait(a);
    CHECK(!idle);
    pool_free(a, idle);
    pool_free(b, idle);
    capturing = false;
    CHECK(pool_kept_bytes() == 0);
    CHECK(block(100000) != a && block(300000) != b);
}
// a capture in relaxed mode survives the wait for a plan's last call
static void relaxed_capture()
{
    void *a = block(100000);
    relaxed = true;
    CHECK(pool_wait(a));
    pool_free(a, true);
    CHECK(!lost && block(100000) == a);
}
static void refused_wait_of_a_call()
{
    void *a = nullptr, *pinned = nullptr;
    {
        Scratch s(nullptr);
        CHECK(s.take(&a, 100000) == hipSuccess);
        pinned = s.pinned();
        CHECK(pinned);
        capturing = true;
    }
    capturing = false;
    CHECK(pool_kept_bytes() == 0);
    CHECK(block(100000, true) != a && pinned_take() != pinned);
}

// after a reset of the device nothing kept is handed out or freed: what lies there now is the caller's
static void device_reset()
{
    void *a = block(100000), *b = block(300000), *c = block(100000);
    pool_free(a, true);
    pool_free(b, true);
    void *pinned = pinned_take();
    pinned_give(pinned, true);
    reset();
    void *mine[2], *my_host;
    CHECK(hipMalloc(&mine[0], sizes[a]) == hipSuccess && hipMalloc(&mine[1], sizes[b]) == hipSuccess);
    CHECK((mine[0] == a || mine[0] == c) && mine[1] == b);
    CHECK(hipHostMalloc(&my_host, sizes[pinned], 0) == hipSuccess && my_host == pinned);
    void *fresh = block(100000);
    CHECK(fresh != mine[0] && device_blocks.count(fresh));
    CHECK(pinned_take() != my_host);
    CHECK(pool_return(c) != hipSuccess || c == fresh);
    pool_release();
    CHECK(device_blocks.count(mine[0]) && device_blocks.count(mine[1]));
}

int main(int argc, char **argv)
{
    const struct {
        const char *name;
        void (*run)();
    } cases[] = {{"kept", kept}, {"refused_wait_of_a_plan", refused_wait_of_a_plan}, {"refused_wait_of_a_call", refused_wait_of_a_call}, {"relaxed_capture", relaxed_capture}, {"device_reset", device_reset}};
    for (const auto &c : cases)
        if (argc == 2 && !strcmp(argv[1], c.name)) return c.run(), 0;
    return 2;
}

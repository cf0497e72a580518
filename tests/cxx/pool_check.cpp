// The pool of device memory on a HIP that is played here: memory is the host's, streams are always done, and what waits is
// refused while `capturing`; while it is `relaxed`, only a wait for the device as such is, and the capture is lost by it.  Usage: pool_check CASE; exit status 0 where the case holds.
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <map>

#include "../../library_amd/csrc/asx_pool.hpp"

namespace {
bool capturing = false, relaxed = false, lost = false;
std::map<void *, size_t> device_blocks, host_blocks;
int frees_refused = 0;
}  // namespace

extern "C" {
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n)
{
    if (capturing) return *p = nullptr, hipErrorStreamCaptureUnsupported;
    *p = malloc(n);
    device_blocks[*p] = n;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    if (capturing) return ++frees_refused, hipErrorStreamCaptureUnsupported;
    if (!device_blocks.erase(p)) return hipErrorInvalidValue;
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    *p = malloc(n);
    host_blocks[*p] = n;
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    if (capturing) return ++frees_refused, hipErrorStreamCaptureUnsupported;
    if (!host_blocks.erase(p)) return hipErrorInvalidValue;
    free(p);
    return hipSuccess;
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

int main(int argc, char **argv)
{
    const struct {
        const char *name;
        void (*run)();
    } cases[] = {{"kept", kept}, {"refused_wait_of_a_plan", refused_wait_of_a_plan}, {"refused_wait_of_a_call", refused_wait_of_a_call}, {"relaxed_capture", relaxed_capture}};
    for (const auto &c : cases)
        if (argc == 2 && !strcmp(argv[1], c.name)) return c.run(), 0;
    return 2;
}

// The engine's memory when there is little of it, on a host model of the HIP
// calls that hand it out: device memory of a given capacity, pinned memory
// that can be had or not, and a last error that stays until it is read.  The
// definitions here take the place of the runtime's in the library.
#include <cstdio>
#include <cstdlib>
#include <map>

#include "engine.h"

static std::map<void *, size_t> live;
static size_t used = 0, cap = (size_t)1 << 30;
static bool pinned = true;
static hipError_t last = hipSuccess;

static hipError_t set(hipError_t e) {
    if (e != hipSuccess) last = e;
    return e;
}
static hipError_t give(void **p, size_t n, bool ok) {
    if (!ok) return set(hipErrorOutOfMemory);
    *p = malloc(n);
    live[*p] = n;
    used += n;
    return hipSuccess;
}
static hipError_t take(void *p) {
    if (!p) return hipSuccess;
    if (!live.count(p)) abort();
    used -= live[p];
    live.erase(p);
    free(p);
    return hipSuccess;
}
extern "C" {
hipError_t hipMalloc(void **p, size_t n) { return give(p, n, used + n <= cap); }
hipError_t hipFree(void *p) { return take(p); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return give(p, n, pinned); }
hipError_t hipHostFree(void *p) { return take(p); }
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipMemGetInfo(size_t *f, size_t *t) {
    *f = cap - used;
    *t = cap;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipGetDevice(int *d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
}

static int bad = 0;
#define CHECK(c)                                    \
    do {                                            \
        if (!(c)) {                                 \
            printf("line %d: %s\n", __LINE__, #c);  \
            bad++;                                  \
        }                                           \
    } while (0)

int main() {
    {
        // no pinned memory: a small copy goes from the caller's, and the
        // checks after the next launches find no error of it
        pxa::Engine e;
        pinned = false;
        CHECK(e.small_block(100) == nullptr);
        CHECK(hipGetLastError() == hipSuccess);
        CHECK(e.last_error().empty());
        // where it can't be done without, the caller is told
        CHECK(e.host_block(100) == nullptr);
        CHECK(hipGetLastError() == hipSuccess);
        CHECK(!e.last_error().empty());
        pinned = true;
        void *p = e.small_block(100);
        CHECK(p != nullptr);
        CHECK(e.small_block(pxa::Engine::SMALL_COPY) == p);
        CHECK(e.small_block(pxa::Engine::SMALL_COPY + 1) == nullptr);
    }
    {
        // wide sweeps give way to another allocation
        pxa::Engine e;
        CHECK(e.reserve_sweep(1) == 0);
        const int64_t base = e.device_bytes();
        CHECK(base > 0);
        CHECK(e.reserve_sweep(pxa::Engine::SWEEP_COLS) == 0 && e.device_bytes() == base);
        e.keep_sweep = true;
        CHECK(e.reserve_sweep(100) == 0 && e.device_bytes() == base);
        e.keep_sweep = false;
        CHECK(e.reserve_sweep(100) == 0);
        const int64_t wide = e.device_bytes();
        CHECK(wide == 2 * base);
        cap = used + 100;
        void *p = e.alloc(200);
        CHECK(p != nullptr && e.device_bytes() == base + 200);
        CHECK(e.last_error().empty() && hipGetLastError() == hipSuccess);
        // no room for them any more, and an error only where nothing can give way
        cap = used + 3 * pxa::LOAD_PAD;
        CHECK(e.reserve_sweep(100) == 0 && e.device_bytes() == base + 200);
        CHECK(e.alloc(1000) == nullptr && !e.last_error().empty() && hipGetLastError() == hipSuccess);
        e.release(p);
        cap = (size_t)1 << 30;
        CHECK(e.reserve_sweep(100) == 0 && e.device_bytes() == wide);
    }
    CHECK(live.empty());
    printf("%d failures\n", bad);
    return bad != 0;
}

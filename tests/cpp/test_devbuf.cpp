// DevBuf::reserve on the host: the runtime calls it makes are stubs over host
// memory, so that what a growth copies can be seen without a GPU.
#include <cstdio>
#include <cstdlib>

#include "../../extensions-photonmapping_amd/csrc/pm_internal.h"

static size_t g_held = 0, g_copied = 0;   // bytes of the last buffer copied from, and of the copy
static size_t size_of(const void *p) { return reinterpret_cast<const size_t *>(p)[-2]; }

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
    size_t *q = static_cast<size_t *>(std::malloc(n + 16));
    q[0] = n;
    *p = q + 2;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    std::free(static_cast<size_t *>(p) - 2);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    g_held = size_of(s);
    g_copied = n;
    std::memcpy(d, s, n < g_held ? n : g_held);
    return hipSuccess;
}
hipError_t hipHostFree(void *) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }
}

int main() {
    pmkd::DevBuf<int> b;
    b.reserve(300, nullptr, 0);
    const size_t cap = b.cap;
    b.reserve(cap, nullptr, 5 * cap);          // fits: nothing is copied
    if (b.cap != cap || g_copied) return std::printf("a buffer that fits was copied\n"), 1;
    b.ptr[cap - 1] = 7;
    b.reserve(cap + 1, nullptr, cap);          // all of it kept
    if (g_copied != cap * sizeof(int) || b.ptr[cap - 1] != 7) return std::printf("contents lost\n"), 1;
    const size_t now = b.cap;
    try {
        b.reserve(4 * now, nullptr, now + 1);  // more than it holds
        return std::printf("copied %zu bytes out of %zu\n", g_copied, g_held), 1;
    } catch (const pmkd::Error &e) {
        if (e.code != PM_ERR_INTERNAL || b.cap != now) return std::printf("wrong error\n"), 1;
    }
    std::printf("DevBuf OK\n");
    return 0;
}

// pm_static.hip -- the scratch of the allocation-free trace (pm_trace_noalloc).
//
// Callers that cannot allocate device memory (code under HIP graph capture,
// tight serving loops) trace through pm_trace_noalloc, whose kernels keep
// their scratch -- the tracers' work counter; the coherent ray order is not
// used at the sizes it takes -- in the file-scope device variable below instead
// of context buffers.  It lives in the code object, so every GPU the library
// runs on holds its own copy until the process ends; its address on a device is
// looked up once, with that device current, and kept per device.  In host code
// `work_counter` names a host-side stand-in, never the device memory: only the
// looked-up pointers are passed to kernels.  Every call on a GPU shares that
// GPU's counter: calls that overlap on one GPU (two streams, two threads) race.
#include <mutex>

#include "pm_internal.h"

namespace pmkd {

namespace {

static __device__ __align__(256) int work_counter;

constexpr int MAX_DEVICES = 64;
std::mutex g_lock;
int *g_work[MAX_DEVICES] = {};

}  // namespace

int *static_work(int device) {
    if (device < 0 || device >= MAX_DEVICES) throw Error{PM_ERR_ARG, "device index out of range"};
    std::lock_guard<std::mutex> lk(g_lock);
    if (!g_work[device]) {
        int *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(reinterpret_cast<void **>(&p), HIP_SYMBOL(work_counter));
        if (e != hipSuccess || !p)
            throw Error{PM_ERR_HIP, std::string("hipGetSymbolAddress(work_counter): ") + hipGetErrorString(e)};
        g_work[device] = p;
    }
    return g_work[device];
}

}  // namespace pmkd

// The device array of puter_hip_matmul_noalloc: a file-scope array, so that no call ever
// allocates it.  It stands in a file, hence a code object, of its own: the runtime loads a
// code object on the first use of anything in it, and a process that never makes the call
// neither holds the array nor waits the 30 ms that loading it takes.  Host code never passes
// the array's name to a kernel (in host code it is a stand-in, not a device address): it
// passes the address hipGetSymbolAddress returns, looked up once per device on that device's
// first call.
#include "common.hpp"

#include <mutex>

namespace puter {

static __device__ __align__(256) char noalloc_array[kNoAllocBytes];   // (zero when loaded)
static std::mutex g_noalloc_mu;
static void *g_noalloc_ptr[64];   // per device: the array's device address

int noalloc_scratch(void **out) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64)
        return fail(PUTER_ERR_UNAVAILABLE, "matmul (no-alloc): no device");
    std::lock_guard<std::mutex> g(g_noalloc_mu);
    if (!g_noalloc_ptr[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(noalloc_array));
        if (e != hipSuccess || !p)
            return fail(PUTER_ERR_UNAVAILABLE, "matmul (no-alloc): scratch address: %s", hipGetErrorString(e));
        g_noalloc_ptr[dev] = p;
    }
    *out = g_noalloc_ptr[dev];
    return PUTER_OK;
}

}  // namespace puter

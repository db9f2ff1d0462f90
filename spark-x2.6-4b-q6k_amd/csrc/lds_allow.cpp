/* lds_allow.cpp — lds_allow.h's one function. A second device asks for
 * itself, and a smaller request that raced a larger one does not take its
 * allowance back. */
#include "lds_allow.h"

#include <mutex>

namespace sparkmv {

int lds_allow(LdsAllowed & a, const void * fn, size_t lds, const char * what) {
    if (lds <= 65536) return 0;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return fail_hip(what, e);
    std::atomic<size_t> * seen = dev >= 0 && dev < 64 ? &a.bytes[dev] : nullptr;
    if (seen && lds <= seen->load()) return 0;
    static std::mutex one;
    std::lock_guard<std::mutex> hold(one);
    if (seen && lds <= seen->load()) return 0;
    e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds);
    if (e != hipSuccess) return fail_hip(what, e);
    if (seen) seen->store(lds);
    return 0;
}

}  // namespace sparkmv

/* lds_allow.h — dynamic LDS above 64 KB has to be allowed to a kernel first,
 * on each device that launches it. A launcher keeps one LdsAllowed per kernel
 * and calls lds_allow before each launch: 0, or -1 with the error set under
 * `what`. */
#pragma once

#include <hip/hip_runtime_api.h>
#include <stddef.h>

#include <atomic>

namespace sparkmv {

int fail_hip(const char * what, hipError_t e);

struct LdsAllowed {
    std::atomic<size_t> bytes[64] = {};   /* by device */
};

int lds_allow(LdsAllowed & a, const void * fn, size_t lds, const char * what);

}  // namespace sparkmv

// device_util.hpp -- what the dispatch rules ask of the device.
#pragma once

#include <hip/hip_runtime.h>

namespace sixi {

// Compute units of the device that is current at the first call; MI355X's 256 where there is none, so
// that sizes can be asked for on any host.
inline int device_cu_count() {
    static int cached = -1;
    if (cached < 0) {
        int dev = 0, n = 0;
        cached = hipGetDevice(&dev) == hipSuccess &&
                         hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0
                     ? n
                     : 256;
    }
    return cached;
}

}  // namespace sixi

// Device helpers shared by the kernel files.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace zk {

// largest j in [0, n) with pre[j] <= x (pre ascending, pre[0] == 0)
__device__ __forceinline__ uint32_t upper_index(const uint64_t* pre, uint32_t n, uint64_t x) {
    uint32_t lo = 0, hi = n;  // invariant: pre[lo] <= x < pre[hi] (pre[n] = inf)
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (pre[mid] <= x) lo = mid;
        else hi = mid;
    }
    return lo;
}

}  // namespace zk

// bounds.h -- the small arithmetic by which a kernel decides what it may leave
// out, apart from the kernels so that a host compiler builds it as well: the
// tests run these functions themselves.
#pragma once

#include <math.h>
#include <stdint.h>

#if defined(__HIPCC__)
#define ATHX_BOTH __host__ __device__ inline
#else
#define ATHX_BOTH static inline
#endif

namespace athx {

// Of the pairs [lo, lo + count) of a tile, the ones below `last`, in records
// of `size` bytes. The count is bounded before it is scaled: a tile may hold
// 2^30 pairs, more than 32 bits hold of their bytes.
ATHX_BOTH uint32_t bytes_below(uint32_t last, uint32_t lo, uint32_t count, uint32_t size) {
    const uint32_t n = last > lo ? last - lo : 0u;
    return (n < count ? n : count) * size;
}

}  // namespace athx

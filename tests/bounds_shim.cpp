// The kernels' bounds (csrc/bounds.h) over arrays, for the tests.
#include "../athenea_amd/csrc/bounds.h"

extern "C" void bytes_below_n(const uint32_t* last, const uint32_t* lo, const uint32_t* count, uint32_t size, uint32_t n,
                              uint32_t* out) {
    for (uint32_t i = 0; i < n; ++i) {
        out[i] = athx::bytes_below(last[i], lo[i], count[i], size);
    }
}

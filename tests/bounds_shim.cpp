// The kernels' bounds (csrc/bounds.h) over arrays, for the tests.
#include "../athenea_amd/csrc/bounds.h"

extern "C" void bytes_below_n(const uint32_t* last, const uint32_t* lo, const uint32_t* count, uint32_t size, uint32_t n,
                              uint32_t* out) {
    for (uint32_t i = 0; i < n; ++i) {
        out[i] = athx::bytes_below(last[i], lo[i], count[i], size);
    }
}

extern "C" void apart_n(const float* a, const float* b, const float* c, const float* cutoff, const float* cx,
                        const float* cy, uint32_t T, uint32_t W, uint32_t H, const uint32_t* x0, const uint32_t* y0,
                        const uint32_t* w, const uint32_t* h, const uint32_t* tx, const uint32_t* ty, uint32_t n,
                        uint8_t* out) {
    for (uint32_t i = 0; i < n; ++i) {
        const athx::AxisReach r = athx::axis_reach(a[i], b[i], c[i], cutoff[i], cx[i], cy[i], T, W, H, x0[i], y0[i],
                                                   w[i], h[i]);
        out[i] = athx::apart(r, cx[i], cy[i], T, tx[i], ty[i]);
    }
}

// The kernels' bounds (csrc/bounds.h) over arrays, for the tests.
#include "../athenea_amd/csrc/bounds.h"

extern "C" void bytes_below_n(const uint32_t* last, const uint32_t* lo, const uint32_t* count, uint32_t size,
                              uint32_t n, uint32_t* out) {
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

extern "C" void columns_meeting_n(const float* xa, const float* xb, const float* cx, const float* margin, uint32_t T,
                                  const uint32_t* W, const uint32_t* tx0, const uint32_t* c0, const uint32_t* c1,
                                  uint32_t n, uint32_t* out) {
    for (uint32_t i = 0; i < n; ++i) {
        out[i] = athx::columns_meeting(xa[i], xb[i], cx[i], margin[i], T, W[i], tx0[i], c0[i], c1[i]);
    }
}

struct Footprint {
    float cx, a, b, c, ia, ic, cutoff;
};

// The columns surely touched, and those left to the float test in the upper half.
extern "C" void decide_columns_n(const float* a, const float* b, const float* c, const float* cutoff, const float* cx,
                                 const float* ylo, const float* yhi, uint32_t T, uint32_t W, const uint32_t* tx0,
                                 const uint32_t* c0, const uint32_t* c1, uint32_t n, uint32_t* out) {
    for (uint32_t i = 0; i < n; ++i) {
        const Footprint g{cx[i], a[i], b[i], c[i], 1.0f / a[i], 1.0f / c[i], cutoff[i]};
        const athx::Decided d = athx::decide_columns(g, athx::slice_terms(a[i], b[i], c[i]), ylo[i], yhi[i], T, W,
                                                     tx0[i], c0[i], c1[i]);
        out[i] = d.sure | d.test << 16;
    }
}

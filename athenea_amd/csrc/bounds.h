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

// v_rcp_f32 and its like, within an ulp; a host build's quotient.
ATHX_BOTH float approx_rcp(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rcpf(x);
#else
    return 1.0f / x;
#endif
}
ATHX_BOTH float approx_sqrt(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_sqrtf(x);
#else
    return sqrtf(x);
#endif
}
ATHX_BOTH float approx_rsqrt(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rsqf(x);
#else
    return 1.0f / sqrtf(x);
#endif
}

// The median of x, lo and hi (x clamped, lo <= hi).
ATHX_BOTH float median(float x, float lo, float hi) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_fmed3f(x, lo, hi);
#else
    return fmaxf(fminf(x, hi), lo);
#endif
}
// A product of 24-bit factors (a coordinate below 65536 times a tile's side).
ATHX_BOTH uint32_t times24(uint32_t x, uint32_t y) { return (x & 0xFFFFFFu) * (y & 0xFFFFFFu); }

// What a float evaluation of a x^2 + 2 b x y + c y^2 differs from the exact
// power by, in units of M = a X^2 + 2 |b| X Y + c Y^2 with X, Y the largest
// distances from the centre: a few of 2^-24, with a wide margin.
constexpr float kSlack = 256.0f * 0x1p-24f;

// How far from a footprint's axis a tile may lie and still be touched. A long
// thin footprint's rectangle (w x h tiles of T pixels from tile x0, y0) holds
// thousands of tiles that its sliver never comes near. q >= l (u . p)^2 with l
// the conic's larger eigenvalue and u its unit direction, and a tile's |u . p|
// is at least its centre's less what its half sides span: a tile is apart when
// that exceeds the sliver's half width at the power that the float tile test
// may still take for the cut, cutoff + kSlack M over the rectangle. (Where M
// is large -- a sliver of many thousand pixels, or one far off screen -- the
// test does touch tiles that lie pixels beyond the cut, and so the frame draws
// them: 1 % and a hundredth of a pixel beside the half width cover pictures of
// some 2000 pixels a side and no more. The slack also covers a conic whose
// smaller eigenvalue has rounded below zero.) A NaN leaves nothing out.
struct AxisReach {
    float ux, uy, reach;
};

ATHX_BOTH AxisReach axis_reach(float a, float b, float c, float cutoff, float cx, float cy, uint32_t T, uint32_t W,
                               uint32_t H, uint32_t x0, uint32_t y0, uint32_t w, uint32_t h) {
    const float mean = 0.5f * (a + c), half = 0.5f * (a - c);
    const float root = approx_sqrt(half * half + b * b), larger = mean + root;
    const float vx = half >= 0.0f ? half + root : b, vy = half >= 0.0f ? b : root - half;
    const float norm = approx_rsqrt(fmaxf(vx * vx + vy * vy, 1e-30f));
    AxisReach r;
    r.ux = vx * norm;
    r.uy = vy * norm;
    const float left = (float)times24(x0, T) - cx, right = (float)times24(x0 + w, T) - cx;
    const float top = (float)times24(y0, T) - cy, bottom = (float)times24(y0 + h, T) - cy;
    const float X = fmaxf(fabsf(left), fabsf(right)), Y = fmaxf(fabsf(top), fabsf(bottom));
    const float M = a * X * X + 2.0f * fabsf(b) * X * Y + c * Y * Y;
    r.reach = approx_sqrt((1.01f * cutoff + kSlack * M) * approx_rcp(larger)) +
              0.5f * (float)T * (fabsf(r.ux) + fabsf(r.uy)) + 0.01f +
              1e-5f * (fabsf(cx) + fabsf(cy) + (float)(W + H));
    return r;
}

// Tile (tx, ty) lies beyond it.
ATHX_BOTH bool apart(const AxisReach& r, float cx, float cy, uint32_t T, uint32_t tx, uint32_t ty) {
    const float side = 0.5f * (float)T;
    const float px = ((float)times24(tx, T) + side) - cx, py = ((float)times24(ty, T) + side) - cy;
    return fabsf(r.ux * px + r.uy * py) > r.reach;
}

// Deciding most of an entry's tiles without the float tile test. The test
// (box_hit) evaluates a x^2 + 2 b x y + c y^2 at points of the tile's box
// whose coordinates are the box edges rounded relative to the centre, in
// about ten float operations; its result differs from the exact least power
// over the exact box by a few units of 2^-24 M, M = a X^2 + 2 |b| X Y + c Y^2
// with X, Y the box's largest distances from the centre. The exact least
// power over a tile box is at most C exactly when the box's x-range meets
// the x-extent of the ellipse q <= C sliced by the box's row band (the slice
// is convex and spans the band's height). That extent is computed here in
// float, once an entry, at C = cutoff -+ kSlack M: a tile meeting the inner
// one is touched by the float test, a tile missing the outer one is not, and
// only the tiles in between are tested. The extent's own rounding is of the
// same order in power (where its square root is ill-conditioned, at the
// ellipse's top and bottom, the power's x-gradient vanishes), and the
// determinant is taken in FP64, where a thin ellipse's does not cancel;
// kSlack covers both with a wide margin.

// [xa, xb]: the x-extent of {(x, y) : y0 <= y <= y1, q(x, y) <= C}
// (coordinates relative to the centre; sa = sqrt(a / det), sc = sqrt(c /
// det)); false when it is empty.
ATHX_BOTH bool band_extent(float a, float b, float ia, float ic, float det, float sa, float sc, float C,
                           float y0, float y1, float& xa, float& xb) {
    if (!(C > 0.0f)) {
        return false;
    }
    // The ellipse's rows: |y| <= sqrt(a C / det); its widest points (x = -+xg)
    // at y = +-b xg / c.
    const float sC = approx_sqrt(C);
    const float ym = sC * sa, xg = sC * sc;
    const float ya = fmaxf(y0, -ym), yb = fminf(y1, ym);
    if (ya > yb) {
        return false;
    }
    // Right end r(y) = (-b y + sqrt(a C - det y^2)) / a is concave, the left
    // end convex: each is extreme at its widest point's row, clamped to the band.
    const float yr = median((-b * xg) * ic, ya, yb);
    const float yl = median((b * xg) * ic, ya, yb);
    const float aC = a * C;
    xb = (-b * yr + approx_sqrt(fmaxf(aC - det * yr * yr, 0.0f))) * ia;
    xa = (-b * yl - approx_sqrt(fmaxf(aC - det * yl * yl, 0.0f))) * ia;
    return true;
}

// The strip columns c0 .. c1 whose box x-range meets [xa, xb] (relative to
// the centre cx), to within a margin: bit j for column tx0 + j. A column's box
// is [tx T + 0.5, min((tx + 1) T, W) - 0.5] in pixel centres, so the columns run
// from the first whose right edge reaches xa to the last whose left edge is at
// most xb, both found by arithmetic (T is a power of two). The edges and the
// sums round by a few units of 2^-24 (|cx| + W); `margin` is 2^-20 of that, to
// be met by columns that must surely meet the extent (positive) or missed by
// columns that surely do not (negative): a column in between is one the float
// test decides. (Stepping to the exact columns with the edges as the float
// test rounds them took four loops and some 95 of an entry's operations, this
// 20.)
ATHX_BOTH uint32_t columns_meeting(float xa, float xb, float cx, float margin, uint32_t T, uint32_t W,
                                   uint32_t tx0, uint32_t c0, uint32_t c1) {
    const float inv_t = approx_rcp((float)T);
    const float lo = (float)c0, hi = (float)c1;
    const float left = xa + cx, right = xb + cx;
    const float first = median(ceilf((left + (0.5f + margin)) * inv_t - 1.0f), lo, hi + 1.0f);
    const float last = median(floorf((right - (0.5f + margin)) * inv_t), lo - 1.0f, hi);
    // The view's last column may be cut short: its right edge is W - 0.5.
    if (first > last || (margin > 0.0f && left + margin > (float)W - 0.5f)) {
        return 0u;
    }
    const uint32_t f = (uint32_t)(int)first, l = (uint32_t)(int)last;
    return ((2u << (l - f)) - 1u) << (f - tx0);
}

// An entry's strip columns c0 .. c1 (its tile row's first and last pixel
// centres ylo, yhi relative to the centre): the columns surely touched, and
// those the float test must decide.
struct Decided {
    uint32_t sure, test;
};

// A footprint's slice terms: its conic's determinant a c - b^2 (taken in
// FP64, where a thin ellipse's does not cancel, and rounded once),
// sqrt(a / det) and sqrt(c / det); det = 0 marks a conic the extents do
// not handle (not positive definite, or a determinant outside the normal
// float range), whose columns all go to the float test.
struct SliceTerms {
    float det, sa, sc;
};

ATHX_BOTH SliceTerms slice_terms(float a, float b, float c) {
    SliceTerms t{0.0f, 0.0f, 0.0f};
    const double detd = (double)a * (double)c - (double)b * (double)b;
    const float det = (float)detd;
    if (a > 1e-9f && c > 1e-9f && det >= 0x1p-126f && det <= 0x1p126f) {
        const float inv_det = approx_rcp(det);
        t.det = det;
        t.sa = approx_sqrt(a * inv_det);
        t.sc = approx_sqrt(c * inv_det);
    }
    return t;
}

// (Footprint: centre cx, conic a, b, c, ia and ic the reciprocals of a and c,
// cutoff.)
template <typename Footprint>
ATHX_BOTH Decided decide_columns(const Footprint& g, const SliceTerms& S, float ylo, float yhi, uint32_t T,
                                  uint32_t W, uint32_t tx0, uint32_t c0, uint32_t c1) {
    Decided d{0u, 0u};
    if (c1 < c0) {
        return d;
    }
    if (S.det == 0.0f) {
        d.test = ((1u << (c1 - c0 + 1u)) - 1u) << (c0 - tx0);
        return d;
    }
    const uint32_t ex = times24(c1 + 1u, T) < W ? times24(c1 + 1u, T) : W;
    const float X = fmaxf(fabsf(((float)times24(c0, T) + 0.5f) - g.cx), fabsf(((float)(ex - 1u) + 0.5f) - g.cx));
    const float Yb = fmaxf(fabsf(ylo), fabsf(yhi));
    const float slack = kSlack * (g.a * X * X + 2.0f * fabsf(g.b) * X * Yb + g.c * Yb * Yb);
    const float margin = 0x1p-20f * (fabsf(g.cx) + (float)W);
    float xa = 0.0f, xb = 0.0f;
    d.sure = band_extent(g.a, g.b, g.ia, g.ic, S.det, S.sa, S.sc, g.cutoff - slack, ylo, yhi, xa, xb)
                 ? columns_meeting(xa, xb, g.cx, margin, T, W, tx0, c0, c1)
                 : 0u;
    uint32_t maybe = 0u;
    if (band_extent(g.a, g.b, g.ia, g.ic, S.det, S.sa, S.sc, g.cutoff + slack, ylo, yhi, xa, xb)) {
        // (An extent that is not one -- a NaN -- leaves every column to the test.)
        maybe = xa <= xb ? columns_meeting(xa, xb, g.cx, -margin, T, W, tx0, c0, c1)
                         : ((2u << (c1 - c0)) - 1u) << (c0 - tx0);
    }
    d.test = maybe & ~d.sure;
    return d;
}

}  // namespace athx

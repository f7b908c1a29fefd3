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

}  // namespace athx

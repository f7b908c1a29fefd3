"""The settle pass's half-width test for long thin footprints (bounds.h
axis_reach and apart, the kernel's own source built by the host compiler),
against the float tile test. No tile that a footprint touches is ever left out.
Every tile side, pictures with cut last tiles, slivers of any angle and up to
1:1000, centres on and off screen, tiles chosen about the ellipse's edge; then
slivers past the corner of pictures of up to 65 535 pixels, where the float test
touches tiles that lie pixels beyond the cut."""
from __future__ import annotations

import numpy as np
import pytest

from tests import bounds_lib
from tests.test_strip_classify import min_power

f32 = np.float32


def box(tx, ty, cx, cy, T, W, H):
    """A tile's first and last pixel centres relative to the centre."""
    return (((tx * T).astype(f32) + f32(0.5)) - cx, ((ty * T).astype(f32) + f32(0.5)) - cy,
            ((np.minimum((tx + 1) * T, W) - 1).astype(f32) + f32(0.5)) - cx,
            ((np.minimum((ty + 1) * T, H) - 1).astype(f32) + f32(0.5)) - cy)


def tile_rect(a, b, c, cutoff, cx, cy, T, W, H):
    """frame.slang:383-402: (first column, first row, last column, last row), and which are on screen."""
    with np.errstate(all="ignore"):
        det = a * c - b * b
        inv = np.where(det > f32(1e-20), f32(1) / det, f32(0))
        ex, ey = np.sqrt(np.maximum(cutoff * c * inv, f32(0))), np.sqrt(np.maximum(cutoff * a * inv, f32(0)))
        lx, ly, hx, hy = cx - ex, cy - ey, cx + ex, cy + ey
        on = (hx >= 0) & (hy >= 0) & (lx < W) & (ly < H)
        x0, y0 = np.maximum(lx, 0), np.maximum(ly, 0)
        x1, y1 = np.minimum(hx, f32(W) - f32(1)), np.minimum(hy, f32(H) - f32(1))
        r = [(np.where(on, v, 0) // T).astype(np.int64) for v in (x0, y0, x1, y1)]
    return r, on & (r[0] <= r[2]) & (r[1] <= r[3])


def left_out(a, b, c, cutoff, cx, cy, T, W, H, rect, tx, ty):
    u = [v.astype(np.uint32) for v in (rect[0], rect[1], rect[2] - rect[0] + 1, rect[3] - rect[1] + 1, tx, ty)]
    return bounds_lib.call("apart_n", a.size, np.uint8, a, b, c, cutoff, cx, cy, T, W, H, *u).astype(bool)


@pytest.mark.parametrize("T", [8, 16, 32])
@pytest.mark.parametrize("W,H", [(1920, 1080), (641, 359), (13, 7)])
def test_no_touched_tile_is_left_out(T, W, H):
    rng = np.random.default_rng(T + W)
    n = 300000
    sx = np.exp(rng.uniform(np.log(0.3), np.log(600), n))
    sy = sx / np.exp(rng.uniform(0, np.log(1000), n))
    th = rng.uniform(0, np.pi, n)
    ct, st = np.cos(th), np.sin(th)
    va = ct**2 * sx**2 + st**2 * sy**2 + 0.3
    vc = st**2 * sx**2 + ct**2 * sy**2 + 0.3
    vb = ct * st * (sx**2 - sy**2)
    det = va * vc - vb**2
    a, b, c = f32(vc / det), f32(-vb / det), f32(va / det)
    cutoff = rng.uniform(1e-3, 9, n).astype(f32)
    cx, cy = rng.uniform(-0.3, 1.3, n).astype(f32) * f32(W), rng.uniform(-0.3, 1.3, n).astype(f32) * f32(H)

    ph, k = rng.uniform(0, 2 * np.pi, n), rng.uniform(0.8, 1.4, n)
    ex = np.sqrt(va * cutoff) * np.cos(ph) * k
    ey = (vb / np.sqrt(va) * np.cos(ph) + np.sqrt(np.maximum(vc - vb**2 / va, 0)) * np.sin(ph)) * np.sqrt(cutoff) * k
    tx = np.clip(((cx + ex) / T).astype(int), 0, (W + T - 1) // T - 1)
    ty = np.clip(((cy + ey) / T).astype(int), 0, (H + T - 1) // T - 1)
    hit = min_power(a, b, c, *box(tx, ty, cx, cy, T, W, H)) <= cutoff
    rect, on = tile_rect(a, b, c, cutoff, cx, cy, T, W, H)
    on &= (tx >= rect[0]) & (tx <= rect[2]) & (ty >= rect[1]) & (ty <= rect[3])
    apart = left_out(a, b, c, cutoff, cx, cy, T, W, H, rect, tx, ty)
    assert on.any() and not np.any(hit & apart)
    # It does its work: in a large picture most untouched tiles here are left out.
    if W == 1920 and T <= 16:
        assert np.mean(apart[on & ~hit]) > 0.5


@pytest.mark.parametrize("T", [8, 16, 32])
@pytest.mark.parametrize("side", [1920, 4096, 16384, 65535])
def test_long_slivers_past_a_corner(T, side):
    """Slivers as long as a large picture that pass its corner by some pixels.
    The float test's rounding there (a few units of 2^-24 of terms in the
    millions) is worth pixels, and the frame draws what it says: a footprint
    that it touches in a tile at all has a tile left in."""
    rng = np.random.default_rng(T + side)
    n = 400000
    sx, sy = np.exp(rng.uniform(np.log(side / 8), np.log(side * 2), n)), np.exp(rng.uniform(np.log(0.3), np.log(8), n))
    th = 3 * np.pi / 4 + rng.normal(0, 0.2, n)
    ct, st = np.cos(th), np.sin(th)
    va, vc = ct**2 * sx**2 + st**2 * sy**2 + 0.3, st**2 * sx**2 + ct**2 * sy**2 + 0.3
    vb = ct * st * (sx**2 - sy**2)
    # Half the conics from a covariance held in float32, as a projection leaves it.
    short = rng.random(n) < 0.5
    va, vb, vc = (np.where(short, v.astype(f32), v) for v in (va, vb, vc))
    det = np.where(short, va.astype(f32) * vc.astype(f32) - vb.astype(f32) ** 2, va * vc - vb**2)
    ok = det > 1e-12
    a, b, c = (f32(v[ok] / det[ok]) for v in (vc, -vb, va))
    cutoff = rng.uniform(1e-3, 9, n).astype(f32)[ok]
    past = np.sqrt(cutoff * (sy[ok] ** 2 + 0.3)) + rng.uniform(0, 40, a.size)
    along = rng.uniform(-2.5, 2.5, a.size) * sx[ok]
    cx, cy = f32(0.5 - past * st[ok] + along * ct[ok]), f32(0.5 + past * ct[ok] + along * st[ok])
    rect, on = tile_rect(a, b, c, cutoff, cx, cy, T, side, side)
    on &= (rect[0] == 0) & (rect[1] == 0)
    a, b, c, cutoff, cx, cy, *rect = (v[on] for v in (a, b, c, cutoff, cx, cy, *rect))
    touched, left_in = np.zeros(a.size, bool), np.zeros(a.size, bool)
    for tx, ty in np.ndindex(6, 6):
        tile = np.full(a.size, tx), np.full(a.size, ty)
        hit = (min_power(a, b, c, *box(*tile, cx, cy, T, side, side)) <= cutoff) & (rect[2] >= tx) & (rect[3] >= ty)
        touched |= hit
        left_in |= hit & ~left_out(a, b, c, cutoff, cx, cy, T, side, side, rect, *tile)
    assert np.array_equal(touched, left_in)
    if side >= 16384:
        assert touched.any()

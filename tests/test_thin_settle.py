"""The settle pass's half-width test for long thin footprints: float32 in the
kernel's order (project.hip settle_count_kernel), against the float tile test.
No tile that a footprint touches is ever left out. Every tile side, pictures
with cut last tiles, slivers of any angle and up to 1:1000, centres on and off
screen, tiles chosen about the ellipse's edge."""
from __future__ import annotations

import numpy as np
import pytest

from tests.test_strip_classify import min_power

f32 = np.float32


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
    lox, hix = ((tx * T).astype(f32) + f32(0.5)) - cx, ((np.minimum((tx + 1) * T, W) - 1).astype(f32) + f32(0.5)) - cx
    loy, hiy = ((ty * T).astype(f32) + f32(0.5)) - cy, ((np.minimum((ty + 1) * T, H) - 1).astype(f32) + f32(0.5)) - cy
    hit = min_power(a, b, c, lox, loy, hix, hiy) <= cutoff

    mean, half = f32(0.5) * (a + c), f32(0.5) * (a - c)
    root = np.sqrt(half * half + b * b)
    larger = mean + root
    vx, vy = np.where(half >= 0, half + root, b), np.where(half >= 0, b, root - half)
    norm = f32(1) / np.sqrt(np.maximum(vx * vx + vy * vy, f32(1e-30)))
    ux, uy = vx * norm, vy * norm
    side = f32(0.5 * T)
    reach = (np.sqrt(f32(1.01) * cutoff / larger) + side * (np.abs(ux) + np.abs(uy)) + f32(0.01)
             + f32(1e-5) * (np.abs(cx) + np.abs(cy) + f32(W + H)))
    px, py = ((tx * T).astype(f32) + side) - cx, ((ty * T).astype(f32) + side) - cy
    apart = np.abs(ux * px + uy * py) > reach
    assert reach.dtype == np.float32
    assert not np.any(hit & apart)
    # It does its work: in a large picture most untouched tiles here are left out.
    if W == 1920 and T <= 16:
        assert np.mean(apart[~hit]) > 0.5

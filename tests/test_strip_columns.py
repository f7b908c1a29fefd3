"""The strip classifier's columns, found by arithmetic (bounds.h columns_meeting
and decide_columns, the kernels' own source built by the host compiler), against
the edges as the float tile test rounds them and against that test itself. With
its margin a column called sure does meet the extent, and one left out does
not; columns in between go to the float test, and are few. Every tile side,
pictures whose last column is cut, centres far off screen, extents that end
within a unit in the last place of an edge, and slivers across pictures of up
to 65 535 pixels."""
from __future__ import annotations

import numpy as np
import pytest

from tests import bounds_lib
from tests.test_strip_classify import min_power
from tests.test_thin_settle import box, tile_rect

f32 = np.float32


def meets(xa, xb, cx, margin, T, W, column):
    """Whether each column is among those of its own strip that meet its extent."""
    last = (W + T - 1) // T - 1
    tx0 = column // 16 * 16
    args = [v.astype(np.uint32) for v in (W, tx0, tx0, np.minimum(tx0 + 15, last))]
    bits = bounds_lib.call("columns_meeting_n", xa.size, np.uint32, xa, xb, cx, margin, T, *args)
    return (bits >> (column - tx0).astype(np.uint32) & 1).astype(bool)


@pytest.mark.parametrize("T", [8, 16, 32])
def test_columns_within_their_margin(T):
    rng = np.random.default_rng(T)
    n = 400000
    W = rng.integers(1, 4097, n)
    tx = np.minimum(rng.integers(0, 4096 // T, n), (W - 1) // T)
    cx = (rng.uniform(-1, 2, n) * W * rng.choice([1.0, 1.0, 30.0], n)).astype(f32)
    lo = ((tx * T).astype(f32) + f32(0.5)) - cx
    hi = ((np.minimum((tx + 1) * T, W) - 1).astype(f32) + f32(0.5)) - cx
    # Ends near the column's own edges, some exactly on them or a few units off.
    off = rng.choice([0.0, 1e-4, 1e-2, 1.0, 40.0], n) * rng.normal(0, 1, n)
    other = rng.permutation(off)
    xa = (np.where(rng.random(n) < 0.5, hi, lo) + off).astype(f32)
    xb = np.maximum(xa, (np.where(rng.random(n) < 0.5, lo, hi) + other).astype(f32))
    margin = (f32(2.0**-20) * (np.abs(cx) + W.astype(f32))).astype(f32)
    true = (hi >= xa) & (lo <= xb)
    sure = meets(xa, xb, cx, margin, T, W, tx)
    maybe = meets(xa, xb, cx, -margin, T, W, tx)
    assert not np.any(sure & ~true)
    assert not np.any(true & ~maybe)
    # Away from the edges, in a column that is not cut, the margin settles it.
    clear = (np.abs(off) >= 1.0) & (np.abs(other) >= 1.0) & ((tx + 1) * T <= W)
    assert np.mean((maybe & ~sure)[clear]) < 0.01


@pytest.mark.parametrize("T", [8, 16, 32])
@pytest.mark.parametrize("W,H", [(641, 359), (1920, 1080), (16384, 16384), (65535, 65535)])
def test_decided_columns_agree_with_the_float_test(T, W, H):
    rng = np.random.default_rng(T + W)
    n = 500000
    sx = np.exp(rng.uniform(np.log(0.3), np.log(W), n))
    sy = sx / np.exp(rng.uniform(0, np.log(1e5), n))
    th = np.where(rng.random(n) < 0.5, rng.uniform(0, np.pi, n),
                  rng.integers(0, 8, n) * np.pi / 4 + rng.normal(0, 0.02, n))
    ct, st = np.cos(th), np.sin(th)
    va, vc = ct**2 * sx**2 + st**2 * sy**2 + 0.3, st**2 * sx**2 + ct**2 * sy**2 + 0.3
    vb = ct * st * (sx**2 - sy**2)
    # Half the conics from a covariance held in float32, as a projection leaves it.
    short = rng.random(n) < 0.5
    va, vb, vc = (np.where(short, v.astype(f32), v) for v in (va, vb, vc))
    det = np.where(short, va.astype(f32) * vc.astype(f32) - vb.astype(f32) ** 2, va * vc - vb**2)
    ok = det > 1e-12
    a, b, c = (f32(v[ok] / det[ok]) for v in (vc, -vb, va))
    ct, st, sx, sy = (v[ok] for v in (ct, st, sx, sy))
    cutoff = rng.uniform(1e-3, 9, a.size).astype(f32)
    cx, cy = (rng.uniform(-0.3, 1.3, a.size) * W).astype(f32), (rng.uniform(-0.3, 1.3, a.size) * H).astype(f32)
    # Tiles about the ellipse's edge, and some pixels beside it.
    ph, k = rng.uniform(0, 2 * np.pi, a.size), rng.uniform(0.8, 1.2, a.size) * np.sqrt(cutoff)
    along, off = k * sx * np.cos(ph), k * sy * np.sin(ph) + rng.normal(0, 1, a.size) * rng.choice([0, 3, 30], a.size)
    x, y = cx + along * ct - off * st, cy + along * st + off * ct
    rect, on = tile_rect(a, b, c, cutoff, cx, cy, T, W, H)
    tx, ty = np.floor(x / T).astype(np.int64), np.floor(y / T).astype(np.int64)
    on &= (tx >= rect[0]) & (tx <= rect[2]) & (ty >= rect[1]) & (ty <= rect[3])
    a, b, c, cutoff, cx, cy, tx, ty, *rect = (v[on] for v in (a, b, c, cutoff, cx, cy, tx, ty, *rect))
    edges = box(tx, ty, cx, cy, T, W, H)
    hit = min_power(a, b, c, *edges) <= cutoff
    tx0 = tx // 16 * 16
    ends = [v.astype(np.uint32) for v in (tx0, np.maximum(tx0, rect[0]), np.minimum(tx0 + 15, rect[2]))]
    bits = bounds_lib.call("decide_columns_n", a.size, np.uint32, a, b, c, cutoff, cx, edges[1], edges[3], T, W, *ends)
    at = (tx - tx0).astype(np.uint32)
    sure, test = (bits >> at & 1).astype(bool), (bits >> 16 >> at & 1).astype(bool)
    assert hit.sum() > 1000 and (~hit).sum() > 1000
    assert not np.any(sure & ~hit), "a sure hit the float test misses"
    assert not np.any(hit & ~sure & ~test), "a sure miss the float test touches"

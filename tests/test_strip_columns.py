"""The strip classifier's columns, found by arithmetic: float32 in the kernel's
order (project.hip columns_meeting), against the edges as the float tile test
rounds them. With its margin a column called sure does meet the extent, and
one left out does not; columns in between go to the float test, and are few.
Every tile side, pictures whose last column is cut, centres far off screen,
extents that end within a unit in the last place of an edge."""
from __future__ import annotations

import numpy as np
import pytest

f32 = np.float32


def meets(xa, xb, cx, margin, T, W, column):
    left, right = (xa + cx).astype(f32), (xb + cx).astype(f32)
    inv_t = f32(1.0) / f32(T)
    first = np.ceil(((left + (f32(0.5) + margin)).astype(f32) * inv_t - f32(1.0)).astype(f32))
    last = np.floor((right - (f32(0.5) + margin)).astype(f32) * inv_t)
    ok = (column >= first) & (column <= last)
    return ok & ~((margin > 0) & ((left + margin).astype(f32) > (W - 0.5).astype(f32)))


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

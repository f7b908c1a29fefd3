"""Where the adjoint's walk of a batch starts, in bytes of its records, for
tiles of up to 2^30 pairs: the exact count of the pairs below the pixel's last,
at most the batch's, whatever lies between them and the first pair."""
from __future__ import annotations

import numpy as np
import pytest

from tests import bounds_lib


@pytest.mark.parametrize("size", [1, 48])
@pytest.mark.parametrize("batch", [32, 56])
def test_bytes_below(batch, size):
    rng = np.random.default_rng(batch + size)
    edges = np.array([0, 1, batch - 1, batch, batch + 1, 2**31 // 48, 2**32 // 48, 2**32 // 48 + 1, 2**30 - 1, 2**30])
    last = np.concatenate([np.repeat(edges, 400), rng.integers(0, 2**30, 200000)]).astype(np.uint32)
    lo = np.minimum(rng.integers(0, 2**30, last.size) * rng.choice([0, 0, 1], last.size), 2**30).astype(np.uint32)
    near = rng.random(last.size) < 0.5
    lo[near] = np.maximum(last[near].astype(np.int64) - rng.integers(-3, 2 * batch, near.sum()), 0).astype(np.uint32)
    count = rng.integers(1, batch + 1, last.size).astype(np.uint32)
    want = np.clip(last.astype(np.int64) - lo.astype(np.int64), 0, count.astype(np.int64)) * size
    got = bounds_lib.call("bytes_below_n", last.size, np.uint32, last, lo, count, size)
    assert np.array_equal(got, want)
    if size == 48:
        # The product taken before the bound wraps among these cases.
        wrapped = np.where(last > lo, (last - lo) * np.uint32(size), 0).astype(np.uint32)
        assert np.any(np.minimum(wrapped, count * size) != want)

"""Sorts on both sides of the sizes at which the route changes: onesweep's
1024-key partitions, its 4096-key ones, and reduce-scan-scatter."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from athenea_amd import TileRasterizer

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def raster():
    r = TileRasterizer(0)
    yield r
    r.close()


@pytest.mark.parametrize("n", [(1 << 18) - 1, 1 << 18, (1 << 18) + 1, (1 << 21) - 1, 1 << 21, (1 << 21) + 77])
@pytest.mark.parametrize("bits", [11, 32])
def test_sort_about_its_routes(raster, n, bits):
    print("sort routes", n, bits, flush=True)
    rng = np.random.default_rng(n + bits)
    keys = rng.integers(0, 1 << bits, n, dtype=np.uint64)
    k, v = torch.from_numpy(keys.view(np.int64)).cuda(), torch.arange(n, dtype=torch.int32, device="cuda")
    raster.sort_pairs(k, v, bits)
    order = np.argsort(keys, kind="stable")
    assert np.array_equal(v.cpu().numpy(), order)
    assert np.array_equal(k.cpu().numpy().view(np.uint64), keys[order])

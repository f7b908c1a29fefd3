"""Autotuner for the two launch shapes the reference fixes: the tile side
(16 in the reference, TileRasterizer.cpp:19; frame.slang:34) and the blend's
LDS batch depth (256, splat_blend.slang:150-155).

It times the frame on the caller's own workload -- the views, the cloud --
once for every tile side and, where the batch reaches the launch, every batch
depth, and returns the fastest as a RenderSettings. The batch reaches it where
pairs are listed and staged: tiles of 8, frames that keep their walk for the
adjoint (``keep_backward``) or have variants (Cryptomatte, trace), frames past
65 536 strips. A plain frame of 16- or 32-pixel tiles is blended straight from
its strip entries in batches of its own, so such a tile side is timed once, its
time stands for every batch, and the caller's own batch is returned (the
contribution passes over the frame's pairs still stage by it; the adjoint has a
batch of its own).

A plain frame and one that keeps its walk run different blends: a training
loop tunes with ``keep_backward``. Results are kept per workload shape
(Gaussian count, view sizes, SH width, kind of frame) for the process's life,
so a render loop pays the search once.

Every candidate draws the same image: a Gaussian that reaches a pixel reaches
its tile by the exact tile test whatever the tile side, and each tile lists
its Gaussians in (depth key, slot) order, so every pixel walks the same
Gaussians in the same order (the GPU parity tests check each shape against
the oracle, and tests/test_gpu_autotune.py the shapes against each other).
"""
from __future__ import annotations

import dataclasses
import time

import torch

from ._lib import AthxError
from .raster import GaussianCloud, RenderSettings, TileRasterizer

TILES = (8, 16, 32)
BATCHES = (32, 64, 128, 256)

_cache: dict[tuple, tuple[RenderSettings, list[dict]]] = {}


def _shape_key(views: list, cloud: GaussianCloud, base: RenderSettings) -> tuple:
    return (cloud.count, int(cloud.sh.shape[1]), str(cloud.sh.dtype),
            tuple((v.width, v.height) for v in views), base.antialias, base.max_sh_degree, base.cryptomatte,
            base.trace)


def _batch_reaches_the_launch(raster: TileRasterizer, s: RenderSettings, keep_backward: bool) -> bool:
    """Whether the last frame, drawn with ``s``, listed its pairs (capi.hip FrameShape::direct)."""
    return (s.tile == 8 or keep_backward or s.cryptomatte or s.trace or raster.frame_info()["strips"] > 65536)


def autotune(raster: TileRasterizer, views: list, cloud: GaussianCloud, base: RenderSettings | None = None,
             tiles=TILES, batches=BATCHES, reps: int = 3, use_cache: bool = True, keep_backward: bool = False
             ) -> tuple[RenderSettings, list[dict]]:
    """Returns (the fastest settings, every candidate's median ms), for plain
    frames or, with ``keep_backward``, for frames that keep their walk for the
    adjoint. A tile
    side whose frame the rasterizer refuses as too large (more pairs than a
    frame holds: small tiles multiply them) is listed with its reason and
    skipped."""
    base = base or RenderSettings()
    key = (_shape_key(views, cloud, base), keep_backward)
    if use_cache and key in _cache:
        return _cache[key]
    table = []
    best = None
    # The caller's batch first: it stands for the others where they are one launch.
    own = base.batch if base.batch in batches else batches[-1]
    order = [own] + [b for b in batches if b != own]
    for tile in tiles:
        targets = None
        rows = {}
        for batch in order:
            s = dataclasses.replace(base, tile=tile, batch=batch, time_stages=False, count_splats=False)
            try:
                # Warm-up, and sizes the scratch.
                targets, _ = raster.render(views, cloud, s, targets, keep_backward=keep_backward)
            except AthxError as e:
                if e.code != "Unsupported":
                    raise
                rows[batch] = {"tile": tile, "batch": batch, "ms": None, "refused": str(e)}
                break
            torch.cuda.synchronize()
            times = []
            for _ in range(reps):
                t0 = time.perf_counter()
                targets, _ = raster.render(views, cloud, s, targets, keep_backward=keep_backward)
                torch.cuda.synchronize()
                times.append((time.perf_counter() - t0) * 1e3)
            ms = sorted(times)[len(times) // 2]
            rows[batch] = {"tile": tile, "batch": batch, "ms": round(ms, 4)}
            if best is None or ms < best[0]:
                best = (ms, s)
            if not _batch_reaches_the_launch(raster, s, keep_backward):
                rows = {b: {"tile": tile, "batch": b, "ms": round(ms, 4)} for b in batches}
                break
        table += [rows[b] for b in batches if b in rows]
    result = (best[1], table)
    if use_cache:
        _cache[key] = result
    return result

"""A differentiable frame's images and the call that drew them go when the last
reference to them does, with no help from the garbage collector: the autograd
node keeps what its adjoint reads, not its own outputs. On the CPU, with a
rasterizer that only hands out targets."""
from __future__ import annotations

import gc
import weakref

import pytest
import torch

from athenea_amd import camera, synthetic
from athenea_amd.autograd import rasterize
from athenea_amd.raster import FrameStats, RenderTargets


class Hollow:
    """Targets without a picture; notes what its adjoint is handed."""

    serial = 0
    handed = None

    def render(self, views, cloud, settings, keep_backward=False):
        self.serial += 1
        targets = [RenderTargets.allocate(v.width, v.height, "cpu", keep_backward) for v in views]
        for k, t in enumerate(targets):
            t.colour.fill_(k + 1.0)
            t.depth.zero_()
            t.frame_serial = self.serial
        return targets, FrameStats()

    def frame_serial(self):
        return self.serial

    def render_backward(self, views, cloud, settings, targets, dl, grads, overwrite=False):
        self.handed = targets
        for t, d in zip(targets, dl):
            assert t.colour.shape == d.shape and t.final_t is not None and t.last is not None
        for g in grads.values():
            g.fill_(1.0)


@pytest.fixture
def no_collector():
    gc.collect()
    gc.disable()
    yield
    gc.enable()


def call(raster):
    cloud = synthetic.make_cloud(5, 1)
    params = [torch.from_numpy(a).requires_grad_(True)
              for a in (cloud.means, cloud.log_scales, cloud.quats, cloud.opacity_logits, cloud.sh)]
    views = [camera.view_for(synthetic.front_camera(), w, 6) for w in (8, 11)]
    return params, *rasterize(*params, views, raster)


@pytest.mark.parametrize("backward", [False, True])
def test_images_go_with_their_last_reference(no_collector, backward):
    raster = Hollow()
    params, colours, depths = call(raster)
    if backward:
        (colours[0].sum() + 2.0 * colours[1].sum()).backward()
        assert all(p.grad is not None for p in params)
        # The adjoint's targets are the frame's: the same memory, the same frame.
        assert [t.frame_serial for t in raster.handed] == [1, 1]
        assert [t.colour.data_ptr() for t in raster.handed] == [c.data_ptr() for c in colours]
        raster.handed = None
    images = [weakref.ref(t) for t in (*colours, *depths)]
    parameter = weakref.ref(params[0])
    del colours, depths, params
    assert [r() for r in images] == [None] * 4
    assert parameter() is None

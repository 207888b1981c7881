"""Calls on two streams that add into one volume gradient.

Entry points that are given every buffer by the caller, and batch plans, are
not ordered with each other; adjoint outputs are accumulated into.  The sum of
concurrent calls is the sum of the same calls one after the other, up to the
order of float additions: a voxel takes one addition a call from the second pass, and
within a call at most some 1000 additions of bricks' sums, each rounding by 2^-24 of
the largest partial sum: 1e-4 of the largest gradient, as for one call.
"""
import math

import numpy as np
import pytest
import torch

from helpers import camera_scene
from gpu_helpers import dev, gpu_inputs, t32
from diffdvr_amd import batch as bt
from diffdvr_amd import pyrenderer as pr

pytestmark = pytest.mark.gpu

CALLS = 12


def concurrent(run, zero):
    """run(k) adds call k's gradient into the tensor that zero() clears and returns; calls alternate streams."""
    ref = None
    for streams in ([torch.cuda.current_stream()] * 2, [torch.cuda.Stream(), torch.cuda.Stream()]):
        g = zero()
        torch.cuda.synchronize()
        for k in range(CALLS):
            with torch.cuda.stream(streams[k % 2]):
                run(k % 2)
        torch.cuda.synchronize()
        if ref is None:
            ref = g.double()
        else:
            assert ref.abs().max() > 0
            assert float((g.double() - ref).abs().max() / ref.abs().max()) <= 1e-4


@pytest.mark.parametrize("preshaded,shape", [(False, (40, 36, 44)), (False, (37, 33, 30)), (True, (24, 26, 22))])
def test_calls_on_two_streams(preshaded, shape):
    W = H = 96
    calls = []
    adj_volume = torch.zeros(4 if preshaded else 1, *shape, device=dev())
    for k in range(2):
        s = camera_scene(np.random.default_rng(60 + k), W, H, tf_mode=1, camera=0, X=shape[0], Y=shape[1], Z=shape[2], step=0.02)
        inp = gpu_inputs(s)
        if preshaded:
            inp.volume = torch.rand(4, *shape, generator=torch.Generator().manual_seed(k)).to(dev())
            inp.volume_filter_mode = pr.VolumeFilterMode.Preshaded
            inp.tf_mode = pr.TFMode.Preshaded
        o = pr.RendererOutputs(torch.empty(1, H, W, 4, device=dev()), torch.empty(1, H, W, dtype=torch.int32, device=dev()))
        kw = {}
        if not preshaded:
            ck = torch.empty(pr.Renderer.checkpoint_buffer_elements(inp, 16), device=dev())
            pr.Renderer.render_forward(inp, o, path="tiled", checkpoint_interval=16, checkpoints=ck)
            kw = dict(method="checkpoint", checkpoint_interval=16, checkpoints=ck)
        else:
            pr.Renderer.render_forward(inp, o)
        a = pr.AdjointOutputs()
        a.has_volume_derivatives = True
        a.adj_volume = adj_volume
        calls.append((inp, o, torch.rand(1, H, W, 4, generator=torch.Generator().manual_seed(9)).to(dev()), a, kw))

    def run(k):
        inp, o, adj, a, kw = calls[k]
        pr.Renderer.render_adjoint(inp, o, adj, a, **kw)

    concurrent(run, lambda: adj_volume.zero_())


@pytest.mark.parametrize("size", [48, 160])
def test_plans_on_two_streams(size):
    """Few rays for the volume (two passes) and many (one pass)."""
    vol = torch.rand(24, 20, 28, generator=torch.Generator().manual_seed(3)).to(dev())
    tf = t32(np.array([[2.0, 1.0]]))
    g = torch.zeros_like(vol)
    plans = []
    for k in range(2):
        vp = pr.Camera.viewport_from_sphere(torch.zeros(1, 3, dtype=torch.float64), torch.full((1, 1), 2.3 + 0.2 * k, dtype=torch.float64),
                                            torch.full((1, 1), 0.4, dtype=torch.float64), torch.full((1, 1), 2.3, dtype=torch.float64),
                                            pr.Orientation.Yp).float().to(dev())[0]
        adj = torch.rand(size, size, 4, generator=torch.Generator().manual_seed(k)).to(dev())
        view = bt.BatchView(volume=0, tf=0, width=size, height=size, camera=vp, fov_y=math.radians(40.0), step=0.02, adj_color=adj)
        plans.append(bt.BatchPlan([bt.BatchVolume(vol, grad=g)], [bt.BatchTf(tf)], [view], tf_mode=0))
    concurrent(lambda k: plans[k].run(zero_gradients=False), lambda: g.zero_())

"""Volume gradients in two passes (density adjoints stored by the reverse walk, corner gradients added
by a second kernel) against the one-pass instances, which render_fused runs.

Both add the same products; only the order of the float sums differs.  A voxel
of these scenes sums at most about 1000 terms, each addition rounding by 6e-8
relative to a partial sum that the largest gradient of the volume bounds in
order of magnitude: 1e-4 of that largest gradient.
"""
import math

import numpy as np
import pytest
import torch

from helpers import camera_scene, to_f32
from gpu_helpers import dev, gpu_inputs, t32
from diffdvr_amd import batch as bt
from diffdvr_amd import pyrenderer as pr

pytestmark = pytest.mark.gpu


def gradient(shape, layout):
    """Zeros whose elements lie z-fastest, x-fastest, padded with an odd offset, or shared over x."""
    B, X, Y, Z = shape
    if layout == "xfast":
        return torch.zeros(B, Z, Y, X, device=dev()).permute(0, 3, 2, 1)
    if layout == "padded":
        return torch.zeros(B, X + 1, Y + 2, Z + 3, device=dev())[:, 1:, 1:-1, 1:-2]
    if layout == "expanded":
        return torch.zeros(B, 1, Y, Z, device=dev()).expand(B, X, Y, Z)
    return torch.zeros(shape, device=dev())


def both(s, grads=("volume",), layout="contiguous", perBatch=False, K=16):
    inp = gpu_inputs(s)
    B = s["ray_start"].shape[0]
    H, W = s["H"], s["W"]
    shape = (B if perBatch else 1,) + tuple(inp.volume.shape[1:])
    target = torch.rand(B, H, W, 4, generator=torch.Generator().manual_seed(5)).to(dev())
    res = []
    for fused in (True, False):
        color = torch.empty(B, H, W, 4, device=dev())
        term = torch.empty(B, H, W, dtype=torch.int32, device=dev())
        o = pr.RendererOutputs(color, term)
        a = pr.AdjointOutputs()
        a.has_volume_derivatives = True
        a.adj_volume = gradient(shape, layout)
        if "tf" in grads:
            a.has_tf_derivatives = True
            a.adj_tf = torch.zeros_like(inp.tf)
        if "camera" in grads:
            a.has_camera_derivatives = True
            a.adj_camera_ray_start = torch.zeros(B, H, W, 3, device=dev())
            a.adj_camera_ray_dir = torch.zeros(B, H, W, 3, device=dev())
        if fused:
            pr.Renderer.render_fused(inp, o, "l2", target, a, scale=1.0, checkpoint_interval=K)
        else:
            ck = torch.empty(pr.Renderer.checkpoint_buffer_elements(inp, K), device=dev())
            pr.Renderer.render_forward(inp, o, path="tiled", checkpoint_interval=K, checkpoints=ck)
            pr.Renderer.render_adjoint(inp, o, 2 * (color - target), a, method="checkpoint", checkpoint_interval=K,
                                       checkpoints=ck)
        torch.cuda.synchronize()
        res.append([t.double() for t in (a.adj_volume, *([a.adj_tf] if "tf" in grads else []),
                                         *([a.adj_camera_ray_start] if "camera" in grads else []))])
    for one, two in zip(*res):
        assert one.abs().max() > 0
        e = float((one - two).abs().max() / one.abs().max())
        assert e <= 1e-4, e


@pytest.mark.parametrize("filter,tf_mode,grads,layout,shape", [
    (1, 0, ("volume",), "contiguous", (9, 8, 12)), (1, 1, ("volume", "tf"), "xfast", (7, 5, 11)),
    (1, 2, ("volume", "camera"), "padded", (10, 9, 8)), (1, 3, ("volume", "tf", "camera"), "contiguous", (12, 3, 5)),
    (0, 1, ("volume", "tf"), "padded", (9, 7, 6)), (0, 2, ("volume",), "xfast", (6, 10, 9)),
    (1, 1, ("volume",), "expanded", (5, 6, 7)), (1, 1, ("volume",), "contiguous", (2, 2, 3))])
@pytest.mark.parametrize("W,H,B,perBatch", [(13, 11, 3, True), (13, 11, 3, False), (371, 383, 1, False),
                                            (203, 161, 5, True)])
def test_two_passes_match_one(filter, tf_mode, grads, layout, shape, W, H, B, perBatch):
    rng = np.random.default_rng(100 * tf_mode + W + filter)
    s = camera_scene(rng, W, H, B=B, filter=filter, tf_mode=tf_mode, blend=0, camera=0, X=shape[0], Y=shape[1], Z=shape[2],
                     step=0.02)
    both(s, grads, layout, perBatch)


@pytest.mark.parametrize("W", [24, 400])
def test_rays_longer_than_the_store(W):
    """A direction of length 0.3 has 3.3 times the samples the box bounds."""
    s = camera_scene(np.random.default_rng(9), W, 400, tf_mode=1, camera=0, step=0.05)
    s["ray_dir"] = to_f32(s["ray_dir"] * 0.3)
    s["tf"][..., 3] *= 0.1
    both(s)


def test_groups_of_tiles():
    """6400 tiles of 1735 samples a ray exceed the store: two groups."""
    s = camera_scene(np.random.default_rng(11), 640, 640, tf_mode=0, camera=0, step=0.001)
    s["tf"][..., 0] *= 0.05
    both(s)


def test_plan_groups_of_tiles():
    """One view of 7000 samples a ray sizes the store; 6000 tiles then run in two groups.  A plan per view
    has one group each."""
    d = dev()
    vols = [torch.rand(sh, generator=torch.Generator().manual_seed(k)).to(d) for k, sh in enumerate([(267, 271, 269), (11, 14, 9)])]
    tf = t32(np.array([[0.4, 1.0]]))
    yaw = torch.linspace(2.2, 2.7, 3, dtype=torch.float64).reshape(-1, 1)
    vps = pr.Camera.viewport_from_sphere(torch.zeros(3, 3, dtype=torch.float64), yaw, 0.45 + 0 * yaw, 2.3 + 0 * yaw,
                                         pr.Orientation.Yp).float().to(d)
    sizes = [(500, 411, 0.02, 0), (9, 15, 0.00025, 1), (413, 401, 0.03, 0)]
    rng = np.random.default_rng(3)
    res = []
    adj = [t32(rng.standard_normal((h, w, 4))) for w, h, _, _ in sizes]
    views = [bt.BatchView(volume=v, tf=0, width=w, height=h, camera=vps[k], fov_y=math.radians(40.0), step=st,
                          adj_color=adj[k]) for k, (w, h, st, v) in enumerate(sizes)]
    for parts in ([[v] for v in views], [views]):
        g = [torch.zeros_like(v) for v in vols]
        for part in parts:
            plan = bt.BatchPlan([bt.BatchVolume(v, (-0.5, -0.5, -0.5), (1.0, 1.0, 1.0), gv) for v, gv in zip(vols, g)],
                                [bt.BatchTf(tf)], part, tf_mode=0)
            for _ in range(2):  # gradients add up over runs
                plan.run(zero_gradients=False)
            torch.cuda.synchronize()
        res.append([x.double() for x in g])
    for one, two in zip(*res):
        assert one.abs().max() > 0
        assert float((one - two).abs().max() / one.abs().max()) <= 1e-4


@pytest.mark.parametrize("size", [8, 200])
@pytest.mark.parametrize("filter,tf_mode,grads", [(1, 0, ("volume",)), (1, 2, ("volume", "tf")), (0, 1, ("volume", "tf")),
                                                  (1, 3, ("volume", "tf")), (1, 1, ("volume", "tf", "camera"))])
def test_plan_matches_per_call(size, filter, tf_mode, grads):
    """Few rays for the volume (two passes) and many (one pass) against the per-call kernels."""
    d = dev()
    rng = np.random.default_rng(40 + tf_mode)
    s = camera_scene(rng, size, size, filter=filter, tf_mode=tf_mode, blend=0, camera=2, X=9, Y=11, Z=10, step=0.02, smooth=True)
    target = torch.rand(1, size, size, 4, generator=torch.Generator().manual_seed(6)).to(d)
    inp = gpu_inputs(s)
    a = pr.AdjointOutputs()
    a.has_volume_derivatives = True
    a.adj_volume = torch.zeros_like(inp.volume)
    a.has_tf_derivatives = "tf" in grads
    a.adj_tf = torch.zeros_like(inp.tf)
    o = pr.RendererOutputs(torch.empty(1, size, size, 4, device=d), torch.empty(1, size, size, dtype=torch.int32, device=d))
    pr.Renderer.render_fused(inp, o, "l2", target, a, scale=1.0)
    gv, gt = torch.zeros_like(inp.volume[0]), torch.zeros_like(inp.tf[0])
    view = bt.BatchView(volume=0, tf=0, width=size, height=size, camera=t32(s["cam_matrix"])[0], fov_y=s["fov_y"], step=0.02,
                        adj_color=2 * (o.color[0] - target[0]),
                        camera_grad=torch.zeros(3, 3, device=d) if "camera" in grads else None)
    bt.BatchPlan([bt.BatchVolume(inp.volume[0], tuple(s["box_min"][0]), tuple(s["box_size"][0]), gv)],
                 [bt.BatchTf(inp.tf[0], gt if "tf" in grads else None)], [view], volume_filter_mode=filter, tf_mode=tf_mode).run()
    torch.cuda.synchronize()
    for ref, got in [(a.adj_volume[0], gv)] + ([(a.adj_tf[0], gt)] if "tf" in grads else []):
        assert float((ref - got).abs().max() / ref.abs().max()) <= 1e-4


@pytest.mark.parametrize("W,H,B", [(13, 11, 2), (203, 97, 1)])
@pytest.mark.parametrize("layout,blend,grads", [("contiguous", 0, ("volume",)), ("xfast", 1, ("volume",)),
                                                ("padded", 0, ("volume", "camera")), ("contiguous", 1, ("camera",))])
def test_packed_preshaded(W, H, B, layout, blend, grads):
    """Pre-shaded volumes packed into RGBA against the kernels that gather from the four slices (which a
    gradient shared over x makes the call run)."""
    d = dev()
    rng = np.random.default_rng(W + blend)
    s = camera_scene(rng, W, H, B=B, X=7, Y=6, Z=9, step=0.03)
    s["volume"] = to_f32(rng.uniform(0.1, 0.9, (4, 7, 6, 9)) * np.array([1, 1, 1, 4.0 if blend == 0 else 0.3])[:, None, None, None])
    inp = gpu_inputs(s)
    inp.volume_filter_mode = pr.VolumeFilterMode.Preshaded
    inp.tf_mode = pr.TFMode.Preshaded
    inp.blend_mode = pr.BlendMode(blend)
    adj = torch.randn(B, H, W, 4, generator=torch.Generator().manual_seed(8)).to(d)
    o = pr.RendererOutputs(torch.empty(B, H, W, 4, device=d), torch.empty(B, H, W, dtype=torch.int32, device=d))
    pr.Renderer.render_forward(inp, o)
    res = []
    for lay in ("expanded", layout):
        a = pr.AdjointOutputs()
        a.has_volume_derivatives = "volume" in grads or lay == "expanded"
        a.adj_volume = gradient((4, 7, 6, 9), lay)
        a.has_camera_derivatives = True
        a.adj_camera_ray_start = torch.zeros(B, H, W, 3, device=d)
        a.adj_camera_ray_dir = torch.zeros(B, H, W, 3, device=d)
        pr.Renderer.render_adjoint(inp, o, adj, a)
        torch.cuda.synchronize()
        res.append((a.adj_camera_ray_start, a.adj_camera_ray_dir, a.adj_volume))
    for k in range(2):
        assert float((res[0][k] - res[1][k]).abs().max() / res[0][k].abs().max()) <= 1e-4
    if "volume" in grads:  # the shared gradient is the sum over x
        one, two = res[0][2][:, 0], res[1][2].sum(1)
        assert float((one - two).abs().max() / one.abs().max()) <= 1e-4

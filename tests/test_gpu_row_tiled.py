"""Row kernels (16 lanes a ray) against the tiled kernels (one lane a ray) on the same rays.

A 64 x 64 image rendered alone takes the row kernels; the same image repeated
in a batch above every limit of the rules takes the tiled ones, which each test
asserts.  Sample counts, colours, densities and checkpoints are equal bitwise and
either adjoint reads the other forward's buffers.  Gradients differ by the order of float
sums only: at most 100 terms a ray of relative rounding 6e-8 each, whose errors are
independent over the rays that an entry sums: 1e-5 of the gradient's norm.
"""
import numpy as np
import pytest
import torch

from helpers import camera_scene
from gpu_helpers import dev, gpu_inputs, norm_err, t32
from test_gpu_row import adjoint, render
from diffdvr_amd import pyrenderer as pr

pytestmark = pytest.mark.gpu

W = H = 64
MODES = [(1, 0, 0, 16), (1, 1, 1, 8), (1, 2, 0, 32), (1, 3, 0, 64), (0, 1, 0, 16), (0, 2, 1, 16), (1, 3, 1, 8), (1, 2, 1, 64)]


def scene(filter, tf_mode, blend, step, rows=8):
    rng = np.random.default_rng(3300 + 10 * tf_mode + blend + filter)
    s = camera_scene(rng, W, H, filter=filter, tf_mode=tf_mode, blend=blend, camera=0, smooth=True, X=9, Y=8, Z=10, R=rows,
                     step=step)
    if blend == 1:
        s["tf"][..., 0 if tf_mode == 0 else 3] *= 0.5
    return s, t32(rng.standard_normal((1, H, W, 4)))


def lanes(inp, color, term, adj, grads, scratch=True):
    B = color.shape[0]
    a = pr.AdjointOutputs()
    if "tf" in grads:
        a.has_tf_derivatives = True
        a.adj_tf = torch.empty(B, *inp.tf.shape[1:], device=dev())
    if "volume" in grads:
        a.has_volume_derivatives = True
        a.adj_volume = torch.empty(B, *inp.volume.shape[1:], device=dev())
    if "camera" in grads:
        a.has_camera_derivatives = True
        a.adj_camera_ray_start = a.adj_camera_ray_dir = torch.empty(B, H, W, 3, device=dev())
    if "step" in grads:
        a.has_stepsize_derivatives = True
        a.adj_stepsize = torch.empty(B, H, W, device=dev())
    return pr._n.adjoint_lanes_per_ray(inp, pr.RendererOutputs(color, term), adj, a, scratch)


def check(mode, many_views, grads_list, step, rows=8):
    filter, tf_mode, blend, K = mode
    print(f"case mode={mode} views={many_views}", flush=True)
    s, adj = scene(filter, tf_mode, blend, step, rows)
    few, many = render(s, 1, K), render(s, many_views, K)
    assert pr._n.forward_lanes_per_ray(few[0]) == 16 and pr._n.forward_lanes_per_ray(many[0]) == 1
    assert bool((many[2] == few[2]).all()) and bool((many[1] == few[1]).all())
    bits = lambda t: torch.nan_to_num(t, nan=-1.0)   # not written by either
    for k in (3, 4):
        assert bool((bits(many[k]).reshape(many_views, -1) == bits(few[k])).all())
    # crosswise: buffers of the other forward's contents (the library knows a checkpoint buffer by its address)
    few_x, many_x = [t.clone() for t in few[3:]], [t.clone() for t in many[3:]]
    for r, x in ((few, few_x), (many, many_x)):
        pr.Renderer.render_forward(r[0], pr.RendererOutputs(r[1], r[2]), path="tiled", checkpoint_interval=K,
                                   checkpoints=x[0], densities=x[1])
    for f, fx, m, mx in zip(few[3:], few_x, many[3:], many_x):
        fx.copy_(m[:fx.numel()])
        mx.reshape(many_views, -1).copy_(f.expand(many_views, -1))
    adj_many = adj.expand(many_views, H, W, 4).contiguous()
    for grads in grads_list:
        if filter == 0 and "camera" in grads:
            continue
        assert lanes(*few[:3], adj, grads) == 16 and lanes(*many[:3], adj_many, grads) == 1
        if "tf" in grads:  # no memory for the double sums
            assert lanes(*few[:3], adj, grads, scratch=False) == 1
        for hand_few, hand_many in ((few[3:], many[3:]), (few_x, many_x), ((), ())):
            got = adjoint(*few[:3], adj, grads, K, hand_few)
            want = adjoint(*many[:3], adj_many, grads, K, hand_many)
            for k in want:
                for b in (0, many_views // 2, many_views - 1):
                    e = norm_err(got[k][0].cpu(), want[k][b].cpu())
                    assert e < 1e-5, (grads, k, len(hand_few), b, e)


@pytest.mark.parametrize("mode", MODES)
def test_tf_and_volume_gradients(mode):
    """36 views: 2304 tiles."""
    check(mode, 36, [("tf",), ("volume",), ("tf", "volume"), ("tf", "camera"), ("tf", "volume", "camera", "step")], 0.02)


@pytest.mark.parametrize("tf_mode,rows", [(1, 1024), (2, 819), (3, 682)])
def test_largest_tables(tf_mode, rows):
    """R * C up to 4096: the staged table, the double sums and the chunk tables take up to 100 KB of LDS."""
    check((1, tf_mode, 0, 16), 36, [("tf",), ("tf", "volume"), ("tf", "volume", "camera", "step")], 0.04, rows)


@pytest.mark.parametrize("mode", [m for m in MODES if m[0] == 1])
def test_position_gradients(mode):
    """260 views: 16640 tiles, half-voxel steps."""
    check(mode, 260, [("camera", "step"), ("camera",), ("step",)], 0.07)


@pytest.mark.parametrize("mode,rows", [(m, 8) for m in MODES] + [((1, 1, 0, 16), 1024), ((1, 2, 0, 16), 819), ((1, 3, 0, 16), 682)])
def test_one_pass_and_fused(mode, rows):
    """Volume gradients of the one-pass instances, which fused launches run: the rule is that of a gradient whose
    elements overlap (no second pass)."""
    filter, tf_mode, blend, K = mode
    views = 36
    s, _ = scene(filter, tf_mode, blend, 0.02, rows)
    target = torch.rand(1, H, W, 4, generator=torch.Generator().manual_seed(5)).to(dev())
    res = []
    for B in (1, views):
        sb = dict(s, ray_start=np.repeat(s["ray_start"], B, 0), ray_dir=np.repeat(s["ray_dir"], B, 0))
        inp = gpu_inputs(sb)
        o = pr.RendererOutputs(torch.empty(B, H, W, 4, device=dev()), torch.empty(B, H, W, dtype=torch.int32, device=dev()))
        a = pr.AdjointOutputs()
        a.has_tf_derivatives = a.has_volume_derivatives = True
        a.adj_tf = torch.zeros(B, *inp.tf.shape[1:], device=dev())
        a.adj_volume = torch.zeros(B, 1, *inp.volume.shape[2:], device=dev()).expand(B, *inp.volume.shape[1:])
        tg = target.expand(B, H, W, 4).contiguous()
        assert pr._n.adjoint_lanes_per_ray(inp, o, tg, a, True) == (16 if B == 1 else 1)
        a.adj_volume = torch.zeros(B, *inp.volume.shape[1:], device=dev())
        loss = torch.zeros(1, device=dev())
        pr.Renderer.render_fused(inp, o, "l2", tg, a, loss_out=loss, scale=1.0, checkpoint_interval=K)
        torch.cuda.synchronize()
        res.append((o.color, o.terminationIndex, a.adj_tf, a.adj_volume, float(loss) / B))
    assert bool((res[1][0] == res[0][0]).all()) and bool((res[1][1] == res[0][1]).all())
    for k in (2, 3):
        for b in (0, views - 1):
            assert norm_err(res[0][k][0].cpu(), res[1][k][b].cpu()) < 1e-5
    # shares of rays and waves in float32, doubles beyond (test_gpu_sums.py)
    assert abs(res[0][4] - res[1][4]) <= 30 * 2.0 ** -24 * res[0][4]

"""Sums of one call over all its rays: the fused loss.

The reference is the same sum in doubles over the colours that the call wrote.
A ray's share is formed in float32 (at most 8 roundings of 2^-24 each) and so
are the sums over the rays of a wave (at most 6 more) and the last rounding to the
float32 scalar: 15 * 2^-24 = 9e-7 at worst, whatever the number of rays.  Where
the shares of the workgroups are added in float32, each addition may round by
2^-24 of the sum.
"""
import numpy as np
import pytest
import torch

from helpers import camera_scene
from gpu_helpers import dev, gpu_inputs
from diffdvr_amd import pyrenderer as pr

pytestmark = pytest.mark.gpu

ULP = 2.0 ** -24


def fused_loss(W, H, B, grads, loss, K, step, noalloc, first=0.25):
    s = camera_scene(np.random.default_rng(W + H), W, H, B=B, tf_mode=1, camera=0, step=step)
    inp = gpu_inputs(s)
    color = torch.full((B, H, W, 4), float("nan"), device=dev())
    term = torch.empty(B, H, W, dtype=torch.int32, device=dev())
    target = torch.rand(B, H, W, 4, generator=torch.Generator().manual_seed(1)).to(dev())
    a = pr.AdjointOutputs()
    if "tf" in grads:
        a.has_tf_derivatives = True
        a.adj_tf = torch.zeros_like(inp.tf)
    if "volume" in grads:
        a.has_volume_derivatives = True
        a.adj_volume = torch.zeros_like(inp.volume)
    if "camera" in grads:
        a.has_camera_derivatives = True
        a.adj_camera_ray_start = torch.zeros(B, H, W, 3, device=dev())
        a.adj_camera_ray_dir = torch.zeros(B, H, W, 3, device=dev())
    out = torch.full((1,), first, device=dev())  # the loss is added to it
    fn = pr._n.render_fused_noalloc if noalloc else pr._n.render_fused
    fn(inp, pr.RendererOutputs(color, term), loss, target, a, out, 1.0, K)
    torch.cuda.synchronize()
    d = color.double() - target.double()
    want = first + float((d.abs() if loss == "l1" else d * d).sum())
    return abs(float(out.item()) - want) / want, pr.Renderer.checkpoint_buffer_elements(inp, K)


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("W,H,B,grads,loss", [
    (5, 3, 1, ("tf",), "l2"), (128, 128, 4, ("tf", "volume"), "l2"), (256, 256, 1, ("tf",), "l1"),
    (512, 512, 1, ("volume",), "l2"), (509, 507, 2, ("camera",), "l2"), (1024, 1024, 1, ("camera",), "l1"),
    (1024, 1024, 1, ("tf",), "l2")])
def test_fused_loss(W, H, B, grads, loss, noalloc):
    err, _ = fused_loss(W, H, B, grads, loss, 64, 0.05, noalloc)
    assert err <= 15 * ULP, err


def test_fused_loss_without_room_in_the_static_scratch():
    """Checkpoints that fill the static scratch leave no room for the sums: one float addition a tile."""
    err, need = fused_loss(512, 256, 1, ("camera",), "l2", 8, 1.7378147 / 508, True)
    assert need == pr._n.NOALLOC_SCRATCH_FLOATS
    assert err <= (2048 + 15) * ULP, err

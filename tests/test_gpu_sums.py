"""Sums of one call over all its rays: the fused loss and TF gradients.

The reference of the loss is the same sum in doubles over the colours that the call wrote.
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


def tf_gradient(entry, inp, color, term, adj, target, K, perView):
    B, H, W, _ = color.shape
    a = pr.AdjointOutputs()
    a.has_tf_derivatives = True
    a.adj_tf = torch.zeros(B if perView else 1, *inp.tf.shape[1:], device=dev())
    o = pr.RendererOutputs(color, term)
    if entry == "replay":  # checkpoints in the library's scratch
        pr.Renderer.render_adjoint(inp, o, adj, a, method="checkpoint", checkpoint_interval=K)
    elif entry == "checkpoints":
        ck = torch.empty(pr.Renderer.checkpoint_buffer_elements(inp, K), device=dev())
        pr.Renderer.render_forward(inp, o, path="tiled", checkpoint_interval=K, checkpoints=ck)
        pr.Renderer.render_adjoint(inp, o, adj, a, method="checkpoint", checkpoint_interval=K, checkpoints=ck)
    else:
        fn = pr._n.render_fused_noalloc if entry == "noalloc" else pr._n.render_fused
        fn(inp, o, "l2", target, a, None, 1.0, K)
    torch.cuda.synchronize()
    return a.adj_tf.double()


@pytest.mark.parametrize("entry", ["replay", "checkpoints", "fused", "noalloc"])
@pytest.mark.parametrize("W,H,B,tf_mode,perView", [(128, 128, 1, 1, False), (131, 125, 1, 2, False), (128, 128, 4, 0, False),
                                                   (128, 128, 4, 3, False), (256, 256, 3, 1, True)])
def test_tf_gradient_does_not_depend_on_the_order(W, H, B, tf_mode, perView, entry):
    """The order in which the workgroups add is another each time.  Added in doubles it moves an entry by
    less than the last rounding to float32: two runs differ by 2 * 2^-24 of the entry at most."""
    K = 64
    s = camera_scene(np.random.default_rng(W + H), W, H, B=B, tf_mode=tf_mode, camera=0, step=0.03)
    inp = gpu_inputs(s)
    color = torch.empty(B, H, W, 4, device=dev())
    term = torch.empty(B, H, W, dtype=torch.int32, device=dev())
    pr.Renderer.render_forward(inp, pr.RendererOutputs(color, term))
    g = torch.Generator().manual_seed(2)
    adj, target = (torch.rand(B, H, W, 4, generator=g).to(dev()) for _ in range(2))
    first = tf_gradient(entry, inp, color, term, adj, target, K, perView)
    assert first.abs().max() > 0
    for _ in range(5):
        again = tf_gradient(entry, inp, color, term, adj, target, K, perView)
        assert bool(((again - first).abs() <= 2 * ULP * first.abs()).all()), float(((again - first) / first).abs().nan_to_num().max())

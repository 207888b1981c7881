"""Row kernels (16 lanes a ray) against the FP64 oracle and against the one-ray-per-lane tiled kernels.

Small launches take the row kernels, large ones the tiled kernels.  An 8 x 8
image rendered alone and the same image rendered 4200 times in one batch (more
tiles than any of the limits) therefore run both on the same rays: sample counts,
colours, densities and checkpoints must be equal, gradients may differ by the order of float sums only
(at most 100 terms a ray of relative rounding 6e-8 each, so 1e-5; the
gradients' sums run over 64 rays more).
"""
import numpy as np
import pytest
import torch

from helpers import oracle, camera_scene
from gpu_helpers import gpu_inputs, t32, dev, norm_err, rel_err
from diffdvr_amd import pyrenderer as pr

pytestmark = pytest.mark.gpu

MANY = 4200
GRADS = [("tf",), ("volume",), ("camera", "step"), ("tf", "volume"), ("tf", "camera"), ("tf", "volume", "camera", "step")]


def render(s, B, K):
    s = dict(s, ray_start=np.repeat(s["ray_start"], B, 0), ray_dir=np.repeat(s["ray_dir"], B, 0))
    inp = gpu_inputs(s)
    H, W = s["H"], s["W"]
    color = torch.full((B, H, W, 4), float("nan"), device=dev())
    term = torch.full((B, H, W), -7, dtype=torch.int32, device=dev())
    ck = torch.full((pr.Renderer.checkpoint_buffer_elements(inp, K),), float("nan"), device=dev())
    ds = torch.full((pr.Renderer.density_buffer_elements(inp),), float("nan"), device=dev())
    pr.Renderer.render_forward(inp, pr.RendererOutputs(color, term), path="tiled", checkpoint_interval=K,
                               checkpoints=ck, densities=ds)
    torch.cuda.synchronize()
    return inp, color, term, ck, ds


def adjoint(inp, color, term, adj_color, grads, K, handover):
    """handover: (checkpoints, densities), (checkpoints,) or () (the adjoint replays the forward)."""
    B, H, W, _ = color.shape
    a = pr.AdjointOutputs()
    out = {}
    if "tf" in grads:
        a.has_tf_derivatives = True
        out["tf"] = a.adj_tf = torch.zeros(B, *inp.tf.shape[1:], device=dev())
    if "volume" in grads:
        a.has_volume_derivatives = True
        out["volume"] = a.adj_volume = torch.zeros(B, *inp.volume.shape[1:], device=dev())
    if "camera" in grads:
        a.has_camera_derivatives = True
        out["ray_start"] = a.adj_camera_ray_start = torch.zeros(B, H, W, 3, device=dev())
        out["ray_dir"] = a.adj_camera_ray_dir = torch.zeros(B, H, W, 3, device=dev())
    if "step" in grads:
        a.has_stepsize_derivatives = True
        out["step"] = a.adj_stepsize = torch.zeros(B, H, W, device=dev())
    kw = dict(zip(("checkpoints", "densities"), handover))
    pr.Renderer.render_adjoint(inp, pr.RendererOutputs(color, term), adj_color, a, method="checkpoint",
                               checkpoint_interval=K, **kw)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("filter,tf_mode,blend,K", [(1, 0, 0, 16), (1, 1, 1, 8), (1, 2, 0, 32), (1, 3, 0, 64),
                                                    (0, 1, 0, 16), (0, 2, 1, 16), (1, 3, 1, 8), (1, 2, 1, 64)])
def test_row_and_tiled_agree(filter, tf_mode, blend, K):
    rng = np.random.default_rng(3100 + 10 * tf_mode + blend + filter)
    s = camera_scene(rng, 8, 8, filter=filter, tf_mode=tf_mode, blend=blend, camera=0, smooth=True, X=9, Y=8, Z=10,
                     step=0.02)
    if blend == 1:
        s["tf"][..., 0 if tf_mode == 0 else 3] *= 0.5
    few, many = render(s, 1, K), render(s, MANY, K)
    for b in (0, MANY // 2, MANY - 1):
        assert torch.equal(many[2][b], few[2][0])
        assert torch.equal(many[1][b], few[1][0])
    # both forwards wrote the same densities and transmittances, wherever either wrote one
    for k in (3, 4):
        n = few[k].numel()
        a, b = few[k].reshape(1, -1), many[k].reshape(MANY, n)[:1]
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.nan_to_num(a), torch.nan_to_num(b))
    adj = t32(rng.standard_normal((1, 8, 8, 4)))
    for grads in GRADS:
        if filter == 0 and "camera" in grads:
            continue
        # every kind of handover, crosswise: the row adjoint reads the tiled forward's buffers and its own
        want = adjoint(*many[:3], adj.expand(MANY, 8, 8, 4).contiguous(), grads, K, many[3:])
        for handover in (few[3:], (many[3][:few[3].numel()].clone(),), ()):
            if len(handover) == 1:
                pr.Renderer.render_forward(few[0], pr.RendererOutputs(few[1], few[2]), path="tiled",
                                           checkpoint_interval=K, checkpoints=handover[0])
            got = adjoint(*few[:3], adj, grads, K, handover)
            for k in want:
                e = norm_err(got[k][0].cpu(), want[k][MANY // 2].cpu())
                assert e < 1e-5, (grads, k, len(handover), e)


@pytest.mark.parametrize("W,H,B", [(1, 1, 1), (9, 7, 1), (130, 3, 2), (31, 33, 3)])
def test_row_remainders_match_oracle(W, H, B):
    rng = np.random.default_rng(3200 + W)
    s = camera_scene(rng, W, H, B=B, tf_mode=1, camera=0, smooth=True, X=12, Y=11, Z=10, step=0.011)
    s["tf"][..., 3] *= 4.0   # some rays reach the early-out threshold
    inp, color, term = (gpu_inputs(s), torch.empty(B, H, W, 4, device=dev()),
                        torch.empty(B, H, W, dtype=torch.int32, device=dev()))
    pr.Renderer.render_forward(inp, pr.RendererOutputs(color, term))
    t = term.cpu().numpy()
    c, t_free = oracle.forward(s)
    assert np.mean(t_free == t) >= 0.99 and np.abs(t_free - t).max() <= 1
    c, _ = oracle.forward(s, frozen_term=t)
    assert rel_err(color.double().cpu(), c) < 1e-5
    adj = rng.standard_normal(color.shape)
    want = oracle.adjoint(s, c, t, adj, grads=("tf", "volume", "camera", "step"), method=oracle.EXACT_REPLAY)
    for grads in GRADS:
        got = adjoint(inp, color, term, t32(adj), grads, 16, ())
        for k, g in got.items():
            g = g.double().cpu().numpy()
            if k in ("tf", "volume"):
                g = g.sum(0, keepdims=True)
            assert norm_err(g, want[k]) < 1e-4, (grads, k, norm_err(g, want[k]))

"""Volume gradients in two passes against the FP64 oracle, at the size of their rounding.

The bound is 3 times the error of the oracle's FP32 CPU twin (the same products
in the same precision) and 2e-6 for the sums: a voxel adds up to about 1000 terms,
each rounding by at most 2^-24 of the partial sum, with errors that are independent
of each other (sqrt(1000) * 2^-24 = 1.9e-6).  Packed pre-shaded volumes are compared with
the kernels that gather from the four slices (the same blend inversion): twice that for
the sums and, beside them, the roundings of some 50 samples a ray in another order of
operations, independent over the rays (50 * 2^-24 = 3e-6).
"""
import numpy as np
import pytest
import torch

from helpers import camera_scene, oracle, to_f32
from gpu_helpers import dev, gpu_inputs, norm_err, t32
from diffdvr_amd import pyrenderer as pr

pytestmark = pytest.mark.gpu

SUMS = 2e-6


@pytest.mark.parametrize("filter,tf_mode,blend,W,H,B", [
    (1, 0, 0, 41, 37, 2), (1, 1, 1, 41, 37, 2), (1, 2, 0, 24, 90, 1), (1, 3, 0, 41, 37, 2), (0, 1, 0, 41, 37, 2),
    (0, 2, 1, 130, 20, 1), (1, 1, 0, 290, 250, 1)])
def test_two_passes_match_oracle(filter, tf_mode, blend, W, H, B):
    print(f"case filter={filter} tf_mode={tf_mode} blend={blend} {W}x{H}x{B}", flush=True)
    rng = np.random.default_rng(900 + 10 * tf_mode + blend)
    s = camera_scene(rng, W, H, B=B, filter=filter, tf_mode=tf_mode, blend=blend, camera=0, smooth=True, X=17, Y=13, Z=19,
                     step=0.02)
    if blend == 1:
        s["tf"][..., 0 if tf_mode == 0 else 3] *= 0.5
    inp = gpu_inputs(s)
    color = torch.empty(B, H, W, 4, device=dev())
    term = torch.empty(B, H, W, dtype=torch.int32, device=dev())
    o = pr.RendererOutputs(color, term)
    ck = torch.empty(pr.Renderer.checkpoint_buffer_elements(inp, 16), device=dev())
    pr.Renderer.render_forward(inp, o, path="tiled", checkpoint_interval=16, checkpoints=ck)
    t = term.cpu().numpy()
    # rays with a sample at a kink of the TF or (nearest) between two voxels get no adjoint: FP32 may take the other side
    adj = to_f32(rng.standard_normal(color.shape))
    adj[oracle.kink_census(s, t) > 0] = 0.0
    a = pr.AdjointOutputs()
    a.has_volume_derivatives = True
    a.adj_volume = torch.zeros_like(inp.volume)
    pr.Renderer.render_adjoint(inp, o, t32(adj), a, method="checkpoint", checkpoint_interval=16, checkpoints=ck)
    torch.cuda.synchronize()
    g = {}
    for dtype in (np.float64, np.float32):
        c, _ = oracle.forward(s, dtype=dtype, frozen_term=t)
        g[dtype] = oracle.adjoint(s, c, t, adj, grads=("volume",), dtype=dtype, method=oracle.EXACT_REPLAY)["volume"]
    want = g[np.float64]
    twin, err = norm_err(g[np.float32], want), norm_err(a.adj_volume.double().cpu().numpy(), want)
    print(f"error {err:.1e}, FP32 twin {twin:.1e}")
    assert err <= 3 * twin + SUMS, (err, twin)


@pytest.mark.parametrize("W,H,B,blend", [(13, 11, 2, 0), (203, 97, 1, 1), (61, 67, 3, 0)])
def test_packed_preshaded_rounding(W, H, B, blend):
    d, shape = dev(), (4, 9, 12, 11)
    rng = np.random.default_rng(W)
    s = camera_scene(rng, W, H, B=B, X=9, Y=12, Z=11, step=0.03)
    inp = gpu_inputs(s)
    scale = np.array([1, 1, 1, 2.0 if blend == 0 else 0.3])[:, None, None, None]
    inp.volume = t32(rng.uniform(0.1, 0.9, shape) * scale)
    inp.volume_filter_mode = pr.VolumeFilterMode.Preshaded
    inp.tf_mode = pr.TFMode.Preshaded
    inp.blend_mode = pr.BlendMode(blend)
    adj = torch.randn(B, H, W, 4, generator=torch.Generator().manual_seed(8)).to(d)
    o = pr.RendererOutputs(torch.empty(B, H, W, 4, device=d), torch.empty(B, H, W, dtype=torch.int32, device=d))
    pr.Renderer.render_forward(inp, o)
    res = []
    for memory in (torch.zeros(4, 1, *shape[2:], device=d).expand(shape), torch.zeros(shape, device=d)):
        a = pr.AdjointOutputs()
        a.has_volume_derivatives = True
        a.adj_volume = memory  # shared over x: no packing and no second pass
        pr.Renderer.render_adjoint(inp, o, adj, a)
        torch.cuda.synchronize()
        res.append(a.adj_volume[:, 0].double() if memory.stride(1) == 0 else a.adj_volume.double().sum(1))
    err = norm_err(res[1].cpu(), res[0].cpu())
    print(f"difference {err:.1e}")
    assert err <= 2 * SUMS + 50 * 2.0 ** -24, err

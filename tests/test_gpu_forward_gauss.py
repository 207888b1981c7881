"""Gaussian TF-only forward mode (its own kernel) against the general kernel, which the same entries take
when the step size is traced beside them.

Both evaluate the same recurrences; the Gaussian weight is formed from a
correctly rounded or a reciprocal-based exponent scale (about z * 1e-7 relative,
z < 20) and the sums differ in order over at most 100 samples: 1e-5 of the
largest derivative.
"""
import numpy as np
import pytest
import torch

from helpers import camera_scene
from gpu_helpers import gpu_inputs, dev
from diffdvr_amd import pyrenderer as pr

pytestmark = pytest.mark.gpu


def run(s, index, D, step, strided):
    inp = gpu_inputs(s)
    B, H, W = s["ray_start"].shape[0], s["H"], s["W"]
    fd = pr.ForwardDifferencesSettings()
    fd.has_tf_derivatives = True
    fd.d_tf = torch.as_tensor(index, dtype=torch.int32).reshape(1, *s["tf"].shape[1:]).to(dev())
    if step:
        fd.d_stepsize = D
    fd.D = D + int(step)
    color = torch.full((B, H, W, 4), float("nan"), device=dev())
    term = torch.full((B, H, W), -7, dtype=torch.int32, device=dev())
    if strided:
        g = torch.full((B, H, W, fd.D, 5), float("nan"), device=dev())[..., :4]
    else:
        g = torch.full((B, H, W, fd.D, 4), float("nan"), device=dev())
    pr.Renderer.render_forward_gradients(inp, fd, pr.RendererOutputs(color, term), g)
    torch.cuda.synchronize()
    return color, term, g[:, :, :, :D].double()


@pytest.mark.parametrize("rows,D", [(1, 1), (2, 8), (2, 9), (4, 24), (9, 17)])
@pytest.mark.parametrize("filter,blend,strided", [(1, 0, False), (1, 1, True), (0, 0, True)])
def test_gauss_entries_match_general_kernel(rows, D, filter, blend, strided):
    rng = np.random.default_rng(700 + rows)
    s = camera_scene(rng, 21, 13, B=2, filter=filter, tf_mode=3, blend=blend, camera=0, X=9, Y=8, Z=7, R=rows, step=0.03)
    if blend == 1:
        s["tf"][..., 3] *= 0.3
    index = np.full(rows * 6, -1)  # D of the entries, in any order
    index[rng.permutation(rows * 6)[:D]] = rng.permutation(D)[:min(D, rows * 6)]
    c0, t0, g0 = run(s, index, D, True, strided)
    c1, t1, g1 = run(s, index, D, False, strided)
    assert torch.equal(c0, c1) and torch.equal(t0, t1)
    assert g0.abs().max() > 0
    assert float((g0 - g1).abs().max() / g0.abs().max()) <= 1e-5

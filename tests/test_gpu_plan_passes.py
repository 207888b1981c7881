"""Plans choose one or two passes of the volume gradients; both give the same gradients.

Many close views with short steps take one pass below the density limit too; a plan of one of these views
takes two.  The sum of 12 plans of nine views is compared with one plan of all 108: every plan adds floats once,
so that 12 additions of at most 6e-8 of the partial sums, and the single precision of the samples' adjoints in
another order of operations (1e-6), stay below 1e-5 of the largest gradient.
"""
import math

import pytest
import torch

from diffdvr_amd import batch as bt
from diffdvr_amd import pyrenderer as pr
from gpu_helpers import dev

pytestmark = pytest.mark.gpu

VIEWS, PART, N, SIZE, STEP = 108, 9, 32, 72, 0.04 / 32


@pytest.mark.parametrize("tf_grad", [False, True])
def test_one_and_two_passes_agree(tf_grad):
    d = dev()
    gen = torch.Generator().manual_seed(5)
    vol = torch.rand(N, N, N, generator=gen).to(d)
    tf = torch.tensor([[0.1, 0.5, 0.9, 0.6, 0.0], [0.8, 0.3, 0.2, 1.5, 0.5], [0.3, 0.9, 0.4, 2.0, 1.0]], device=d)
    yaw = torch.linspace(0.1, 6.1, VIEWS, dtype=torch.float64).reshape(-1, 1)
    pitch = torch.linspace(-0.9, 0.9, VIEWS, dtype=torch.float64).reshape(-1, 1)
    vps = pr.Camera.viewport_from_sphere(torch.zeros(VIEWS, 3, dtype=torch.float64), yaw, pitch, 1.9 + 0 * yaw,
                                         pr.Orientation.Yp).float().to(d)
    adj = torch.rand(VIEWS, SIZE, SIZE, 4, generator=gen).to(d)
    views = [bt.BatchView(volume=0, tf=0, width=SIZE, height=SIZE, camera=vps[k], fov_y=math.radians(30.0), step=STEP,
                          adj_color=adj[k]) for k in range(VIEWS)]
    got = []
    for parts, passes in ((range(0, VIEWS, VIEWS), 1), (range(0, VIEWS, PART), 2)):
        g, gt = torch.zeros_like(vol), torch.zeros_like(tf)
        for first in parts:
            part = views[first:first + VIEWS // len(parts)]
            plan = bt.BatchPlan([bt.BatchVolume(vol, grad=g)], [bt.BatchTf(tf, grad=gt if tf_grad else None)], part, tf_mode=2)
            assert plan.volume_passes == passes
            plan.run(zero_gradients=False)
        torch.cuda.synchronize()
        got.append((g.double(), gt.double()))
    (g1, t1), (g2, t2) = got
    print("largest gradient %.3g, off by %.2g of it" % (g1.abs().max(), (g1 - g2).abs().max() / g1.abs().max()), flush=True)
    assert g1.abs().max() > 0
    assert (g1 - g2).abs().max() <= 1e-5 * g1.abs().max()
    assert (t1 - t2).abs().max() <= 1e-5 * t1.abs().max()

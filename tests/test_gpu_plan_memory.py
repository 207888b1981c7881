"""Device memory of batched plans: the optional store of density adjoints comes after what a plan cannot do
without, leaves the larger part of the free memory to others and is no larger than the plan's layout uses."""
import math

import numpy as np
import pytest
import torch

from gpu_helpers import dev, t32
from diffdvr_amd import batch as bt
from diffdvr_amd import pyrenderer as pr

pytestmark = pytest.mark.gpu

GIB = 1 << 30


def make_plan(n, size, views, **kw):
    """Density gradients of an n^3 volume, half-voxel steps."""
    d = dev()
    vol = torch.rand(n, n, n, generator=torch.Generator().manual_seed(3)).to(d)
    grad = torch.zeros_like(vol)
    tf = t32(np.array([[4.0, 1.0]]))
    yaw = torch.linspace(2.2, 2.7, views, dtype=torch.float64).reshape(-1, 1)
    vps = pr.Camera.viewport_from_sphere(torch.zeros(views, 3, dtype=torch.float64), yaw, 0.45 + 0 * yaw, 2.3 + 0 * yaw,
                                         pr.Orientation.Yp).float().to(d)
    adj = torch.rand(size, size, 4, generator=torch.Generator().manual_seed(4)).to(d)
    vs = [bt.BatchView(volume=0, tf=0, width=size, height=size, camera=v, fov_y=math.radians(40.0), step=0.5 / n,
                       adj_color=adj) for v in vps]
    return bt.BatchPlan([bt.BatchVolume(vol, grad=grad)], [bt.BatchTf(tf)], vs, tf_mode=0, **kw), grad


def test_plan_where_memory_is_short():
    """With 6 GiB free a store for all tiles (5.5 GiB) would leave no room for the densities and for others."""
    plan, grad = make_plan(256, 256, 24)
    plan.run()
    want = grad.double()
    del plan, grad
    torch.cuda.empty_cache()
    make_plan(16, 16, 1)[0].run()  # whatever the runtime allocates once
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    hold = torch.empty(torch.cuda.mem_get_info(dev())[0] - 6 * GIB, dtype=torch.uint8, device=dev())
    try:
        plan, grad = make_plan(256, 256, 24)
        free = torch.cuda.mem_get_info(dev())[0]
        plan.run()
        torch.cuda.synchronize()
        # both schemes add the same products in another order (test_gpu_scatter.py): 1e-4 of the largest gradient
        assert float((grad.double() - want).abs().max() / want.abs().max()) <= 1e-4
        assert free >= 4 * GIB, free
    finally:
        del hold
        torch.cuda.empty_cache()


def test_store_follows_the_layout():
    """A plan laid out anew holds what a new plan of these options holds (grid 1: the same checkpoints and
    densities in all of them)."""
    for width in (8, 32, 4):
        plan, _ = make_plan(12, 9, 1, grid=1, wave_width=32)
        plan.set_options(wave_width=width, grid=1)
        fresh, _ = make_plan(12, 9, 1, grid=1, wave_width=width)
        assert plan.workspace_bytes == fresh.workspace_bytes, width


def test_workspace_counts_the_sums_of_a_run():
    """The double sums of the loss and the TF gradients belong to the plan."""
    d = dev()
    bytes_ = []
    for grads in (False, True):
        tf = torch.rand(1000, 4, generator=torch.Generator().manual_seed(1)).to(d)
        view = bt.BatchView(volume=0, tf=0, width=16, height=16, camera=torch.eye(3, device=d), fov_y=0.7, step=0.1,
                            target=torch.zeros(16, 16, 4, device=d))
        plan = bt.BatchPlan([bt.BatchVolume(torch.rand(8, 8, 8, device=d), grad=torch.zeros(8, 8, 8, device=d))],
                            [bt.BatchTf(tf, torch.zeros_like(tf) if grads else None)], [view], loss="l2",
                            loss_out=torch.zeros(1, device=d) if grads else None)
        bytes_.append(plan.workspace_bytes)
    assert bytes_[1] - bytes_[0] >= 8 * (4000 + 1)


def test_passes_of_the_volume_gradients():
    """Two passes up to 5.5 rays a voxel face of the volume (12^3: 144 faces)."""
    for size, passes in ((12, 2), (28, 2), (29, 1), (64, 1)):
        plan, _ = make_plan(12, size, 2)
        assert plan.volume_passes == passes and plan.chunk_slots >= 32
    view = plan.views[0]
    plan = bt.BatchPlan(plan.volumes, plan.tfs, [view], tf_mode=0, forward_only=True)
    assert plan.volume_passes == 0 and plan.chunk_slots == 0

"""The autotuner searches the default grid too: a tuned plan is no slower than an untuned one.

Far rays (one a voxel face) through a volume larger than the L2s run fastest with five workgroups per
CU, the default there: 1.48 ms, against 1.65 ms with four.  Repeated timings differ by 1 %: 3 % are allowed.
"""
import math

import pytest
import torch

from gpu_helpers import dev
from diffdvr_amd import batch as bt
from diffdvr_amd import scenes

pytestmark = pytest.mark.gpu


def median_ms(plan, reps=10):
    times = []
    for _ in range(7):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(reps):
            plan.run()
        b.record()
        torch.cuda.synchronize()
        times.append(a.elapsed_time(b) / reps)
    return sorted(times)[3]


def test_tuned_no_slower_than_default(monkeypatch):
    monkeypatch.setenv("DVR_AUTOTUNE_CACHE", "")
    d = dev()
    g = torch.Generator().manual_seed(1)
    n, size, views = 256, 256, 8
    vol = scenes.blob_volume(n, 16, 3, device=d)[0].contiguous()
    at = torch.tensor([0.0, 0.3, 0.5, 0.7, 1.0])
    tf = torch.cat([torch.rand(5, 4, generator=g), at[:, None]], 1).contiguous().to(d)
    # a golden-angle spiral: no direction of the volume is favoured
    lat = [math.asin(-0.87 + 2.0 * (i + 1) / (views + 1)) for i in range(views)]
    lon = [(i + 1) * math.pi * (3.0 - math.sqrt(5.0)) + 0.4 for i in range(views)]
    vps = scenes.sphere_viewports(lat, lon, 2.5).to(d)
    target = torch.rand(size, size, 4, generator=g).to(d)
    vs = [bt.BatchView(volume=0, tf=0, width=size, height=size, camera=v, fov_y=math.radians(45.0), step=0.5 / n, target=target)
          for v in vps]
    plan = bt.BatchPlan([bt.BatchVolume(vol)], [bt.BatchTf(tf, torch.zeros_like(tf))], vs, tf_mode=2, loss="l2")
    plan.run()
    torch.cuda.synchronize()
    untuned = median_ms(plan)
    chosen = plan.autotune()
    tuned = median_ms(plan)
    print(f"untuned {untuned:.3f} ms, {chosen}: {tuned:.3f} ms")
    assert tuned <= 1.03 * untuned, (untuned, tuned, chosen)

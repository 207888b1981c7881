"""Batched plans whose volume gradients take one pass, against the FP64 oracle.

Plans with few rays for their volumes take two passes (the views of
test_gpu_batched.py among them), which leaves the walk's chunk table out.  The views here are
above the limit of 5.5 rays a voxel face, so the one-pass instances and their table
of double sums run: every TF mode, volume gradients alone, beside TF gradients and beside
camera gradients, and the smallest table, which a 256-row texture leaves.
Bounds as in test_gpu_batched.py.

Rays with a sample within FP32 rounding (2e-5 voxels, as in test_gpu_preshaded.py) of an
interior cell face get no adjoint where camera gradients are compared: the
trilinear position derivative jumps there, and FP32 may place the sample in the
neighbouring cell (the FP32 CPU twin of the oracle then is off by as much as the GPU: 3.7e-4 of
a view's camera gradient from one of its 1333 rays).
"""
import pytest
import torch

import test_gpu_batched as tb
from gpu_helpers import dev, t32
from helpers import oracle

pytestmark = pytest.mark.gpu

# (volume, tf, W, H, step): 6.7 to 9.4 rays a voxel face of 18 x 16 x 20 and 12 x 14 x 10 voxels
VIEWS = [(0, 0, 46, 47, 0.02), (1, 1, 37, 33, 0.03), (0, 1, 61, 38, 0.025), (1, 0, 31, 43, 0.02)]


def run(monkeypatch, seed, filter, tf_mode, blend, grads, twin=False, rows=8, **kw):
    monkeypatch.setattr(tb, "VIEWS", VIEWS)
    case = tb.Case(seed, filter, tf_mode, blend, grads=grads, tf_rows=rows)
    if filter == 1 and "camera" in grads:
        for i, v in enumerate(case.views):
            scene = case.scene(i)
            _, term = oracle.forward(scene)
            case.adj_colors[i][oracle.kink_census(scene, term, eps_face=2e-5)[0] > 0] = 0.0
            v.adj_color = t32(case.adj_colors[i], dev())
    plan = case.plan(**kw)
    assert plan.volume_passes == 1
    plan.run()
    torch.cuda.synchronize()
    tb.check_against_oracle(case, twin_bound=twin)
    return plan


@pytest.mark.parametrize("tf_mode", [0, 1, 2, 3])
@pytest.mark.parametrize("grads", [("volume",), ("tf", "volume"), ("tf", "volume", "camera")])
def test_one_pass_matches_oracle(monkeypatch, tf_mode, grads):
    seed = 7800 + 10 * tf_mode + len(grads)
    print(f"case tf_mode={tf_mode} grads={grads} seed={seed}", flush=True)
    run(monkeypatch, seed, 1, tf_mode, 0, grads)


@pytest.mark.parametrize("filter,blend,K", [(0, 0, 4), (1, 1, 8), (0, 1, 32), (1, 0, 64)])
def test_one_pass_modes(monkeypatch, filter, blend, K):
    print(f"case filter={filter} blend={blend} K={K}", flush=True)
    run(monkeypatch, 7860 + filter, filter, 2, blend, ("tf", "volume", "camera"), checkpoint_interval=K)


def test_one_pass_with_the_smallest_table(monkeypatch):
    """The 256-texel TF amplifies FP32 density rounding: forward within 3x the FP32 CPU twin."""
    plan = run(monkeypatch, 7880, 1, 1, 0, ("tf", "volume"), twin=True, rows=256, checkpoint_interval=8)
    assert plan.chunk_slots == 32

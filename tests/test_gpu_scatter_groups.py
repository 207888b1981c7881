"""Per-call volume gradients in two passes whose density adjoints exceed the call's store: several groups of tiles.

16 x 256 x 256 rays through 160^3 at half-voxel steps are 16384 tiles of up to 576 stored samples, 158 KB a tile: the
2 GiB of the store hold 13 500.  Rays of many samples that lie close together run in one pass (test_gpu_scatter.py).
Against the one-pass instances of render_fused, within the bound given there.
"""
import numpy as np
import pytest

from helpers import camera_scene
from test_gpu_scatter import both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grads,perBatch", [(("volume",), False), (("volume", "tf", "camera"), False)])
def test_groups_of_tiles(grads, perBatch):
    s = camera_scene(np.random.default_rng(21), 256, 256, B=16, tf_mode=2, camera=0, X=160, Y=160, Z=160, step=0.0031)
    s["tf"][..., 3] *= 0.3
    both(s, grads, "contiguous", perBatch)

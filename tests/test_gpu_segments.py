"""One-pass volume plans walk segments of at most eight samples at every checkpoint interval.

Intervals of eight and more, with the density store and re-interpolating, without camera gradients (their
instances walk whole segments, test_gpu_one_pass.py), against the FP64 oracle at the bounds of
test_gpu_batched.py; rays of some tens of samples leave remainders in segments and intervals.
"""
import pytest

from test_gpu_one_pass import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [8, 16, 32, 64])
@pytest.mark.parametrize("tf_mode,store", [(1, True), (2, True), (2, False), (3, False)])
def test_segments_of_one_pass_plans(monkeypatch, K, tf_mode, store):
    print(f"case K={K} tf_mode={tf_mode} store={store}", flush=True)
    run(monkeypatch, 7900 + tf_mode, 1, tf_mode, 0, ("tf", "volume"), checkpoint_interval=K, density_store=store)

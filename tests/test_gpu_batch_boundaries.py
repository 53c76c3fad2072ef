"""Batches whose scene boundaries take 1 to 9 workgroups of the contact kernels (which are filled up to a multiple of
eight), bit for bit against the oracle."""
import pytest

from diploma_thesis_amd import scenes
from test_gpu_crowded_buckets import run_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [2, 8, 9, 10])
def test_batch_vs_oracle(count):
    print(f"batch boundaries: {count} scenes", flush=True)
    run_both([scenes.mix_scene(200100 // count + 31 * k, 20 + k) for k in range(count)])

"""The contact kernels on both sides of the sizes up to which they take 16 lanes a particle, bit for bit against the
oracle: one scattered scene, one dense scene, several scenes, and the reference's layout."""
import numpy as np
import pytest

from diploma_thesis_amd import scenes
from test_gpu_coop_cells import crowd
from test_gpu_crowded_buckets import run_both
from test_gpu_stages import _forces_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [90112, 90113, 131073])
def test_one_scene(n):
    print(f"16 lanes a particle: one scene of {n}", flush=True)
    run_both([scenes.mix_scene(n, 3)])


@pytest.mark.parametrize("n", [131072, 131073])
def test_one_dense_scene(n):
    print(f"16 lanes a particle: one dense scene of {n}", flush=True)
    run_both([crowd(n, 4, 36.0)])


@pytest.mark.parametrize("counts", [(30000, 43725, 3), (30000, 43725, 4), (60000, 130, 70001)])
def test_several_scenes(counts):
    print(f"16 lanes a particle: scenes of {counts}", flush=True)
    run_both([scenes.mix_scene(n, 5 + k) for k, n in enumerate(counts)])


@pytest.mark.parametrize("n", [90112, 90113])
def test_reference_layout(n):
    print(f"16 lanes a particle: reference layout, {n}", flush=True)
    sc = crowd(n, 6, 40.0)
    f, t, v, ref = _forces_case(sc)
    body, st = sc.rb >= 0, ref[np.float32]
    assert np.abs(st.force).max() > 0
    assert np.array_equal(f[body], st.force[body]) and np.array_equal(t[body], st.torque[body])
    assert np.array_equal(v[~body], st.vel[~body])

"""Contacts queued in LDS before they are evaluated, bit for bit against the oracle: more contacts a particle than
the queue holds, cells across the grid's wrap, one scene, several, and the reference's layout."""
import numpy as np
import pytest

from diploma_thesis_amd import capi
from test_gpu_coop_cells import crowd
from test_gpu_crowded_buckets import run_both
from test_gpu_stages import _forces_case

pytestmark = pytest.mark.gpu


# one scene of more particles than 16 lanes each take; 8 to 40 candidates within a diameter; shifted over the wrap
@pytest.mark.parametrize("n,edge,shift", [(196609, 45.0, 0.0), (200001, 30.0, -20.0)])
def test_engine_dense_scene_vs_oracle(n, edge, shift):
    print(f"contact queue: {n} particles in an edge of {edge}", flush=True)
    sc = crowd(n, 3, edge)
    sc.pos[:, :3] += np.float32(shift)
    sc.rb_pos[:, :3] += np.float32(shift)
    run_both([sc])


def test_engine_dense_batch_vs_oracle():
    print("contact queue: batch", flush=True)
    run_both([crowd(n, 80 + k, edge) for k, (n, edge) in enumerate([(99990, 32.0), (77, 2.0), (100003, 30.0)])])


@pytest.mark.parametrize("flags", [0, capi.COMPAT_REF_UNITS | capi.COMPAT_GRAIN_CLAMP])
def test_reference_layout_vs_oracle(flags):
    print(f"contact queue: reference layout, flags={flags}", flush=True)
    sc = crowd(196611, 5, 36.0)
    f, t, v, ref = _forces_case(sc, flags)
    body = sc.rb >= 0
    st = ref[np.float32]
    assert np.abs(st.force).max() > 0
    assert np.array_equal(f[body], st.force[body]) and np.array_equal(t[body], st.torque[body])
    assert np.array_equal(v[~body], st.vel[~body])

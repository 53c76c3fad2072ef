"""The bucket sort by small workgroups (plans whose measured buckets are all small) against the oracle, bit for bit:
scenes of a particle to tens of thousands, batches and forests, and buckets that turn out far fuller than they
were measured (past what a small workgroup sorts in LDS)."""
import numpy as np
import pytest

import oracle
from diploma_thesis_amd import Engine, capi, scenes
from test_gpu_engine import assert_state_equal

pytestmark = pytest.mark.gpu


def run_both(many, steps=2):
    with Engine(many) as e:
        e.step(steps)
        e.sync()
        got = [e.download(k) for k in range(len(many))]
    for k, sc in enumerate(many):
        st = oracle.State(sc, np.float32)
        st.step(steps)
        assert_state_equal(got[k], st, f"scene {k}")


def gathered(n, seed, method):
    """A mixed scene whose bodies are moved together into a few cells, the particles' first positions (which the
    plan measures) left where they were."""
    sc = scenes.mix_scene(n, seed, method).copy()
    rng = np.random.default_rng(seed)
    sc.rb_pos[:, :3] = 10.0 + rng.uniform(0, 1, (sc.b, 3)) * [8.0, 8.0, 1.0]
    return sc


METHODS = [capi.METHOD_GRID, capi.METHOD_LBVH30, capi.METHOD_LBVH63]


@pytest.mark.parametrize("method", METHODS, ids=["grid", "lbvh30", "lbvh63"])
@pytest.mark.parametrize("n", [1, 63, 1025, 16384, 50021])
def test_small_scene_vs_oracle(n, method):
    print(f"small buckets: {n} particles, method {method}", flush=True)
    run_both([scenes.mix_scene(n, 7 + n % 5, method)])


@pytest.mark.parametrize("n", [511, 512, 513, 65536, 65537])
def test_tile_edges_vs_oracle(n):
    print(f"small buckets: {n} particles at the edges of the tiles", flush=True)
    run_both([scenes.mix_scene(n, 9)])


@pytest.mark.parametrize("method", METHODS[:2], ids=["grid", "lbvh30"])
def test_small_batch_vs_oracle(method):
    print(f"small buckets: batch, method {method}", flush=True)
    run_both([scenes.mix_scene(n, 30 + n % 7, method) for n in (1, 2500, 40, 1024, 6000, 3)])


@pytest.mark.parametrize("method", METHODS, ids=["grid", "lbvh30", "lbvh63"])
def test_buckets_fuller_than_measured_vs_oracle(method):
    print(f"small buckets: gathered bodies, method {method}", flush=True)
    sc = gathered(30000, 11, method)
    st = oracle.State(sc, np.float32)
    st.step(1)
    cells = np.floor(st.pos[:, :3]).astype(np.int64) & 63
    assert np.bincount(cells[:, 2] * 4 + cells[:, 1] // 16).max() > 3840   # particles in a bucket of 2^10 cells
    run_both([sc])

"""The grid sort of scenes whose particles crowd into a few buckets, bit for bit against the oracle."""
import numpy as np
import pytest

import oracle
from diploma_thesis_amd import Engine, scenes
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


def slab(n, seed):
    """A mixed scene in a grid of 256^3 cells, its grains in one plane of cells and its cubes across it."""
    sc = scenes.mix_scene(n, seed).copy()
    rng = np.random.default_rng(seed)
    sc.params.gridSize.x = sc.params.gridSize.y = sc.params.gridSize.z = 256
    sc.params.numCells = 256 ** 3
    grains = sc.rb < 0
    sc.pos[grains, :3] = [4.0, 4.0, 8.1] + rng.uniform(0, 1, (int(grains.sum()), 3)) * [56.0, 56.0, 0.8]
    move = ([4.0, 4.0, 8.5] + rng.uniform(0, 1, (sc.b, 3)) * [56.0, 56.0, 0.0] - sc.rb_pos[:, :3]).astype(np.float32)
    sc.rb_pos[:, :3] += move
    sc.pos[~grains, :3] += move[sc.rb[~grains]]
    return sc


# one scene past the sizes and loads at which it is sorted by digit passes, and below; and several
@pytest.mark.parametrize("counts", [(70000,), (20000,), (3000, 20000), (150000, 50000)])
def test_crowded_buckets_vs_oracle(counts):
    print(f"sort of scenes crowded into a plane: {counts}", flush=True)
    run_both([slab(n, 90 + k) for k, n in enumerate(counts)])

"""A plan of small workgroups whose buckets outgrow them: the engine goes over to the large ones after a read or a
synchronize, in the middle of a run of replayed graphs, and the bits stay the oracle's."""
import numpy as np
import pytest

import oracle
from diploma_thesis_amd import Engine, capi, scenes
from test_gpu_engine import assert_state_equal
from test_gpu_small_buckets import METHODS, gathered

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("learn", ["read", "synchronize", "never"])
@pytest.mark.parametrize("method", METHODS, ids=["grid", "lbvh30", "lbvh63"])
def test_outgrown_vs_oracle(method, learn):
    print(f"outgrown buckets: method {method}, {learn}", flush=True)
    sc = gathered(20000, 13, method)
    st = oracle.State(sc, np.float32)
    with Engine(sc) as e:
        for steps in (1, 2, 1):
            e.step(steps)
            if learn == "read":
                e.render_state(0)
            elif learn == "synchronize":
                e.sync()
        st.step(4)
        assert_state_equal(e.download(), st, "outgrown")


@pytest.mark.parametrize("method", METHODS, ids=["grid", "lbvh30", "lbvh63"])
def test_outgrown_then_rebuilt(method):
    print(f"outgrown buckets: rebuild, method {method}", flush=True)
    sc = gathered(20000, 14, method)
    st = oracle.State(sc, np.float32)
    st.step(4)
    with Engine(sc) as e, Engine(gathered(300, 2, method)) as other:
        e.step(1)
        e.sync()
        e.step(1)
        other.rebuild(e, keep=(0,))
        other.step(1)
        other.sync()
        other.step(1)
        assert_state_equal(other.download(), st, "carried")


@pytest.mark.parametrize("method", [capi.METHOD_LBVH30, capi.METHOD_LBVH63], ids=["lbvh30", "lbvh63"])
@pytest.mark.parametrize("n,size", [(30000, 6.0), (3000, 1e-3)], ids=["bucket", "codes"])
def test_overfull_morton_buckets(method, n, size):
    """Bodies that gather in one Morton bucket, or under one 30-bit code, after a scattered start: from the step
    after the read on the codes are sorted by digit passes."""
    print(f"outgrown buckets: {n} particles gather in {size}, method {method}", flush=True)
    sc = scenes.mix_scene(n, 15, method).copy()
    sc.rb_pos[:, :3] = 20.0 + np.random.default_rng(n).uniform(0, size, (sc.b, 3))
    for a in range(3):
        sc.cfg.boxMax[a] = 4096.0
    sc.cfg.wallMask = 0
    grains = sc.rb < 0
    sc.pos[:, :3] = np.random.default_rng(1).uniform(0, 4096.0, (sc.n, 3))   # (the bodies' own are posed from them)
    sc.vel[grains, :3] = 0.0
    st = oracle.State(sc, np.float32)
    with Engine(sc) as e:
        before = [name for name, _ in e.profile()]
        e.step(2)
        e.render_state(0)
        e.step(1)
        e.sync()
        after = [name for name, _ in e.profile()]
        st.step(5)
        assert_state_equal(e.download(), st, "overfull")
    if n == 30000 or method == capi.METHOD_LBVH63:
        assert before != after

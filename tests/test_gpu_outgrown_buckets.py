"""A plan of small workgroups whose buckets outgrow them: the engine goes over to the large ones after a read or a
synchronize, in the middle of a run of replayed graphs, and the bits stay the oracle's."""
import numpy as np
import pytest

import oracle
from diploma_thesis_amd import Engine, capi
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


def test_outgrown_then_rebuilt():
    print("outgrown buckets: rebuild", flush=True)
    sc = gathered(20000, 14, capi.METHOD_GRID)
    st = oracle.State(sc, np.float32)
    st.step(4)
    with Engine(sc) as e, Engine(gathered(300, 2, capi.METHOD_GRID)) as other:
        e.step(1)
        e.sync()
        e.step(1)
        other.rebuild(e, keep=(0,))
        other.step(1)
        other.sync()
        other.step(1)
        assert_state_equal(other.download(), st, "carried")

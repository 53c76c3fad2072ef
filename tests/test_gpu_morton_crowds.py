"""Scenes in a small part of their Morton box, bit for bit against the oracle: on both sides of the bucket size past
which the codes are sorted by digit passes, and 63-bit codes of which many share their upper 30 bits (runs of one to
thousands, a run's first and last position at the array's ends)."""
import numpy as np
import pytest

import oracle
from diploma_thesis_amd import Engine, capi, scenes
from test_gpu_engine import assert_state_equal
from test_gpu_lbvh_packets import check, grains

pytestmark = pytest.mark.gpu


def in_box(sc, factor):
    for a in range(3):
        sc.cfg.boxMax[a] = sc.cfg.boxMax[a] * factor
    sc.cfg.wallMask = 0
    return sc


def cluster(n, method, factor):
    rng = np.random.default_rng(n)
    return in_box(grains(3.0 + rng.uniform(0, 1.4 * n ** (1 / 3), (n, 3)), n, method), factor)


@pytest.mark.parametrize("n", [7168, 7169, 14336, 14337])
@pytest.mark.parametrize("method", [capi.METHOD_LBVH30, capi.METHOD_LBVH63], ids=["lbvh30", "lbvh63"])
def test_one_bucket(n, method):
    print(f"morton crowds: {n} particles in one bucket, method {method}", flush=True)
    check(cluster(n, method, 64))


@pytest.mark.parametrize("n,factor", [(2, 1 << 14), (9, 1 << 14), (256, 1 << 14), (257, 1 << 14), (300, 512), (5000, 256),
                                      (5000, 2048), (66000, 128)])
def test_equal_upper_codes(n, factor):
    print(f"morton crowds: {n} particles, box {factor} times as wide", flush=True)
    sc = cluster(n, capi.METHOD_LBVH63, factor)
    lo, hi = np.array(sc.cfg.boxMin[:]), np.array(sc.cfg.boxMax[:])
    cells = np.unique(np.floor((sc.pos[:, :3] - lo) / (hi - lo) * 1024.0), axis=0, return_counts=True)[1]
    assert cells.max() > (1 if n < 300 else 16)
    check(sc)


def test_forest():
    print("morton crowds: forest", flush=True)
    many = [scenes.mix_scene(3000, 1, capi.METHOD_LBVH30), in_box(scenes.mix_scene(9000, 2, capi.METHOD_LBVH30), 64),
            scenes.mix_scene(500, 3, capi.METHOD_LBVH30)]
    with Engine(many) as e:
        e.step(2)
        e.sync()
        for k, sc in enumerate(many):
            st = oracle.State(sc, np.float32)
            st.step(2)
            assert_state_equal(e.download(k), st, f"scene {k}")

"""The packet traversal of the LBVH contact kernel and the bucket sort of its codes, bit for bit against the oracle: leaf counts around a packet and a
wave, crowds in which every particle reaches every other (the packet's list outgrows what it expands at once, and
candidates are tested in many rounds), leaves that lie on both sides of a split, and packets that hold the leaves of
several small scenes; codes in one tile and many, in tiles of 1,024 and 4,096, in buckets of every width and in one
bucket too large for LDS, alone and in a forest."""
import numpy as np
import pytest

import oracle
from diploma_thesis_amd import Engine, capi, scenes
from test_gpu_engine import assert_state_equal

pytestmark = pytest.mark.gpu


def grains(pos, seed, method):
    """A scene of free grains at the given positions."""
    sc = scenes.mix_scene(1024, 1, method).copy()
    n = len(pos)
    rng = np.random.default_rng(seed)
    sc.pos, sc.vel = np.zeros((n, 4), np.float32), np.zeros((n, 4), np.float32)
    sc.pos[:, :3], sc.vel[:, :3] = pos, rng.normal(size=(n, 3))
    sc.rb, sc.body_frame = np.full(n, -1, np.int32), np.zeros((n, 4), np.float32)
    for k in ("rb_pos", "rb_vel", "rb_ang", "rb_quat"):
        setattr(sc, k, np.zeros((0, 4), np.float32))
    sc.rb_inertia, sc.rb_mass, sc.ppo = np.zeros((0, 9), np.float32), np.zeros(0, np.float32), np.zeros(0, np.int32)
    sc.params.numBodies = 0
    return sc


def crowd(n, seed, method, size=2.0):
    rng = np.random.default_rng(seed)
    return grains(8.0 + rng.uniform(0, size, (n, 3)), seed, method)


def check(sc, steps=2):
    with Engine(sc) as e:
        e.step(steps)
        e.sync()
        g = e.download()
    st = oracle.State(sc, np.float32)
    st.step(steps)
    assert_state_equal(g, st, f"{sc.n} particles")


@pytest.mark.parametrize("method", [capi.METHOD_LBVH30, capi.METHOD_LBVH63])
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 63, 65, 700])
def test_crowd(n, method):
    print(f"lbvh packets: crowd of {n}, method {method}", flush=True)
    check(crowd(n, n, method))


def test_leaves_on_both_sides_of_a_split():
    print("lbvh packets: split leaves", flush=True)
    rng = np.random.default_rng(3)
    mid = 0.5 * float(scenes.mix_scene(1024, 1).cfg.boxMax[0])
    pos = np.concatenate([mid + rng.uniform(-1.5, 1.5, (333, 3)), rng.uniform(1, 2 * mid - 1, (500, 3))])
    check(grains(pos, 3, capi.METHOD_LBVH30))


def test_forest_of_small_scenes():
    print("lbvh packets: forest", flush=True)
    mix = [crowd(n, 50 + n, capi.METHOD_LBVH30, 1.5) for n in (1, 3, 20, 2, 5, 130, 1, 9, 16, 300)]
    with Engine(mix) as e:
        e.step(2)
        e.sync()
        for k, sc in enumerate(mix):
            st = oracle.State(sc, np.float32)
            st.step(2)
            assert_state_equal(e.download(k), st, f"scene {k}")


def packed(n, seed, method, box):
    """n grains, about eight per unit cube, in a corner of a box of the given edge."""
    sc = crowd(n, seed, method, (n / 8.0) ** (1.0 / 3.0))
    sc.cfg.boxMax[:] = [box] * 3
    return sc


@pytest.mark.parametrize("method", [capi.METHOD_LBVH30, capi.METHOD_LBVH63])
@pytest.mark.parametrize("n,box", [(1023, 16.0), (1025, 30.0), (4097, 16.0), (30000, 26.0), (66001, 30.0), (9000, 2000.0)])
def test_code_buckets(n, box, method):
    print(f"lbvh codes: {n} in a box of {box}, method {method}", flush=True)
    check(packed(n, n, method, box), 1)


def test_forest_code_buckets():
    print("lbvh codes: forest", flush=True)
    mix = [packed(n, k, capi.METHOD_LBVH30, box)
           for k, (n, box) in enumerate([(700, 16.0), (6000, 2000.0), (1, 16.0), (3000, 20.0), (12000, 24.0)])]
    with Engine(mix) as e, Engine(mix[:1]) as other:
        e.step(1)
        for k, sc in enumerate(mix):
            st = oracle.State(sc, np.float32)
            st.step(1)
            assert_state_equal(e.download(k), st, f"scene {k}")
        other.rebuild(e, keep=(1, 4, 2), added=[mix[3]])     # the scenes carried over keep their bucket widths
        other.step(1)
        for k, (src, steps) in enumerate([(1, 2), (4, 2), (2, 2), (3, 1)]):
            st = oracle.State(mix[src], np.float32)
            st.step(steps)
            assert_state_equal(other.download(k), st, f"carried {k}")

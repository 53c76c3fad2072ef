"""The 27-cell contact sums formed by 16 lanes per particle, bit for bit against the oracle: particle
counts around the groups of a workgroup, cells with no, a few and hundreds of candidates, and more
hits than a group lists at once."""
import ctypes as C

import numpy as np
import pytest

import oracle
from diploma_thesis_amd import Engine, capi, scenes
from gpu_util import Dev, sync
from test_gpu_engine import assert_state_equal

pytestmark = pytest.mark.gpu
L = capi.lib


@pytest.mark.parametrize("n,points", [(1, 1), (7, 40), (8, 900), (9, 4000), (130, 30000)])
def test_static_contacts_many_candidates(n, points):
    print(f"static contacts: {n} particles, {points} points", flush=True)
    rng = np.random.default_rng(n)
    sc = scenes.mix_scene(max(n, 130), 3)
    st = oracle.State(sc, np.float32)
    r = float(sc.params.particleRadius)
    # the points in a slab of 4 x 1.5 x 4 particle diameters, the first n particles in and around it
    P, N = np.zeros((points, 4), np.float32), np.zeros((points, 4), np.float32)
    P[:, :3] = 10.0 * r + rng.uniform(0, 1, (points, 3)) * [8 * r, 3 * r, 8 * r]
    N[:, :3] = rng.normal(size=(points, 3)) + [0, 2, 0]
    N[:, :3] /= np.linalg.norm(N[:, :3], axis=1, keepdims=True)
    st.pos[:, :3] = 10.0 * r + rng.uniform(-0.3, 1.3, (sc.n, 3)) * [8 * r, 6 * r, 8 * r]
    st.vel[:, :3] = rng.normal(size=(sc.n, 3))
    st.rel[:, :3] = rng.normal(size=(sc.n, 3))
    h, idx = oracle.calc_hash(st.pos, sc.params)
    _, si = oracle.sort_pairs(h, idx)
    s_pos = st.pos[si].copy()
    s_pos[:, 3] = sc.rb[si].view(np.float32)
    s_vel = st.vel[si].copy()
    hs, ids = oracle.calc_hash(P, sc.params)
    shs, sis = oracle.sort_pairs(hs, ids)
    cs, ce = oracle.cell_bounds(shs, sc.params.numCells)
    st.force[:] = 0
    st.torque[:] = 0
    dF, dT = Dev(st.force), Dev(st.torque)
    args = [Dev(a) for a in (s_pos, s_vel, st.rel, P[sis].copy(), N, si.astype(np.uint32), sis.astype(np.uint32), cs,
                             ce)]
    capi.check(L.arsim_dem_static_grid(dF.p, dT.p, *[a.p for a in args], n, C.byref(sc.params), C.byref(sc.cfg), None))
    sync()
    st.dem_static(cs, ce, P[sis].copy(), N[sis], ref=True)
    rest = si[n:]                                   # sorted particles past n are not part of the call
    st.force[rest] = 0
    st.torque[rest] = 0
    assert np.array_equal(dF.get(), st.force) and np.array_equal(dT.get(), st.torque)
    if points >= 900:
        assert np.abs(st.force).max() > 0


def crowd(n, seed, edge, method=capi.METHOD_GRID):
    """A mixed scene whose particles all lie in a cube of the given edge."""
    sc = scenes.mix_scene(n, seed, method).copy()
    rng = np.random.default_rng(seed)
    grains = sc.rb < 0
    sc.pos[grains, :3] = 5.0 + rng.uniform(0, edge, (int(grains.sum()), 3))
    shift = 5.0 + rng.uniform(0, edge, (sc.b, 3)) - sc.rb_pos[:, :3]
    sc.rb_pos[:, :3] += shift.astype(np.float32)
    sc.rb_vel[:, :3] = rng.normal(size=(sc.b, 3))
    sc.vel[:, :3] = rng.normal(size=(sc.n, 3))
    return sc


@pytest.mark.parametrize("n,edge", [(1, 1.0), (7, 1.0), (9, 1.5), (500, 3.0), (2001, 4.0), (196608, 55.0), (196609, 55.0)])
def test_engine_crowd_vs_oracle(n, edge):
    """Hundreds of candidates a particle, particle counts around a workgroup, both sides of the 16-lane form's limit."""
    print(f"grid contacts: crowd of {n}", flush=True)
    sc = crowd(n, n, edge)
    with Engine(sc) as e:
        e.step(2)
        e.sync()
        g = e.download()
    st = oracle.State(sc, np.float32)
    st.step(2)
    assert_state_equal(g, st, f"crowd of {n}")


def test_engine_small_batch_vs_oracle():
    print("grid contacts: batch of crowds", flush=True)
    mix = [crowd(n, 70 + n, edge) for n, edge in ((3, 1.0), (500, 3.0), (1, 1.0), (129, 2.0), (2000, 5.0))]
    with Engine(mix) as e:
        e.step(2)
        e.sync()
        for k, sc in enumerate(mix):
            st = oracle.State(sc, np.float32)
            st.step(2)
            assert_state_equal(e.download(k), st, f"scene {k}")

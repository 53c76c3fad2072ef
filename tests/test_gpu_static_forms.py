"""Static contacts by one thread or 16 lanes a particle, bit for bit against the oracle: on both sides of the particle
counts that change the workgroups, on sparse and dense points and on both in one call, in the reference's layout and in
the engine."""
import ctypes as C

import numpy as np
import pytest

import oracle
from diploma_thesis_amd import Engine, capi, scenes
from gpu_util import Dev, sync
from test_gpu_engine import assert_state_equal

pytestmark = pytest.mark.gpu


def surface(ext, kind, seed):
    """Points and normals of a floor at y = 5: a cell apart, many to a cell, or both."""
    rng = np.random.default_rng(seed)
    x, z = np.meshgrid(np.arange(1.0, ext), np.arange(1.0, ext), indexing="ij")
    p = np.stack([x.ravel(), np.full(x.size, 5.0), z.ravel()], -1)
    if kind != "sparse":
        part = ext / 5 if kind == "both" else ext
        p = np.concatenate([p, np.stack([rng.uniform(1, part, 30000), rng.normal(5.0, 0.05, 30000), rng.uniform(1, part, 30000)], -1)])
    points, normals = np.zeros((len(p), 4), np.float32), np.zeros((len(p), 4), np.float32)
    points[:, :3] = p
    normals[:, :3] = rng.normal(size=p.shape) * 0.1 + [0, 1, 0]
    normals[:, :3] /= np.linalg.norm(normals[:, :3], axis=1, keepdims=True)
    return points, normals


@pytest.mark.parametrize("n", [65536, 65537, 229377, 262145, 524289])
@pytest.mark.parametrize("kind", ["sparse", "dense", "both"])
def test_reference_layout(n, kind):
    print(f"static forms: {n} particles, {kind} points", flush=True)
    ext = 60.0
    P, N = surface(ext, kind, n)
    sc = scenes.mix_scene(n, 3)
    p = sc.params
    p.gridSize.x, p.gridSize.y, p.gridSize.z = 64, 16, 64
    p.numCells = 64 * 16 * 64
    rng = np.random.default_rng(n)
    st = oracle.State(sc, np.float32)
    st.pos[:, 0], st.pos[:, 2] = rng.uniform(1, ext, n), rng.uniform(1, ext, n)
    st.pos[:, 1] = np.where(rng.random(n) < 0.6, rng.uniform(4.2, 6.2, n), rng.uniform(8, 13, n))
    st.vel[:, :3], st.rel[:, :3] = rng.normal(size=(n, 3)), rng.normal(size=(n, 3))
    h, idx = oracle.calc_hash(st.pos, p)
    _, si = oracle.sort_pairs(h, idx)
    s_pos = st.pos[si].copy()
    s_pos[:, 3] = sc.rb[si].view(np.float32)
    hs, ids = oracle.calc_hash(P, p)
    shs, sis = oracle.sort_pairs(hs, ids)
    cs, ce = oracle.cell_bounds(shs, p.numCells)
    st.force[:], st.torque[:] = 0, 0
    dF, dT = Dev(st.force), Dev(st.torque)
    args = [Dev(a) for a in (s_pos, st.vel[si].copy(), st.rel, P[sis].copy(), N, si.astype(np.uint32),
                             sis.astype(np.uint32), cs, ce)]
    capi.check(capi.lib.arsim_dem_static_grid(dF.p, dT.p, *[a.p for a in args], n, C.byref(p), C.byref(sc.cfg), None))
    sync()
    st.dem_static(cs, ce, P[sis].copy(), N[sis], ref=True)
    assert np.abs(st.force).max() > 0
    assert np.array_equal(dF.get(), st.force) and np.array_equal(dT.get(), st.torque)


@pytest.mark.parametrize("method", [capi.METHOD_GRID, capi.METHOD_LBVH30], ids=["grid", "lbvh30"])
@pytest.mark.parametrize("kind", ["sparse", "both"])
def test_engine(kind, method):
    print(f"static forms: engine, {kind} points, method {method}", flush=True)
    sc = scenes.mix_scene(70001, 4, method).copy()
    ext = float(sc.cfg.boxMax[0])
    rng = np.random.default_rng(4)
    y = 4.0 + rng.uniform(0, 3.0, sc.b).astype(np.float32) - sc.rb_pos[:, 1]
    sc.rb_pos[:, 1] += y
    body = sc.rb >= 0
    sc.pos[body, 1] += y[sc.rb[body]]
    P, N = surface(ext, kind, 4)
    st = oracle.State(sc, np.float32)
    st.set_static(P, N)
    st.step(2)
    with Engine(sc) as e:
        e.set_static(P, N)
        e.step(2)
        e.sync()
        assert_state_equal(e.download(), st, "static forms")

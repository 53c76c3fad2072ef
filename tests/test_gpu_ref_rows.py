"""arsim_dem_grid where a row's three cells are read together, bit for bit against the oracle: rows that wrap or name
a cell more than once, long rows, and a caller's own table whose cells follow each other in any order."""
import ctypes as C

import numpy as np
import pytest

import oracle
from diploma_thesis_amd import capi
from gpu_util import Dev, sync, zeros
from test_gpu_coop_cells import crowd

pytestmark = pytest.mark.gpu
N = 196613


@pytest.mark.parametrize("order", ["ascending", "any"])
@pytest.mark.parametrize("grid", [(1, 256, 256), (2, 256, 256), (4, 128, 512), (512, 16, 32), (64, 64, 64)])
def test_rows_vs_oracle(grid, order):
    print(f"reference layout: grid {grid}, cells in {order} order", flush=True)
    sc = crowd(N, 8, 60.0)
    p = sc.params
    p.gridSize.x, p.gridSize.y, p.gridSize.z = grid
    p.numCells = grid[0] * grid[1] * grid[2]
    h, _ = oracle.calc_hash(sc.pos, p)
    place = np.arange(p.numCells)
    if order == "any":   # blocks of cells moved, so that some rows stay together and some do not
        place = np.random.default_rng(1).permutation(p.numCells // 8)[place // 8] * 8 + place % 8
    si = np.argsort(place[h], kind="stable").astype(np.uint32)
    sh = h[si]
    cs, ce = np.full(p.numCells, 0xffffffff, np.uint32), np.full(p.numCells, 7, np.uint32)   # an empty cell's end: anything
    first = np.nonzero(np.r_[True, sh[1:] != sh[:-1]])[0]
    cs[sh[first]], ce[sh[first]] = first, np.r_[first[1:], sc.n]
    rel = np.zeros((sc.n, 4), np.float32)
    body = sc.rb >= 0
    rel[body, :3] = sc.pos[body, :3] - sc.rb_pos[sc.rb[body], :3]
    s_pos = sc.pos[si].copy()
    s_pos[:, 3] = sc.rb[si].view(np.float32)
    force, torque, vel = zeros((sc.n, 4), np.float32), zeros((sc.n, 4), np.float32), Dev(sc.vel)
    rb, sp, sv, rl, ix, dcs, dce = (Dev(a) for a in (sc.rb, s_pos, sc.vel[si].copy(), rel, si, cs, ce))
    capi.check(capi.lib.arsim_dem_grid(rb.p, force.p, torque.p, vel.p, sp.p, sv.p, rl.p, ix.p, dcs.p, dce.p, sc.n,
                                       C.byref(p), C.byref(sc.cfg), None))
    sync()
    st = oracle.State(sc, np.float32)
    st.rel[:] = rel
    st.dem_grid(si, cs, ce, sc.pos[si], sc.vel[si], sc.rb[si])
    assert np.abs(st.force).max() > 0
    assert np.array_equal(force.get()[body], st.force[body]) and np.array_equal(torque.get()[body], st.torque[body])
    assert np.array_equal(vel.get()[~body], st.vel[~body])

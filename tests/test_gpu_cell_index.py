"""The compact cell index of large sparse grids, bit for bit against the oracle and against the exact table: rows of 8
to 1,024 cells, buckets sorted by one and by two workgroups, a bucket too large for LDS, particles in the cells on
both sides of a grid's edges, and batches on both sides of the rule that chooses it."""
import ctypes as C

import numpy as np
import pytest

import oracle
from diploma_thesis_amd import Engine, capi, scenes
from test_gpu_engine import assert_state_equal

pytestmark = pytest.mark.gpu
N = 200003


def with_grid(sc, gx, gy, gz):
    p = sc.params
    p.gridSize.x, p.gridSize.y, p.gridSize.z = gx, gy, gz
    p.numCells = gx * gy * gz
    return sc


def check(sc, split=0):
    with Engine(sc, bucket_split=split) as e:
        e.step(2)
        e.sync()
        g = e.download()
        # the view of the cell table is restated from the sorted keys: entry c is the first key >= c
        kp, tp, nul = C.c_void_p(), C.c_void_p(), C.POINTER(C.c_void_p)()
        capi.check(capi.lib.arsim_engine_debug_buffers(e.h, C.byref(kp), nul, C.byref(tp), nul, nul, nul, nul, nul, nul,
                                                       nul))
        keys, table = np.zeros(sc.n, np.uint32), np.zeros(sc.params.numCells + 1, np.uint32)
        for dst, src in ((keys, kp), (table, tp)):
            capi.check(capi.lib.arsim_memcpy_dtoh(capi.ptr(dst), src, dst.nbytes, None))
    assert np.array_equal(table, np.searchsorted(keys, np.arange(sc.params.numCells + 1)).astype(np.uint32))
    st = oracle.State(sc, np.float32)
    st.step(2)
    assert_state_equal(g, st, f"grid {sc.params.gridSize.x} x {sc.params.gridSize.y} x {sc.params.gridSize.z}")


@pytest.mark.parametrize("grid", [(8, 512, 1024), (32, 256, 512), (256, 128, 128), (1024, 64, 64)])
@pytest.mark.parametrize("split", [1, 2])
def test_rows_of_cells(grid, split):
    print(f"cell index: grid {grid}, split {split}", flush=True)
    check(with_grid(scenes.mix_scene(N, 5).copy(), *grid), split)


def test_crowded_bucket_and_edges():
    print("cell index: crowd", flush=True)
    sc = with_grid(scenes.mix_scene(N, 6).copy(), 128, 128, 256)
    rng = np.random.default_rng(6)
    grains = np.nonzero(sc.rb < 0)[0]
    sc.pos[grains[:9000], :3] = 40.0 + rng.uniform(0, 12, (9000, 3)) * [1, 1, 0.2]
    sc.pos[grains[9000:15000], :3] = 128.0 + rng.uniform(-2, 2, (6000, 3))      # the grid wraps at 128
    check(sc)


@pytest.mark.parametrize("size,count", [(16384, 16), (24000, 12), (70000, 4)])
def test_batches(size, count):
    print(f"cell index: {count} scenes of about {size}", flush=True)
    mix = [scenes.mix_scene(size + 7 * k, 40 + k) for k in range(count)]
    with Engine(mix) as e:
        e.step(2)
        e.sync()
        for k in (0, 1, count // 2, count - 1):
            st = oracle.State(mix[k], np.float32)
            st.step(2)
            assert_state_equal(e.download(k), st, f"scene {k}")

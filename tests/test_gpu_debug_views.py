"""The debug views between a rebuild and the next step: the buffers hold what the layout before left there, so there
is no last step to view, and asking launches nothing; after the step the views are the new layout's."""
import ctypes as C

import numpy as np
import pytest

from diploma_thesis_amd import Engine, capi, scenes

pytestmark = pytest.mark.gpu


def views(e):
    """(sortedKeys, sortedIndex, cellStart) device addresses, None where there is none."""
    p = [C.c_void_p() for _ in range(3)]
    nul = None
    capi.check(capi.lib.arsim_engine_debug_buffers(e.h, C.byref(p[0]), C.byref(p[1]), C.byref(p[2]), nul, nul, nul, nul,
                                                   nul, nul, nul))
    return [x.value for x in p]


def read(addr, count):
    a = np.zeros(count, np.uint32)
    capi.check(capi.lib.arsim_memcpy_dtoh(capi.ptr(a), C.c_void_p(addr), a.nbytes, None))
    return a


def sparse(n, seed, grid=(256, 128, 128)):
    sc = scenes.mix_scene(n, seed).copy()
    p = sc.params
    p.gridSize.x, p.gridSize.y, p.gridSize.z = grid
    p.numCells = grid[0] * grid[1] * grid[2]
    return sc


def check_table(e, sc):
    keys, idx, table = views(e)
    k = read(keys, sc.n)
    assert np.all(k[1:] >= k[:-1]) and np.array_equal(np.sort(read(idx, sc.n)), np.arange(sc.n))
    assert np.array_equal(read(table, sc.params.numCells + 1),
                          np.searchsorted(k, np.arange(sc.params.numCells + 1)).astype(np.uint32))


# the engine before the rebuild: cell table, compact index with more cells and particles, compact index with fewer
@pytest.mark.parametrize("before", [dict(n=40000, grid=(64, 64, 64)), dict(n=230000, grid=(256, 256, 128)),
                                    dict(n=197000, grid=(128, 128, 128))], ids=["table", "larger", "smaller"])
def test_cell_table_after_a_rebuild(before):
    print(f"debug views: rebuild from {before}", flush=True)
    old, new = sparse(before["n"], 3, before["grid"]), sparse(200003, 4)
    with Engine(old) as e:
        assert views(e)[:2] == [None, None]
        e.step(2)
        e.sync()
        check_table(e, old)
        e.rebuild(None, added=[new])
        assert views(e) == [None, None, None]
        e.step(2)
        e.sync()
        check_table(e, new)

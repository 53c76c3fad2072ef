"""Sequential-impulse sweeps of small islands (groups of contacts that share no body) against the oracle, bit
for bit: contact lists at the edges of what an island may hold, interleaved in the list and with impulses
already there, beside larger ones that take the levels, and engine scenes of both kinds."""
import ctypes as C

import numpy as np
import pytest

import oracle
from diploma_thesis_amd import Engine, capi, scenes
from gpu_util import Dev, sync, zeros
from test_gpu_engine import assert_state_equal
from test_gpu_sis import dense_bodies

pytestmark = pytest.mark.gpu
L = capi.lib


def contact_list(islands, shuffle, rng):
    """islands: (bodies, contacts) each; the contacts of an island link its bodies in a chain, and the rest are
    random pairs, static contacts among them.  Island k's bodies lie scattered among the others'."""
    nb = sum(b for b, _ in islands)
    ids = rng.permutation(nb)
    pairs, at = [], 0
    for b, c in islands:
        own = ids[at:at + b]
        at += b
        mine = [(own[i], own[i + 1]) if rng.random() < 0.5 else (own[i + 1], own[i]) for i in range(b - 1)]
        while len(mine) < c:
            i, j = rng.integers(b), rng.integers(b)
            mine.append((own[i], own[j] if i != j else -1))
        assert len(mine) == c
        pairs += mine
    pairs = np.array(pairs, np.int32)
    return nb, pairs[rng.permutation(len(pairs))] if shuffle else pairs


def solve_both(nb, pairs, seed, iterations=18):
    rng = np.random.default_rng(seed)
    sc = dense_bodies(nb, 4.0, 24.0, seed=seed, k=2)
    st = oracle.State(sc, np.float32)
    st.integrate_bodies()
    n = len(pairs)
    normal, point = np.zeros((n, 4), np.float32), np.zeros((n, 4), np.float32)
    d = rng.normal(size=(n, 3))
    normal[:, :3] = d / np.linalg.norm(d, axis=1, keepdims=True)
    point[:, :3] = st.rb_pos[pairs[:, 0], :3] + rng.normal(scale=0.5, size=(n, 3))
    bias = rng.normal(scale=0.3, size=n).astype(np.float32)
    acc = np.zeros((n, 4), np.float32)
    acc[:, :3] = np.abs(rng.normal(scale=0.2, size=(n, 3)))
    want = {"normal": normal, "point": point, "bodies": pairs.copy(), "bias": bias, "impulse": acc.copy()}
    ws = int(L.arsim_sis_workspace_bytes(n, 0))
    body = [Dev(st.rb_pos), Dev(st.rb_vel), Dev(st.rb_ang), Dev(st.Iw), Dev(st.mass)]
    con = [Dev(normal), Dev(point), Dev(pairs), Dev(bias), Dev(acc)]
    dCnt, dWs = Dev(np.array([n], np.int32)), zeros(ws, np.uint8)
    capi.check(L.arsim_sis_solve(*[c.p for c in con], dCnt.p, n, *[b.p for b in body], nb, iterations,
                                 C.byref(sc.params), dWs.p, ws, None), "sis_solve")
    sync()
    st.sis_solve(want, iterations)
    assert np.isfinite(st.rb_vel).all()
    assert np.array_equal(body[1].get(), st.rb_vel) and np.array_equal(body[2].get(), st.rb_ang)
    assert np.array_equal(con[4].get(), want["impulse"])


# islands of (bodies, contacts): up to 16 bodies and 128 contacts share a wave, up to 128 and 1,024 take one
@pytest.mark.parametrize("islands,shuffle", [
    ([(1, 1)], False),
    ([(2, 1), (1, 3), (2, 7)], True),
    ([(16, 128), (3, 128), (1, 128), (16, 15)], True),
    ([(5, 40)] * 70, False),
    ([(2, 9)] * 257 + [(1, 3)], True),          # two islands a wave, the last one alone
    ([(3, 11), (1, 2), (2, 5)] * 200, True),    # four islands a wave
    ([(1, 4)] * 4096, False),                   # the most bodies
    ([(16, 129), (2, 5)], True),
    ([(17, 40), (2, 5)], True),
    ([(40, 500)] + [(2, 9)] * 300 + [(20, 33), (1, 1400)], True),
    ([(2, 5)] * 150 + [(60, 2100)], False),
    ([(128, 1024), (3, 7)], False),
    ([(128, 1024), (100, 1024), (2, 3)], True),
    ([(129, 600), (2, 5)], True),
    ([(20, 1025), (5, 40)], True),
    ([(17, 20)] * 230, True),
    ([(1, 2)] * 4097, False),
], ids=["one", "three", "full", "seventy", "pairs", "quads", "bodies4096", "contacts129", "bodies17", "mixed",
        "mixed_last", "wave_full", "wave_two", "bodies129", "contacts1025", "waves230", "bodies4097"])
def test_solve_island_sizes_vs_oracle(islands, shuffle):
    print(f"sis islands: {len(islands)} groups, first {islands[0]}", flush=True)
    nb, pairs = contact_list(islands, shuffle, np.random.default_rng(len(islands)))
    solve_both(nb, pairs, 7 + len(islands))


def test_solve_a_body_against_itself_vs_oracle():
    print("sis islands: a contact that names one body twice", flush=True)
    nb, pairs = contact_list([(3, 9), (2, 4)], True, np.random.default_rng(3))
    pairs[5] = pairs[5, 0]
    solve_both(nb, pairs, 11)


def test_engine_scenes_with_and_without_small_islands():
    # sparse scenes (islands), a dense one (levels) and one without contacts in one batch, and each alone
    print("sis islands: batch of both kinds", flush=True)
    mix = [dense_bodies(c, 6.0, s, seed=60 + k, k=3) for k, (c, s) in
           enumerate([(30, 22.0), (90, 10.0), (1, 4.0), (12, 14.0)])]
    floor = scenes.stacked_cubes(4, 3, 2, 3)
    for sc, pts, nrm in [(mix, None, None), floor]:
        many = sc if isinstance(sc, list) else [sc]
        with Engine(sc) as e:
            if pts is not None:
                e.set_static(pts, nrm)
            e.step(5)
            e.sync()
            got = [e.download(s) for s in range(len(many))]
        for s, one in enumerate(many):
            st = oracle.State(one, np.float32)
            if pts is not None:
                st.set_static(pts, nrm)
            st.step(5)
            assert_state_equal(got[s], st, f"scene {s} of {len(many)}")

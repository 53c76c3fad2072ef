"""Reads of the engine's state: several arrays at once (through the pinned buffer up to its size, by copy calls
beyond) against each array read by itself, on both sides of the buffer's size, with and without bodies."""
import ctypes as C

import numpy as np
import pytest

from diploma_thesis_amd import Engine, capi, scenes

pytestmark = pytest.mark.gpu
NAMES = ("pos", "vel", "rel", "force", "torque", "rb_pos", "rb_vel", "rb_ang", "rb_quat", "rb_iw")


def read(e, s, want):
    n, b = e.scenes[s].n, e.scenes[s].b
    out = {k: np.full(((b if k.startswith("rb") else n), 9 if k == "rb_iw" else 4), np.nan, np.float32) for k in want}
    args = [capi.ptr(out[k]) if k in out else None for k in NAMES]
    capi.check(capi.lib.arsim_engine_download(e.h, s, *args), "download")
    return out


@pytest.mark.parametrize("n", [20, 1000, 15000, 29000, 60000, 66000])
def test_arrays_together_equal_arrays_alone(n):
    print(f"fetch: {n} particles", flush=True)
    mix = [scenes.mix_scene(333, 1), scenes.mix_scene(n, 2)]
    with Engine(mix) as e:
        e.step(3)
        for s in (0, 1):
            alone = {k: read(e, s, (k,))[k] for k in NAMES}
            for want in (NAMES, ("pos", "vel"), ("vel", "rb_vel", "rb_iw"), ("pos", "force", "rb_quat")):
                got = read(e, s, want)
                for k in want:
                    assert np.array_equal(got[k], alone[k]), (s, want, k)
            m, q = e.render_state(s)
            assert np.array_equal(q, alone["rb_quat"])
            assert np.array_equal(m[:, 12:15], alone["rb_pos"][:, :3])
            snap = e.snapshot(s)
            assert np.array_equal(snap.pos, alone["pos"]) and np.array_equal(snap.rb_vel, alone["rb_vel"])


def test_relative_positions_survive_a_rebuild():
    """Scenes carried over keep relativePos: zero for grains, whatever the engine's buffers held before."""
    print("fetch: rebuild", flush=True)
    bodies, grains = scenes.mix_scene(6400, 3), scenes.mix_scene(30, 4)   # 30 particles: grains only
    assert grains.b == 0
    with Engine([bodies]) as target, Engine([grains, bodies]) as source:
        target.step(1)                                  # the target's buffers hold the cubes' offsets
        source.step(1)
        want = [read(source, s, ("rel",))["rel"] for s in (0, 1)]
        target.rebuild(source, keep=(0, 1))
        for s in (0, 1):
            assert np.array_equal(read(target, s, ("rel",))["rel"], want[s]), s

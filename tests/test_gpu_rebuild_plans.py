"""A rebuild plans a scene that it carries over from what was measured when the scene came: the carried set takes the
stages that the same scenes take from the host, and steps to the same bits."""
import numpy as np
import pytest

from diploma_thesis_amd import Engine, capi, scenes
from test_gpu_crowded_buckets import slab
from test_gpu_morton_crowds import cluster, in_box

pytestmark = pytest.mark.gpu
STATE = ("pos", "vel", "rb_pos", "rb_vel", "rb_ang", "rb_quat")


def stages(e):
    return [name for name, _ in e.profile()]


def sets():
    big = scenes.mix_scene
    yield "crowded grid", [slab(70000, 90)]
    yield "crowded beside others", [big(20000, 1), slab(190000, 91)]
    yield "small grid scenes", [big(n, 30 + n) for n in (300, 2500, 6000)]
    yield "crowded morton box", [cluster(9000, capi.METHOD_LBVH30, 64)]
    yield "equal codes", [cluster(5000, capi.METHOD_LBVH63, 2048)]
    yield "forest", [big(3000, 1, capi.METHOD_LBVH30), in_box(big(9000, 2, capi.METHOD_LBVH30), 64)]


@pytest.mark.parametrize("name", [n for n, _ in sets()])
def test_carried_set_is_planned_as_from_the_host(name):
    print(f"rebuild plans: {name}", flush=True)
    many = dict(sets())[name]
    other = scenes.mix_scene(100, 5, many[0].cfg.method)
    with Engine(many) as direct, Engine(many) as source, Engine(other) as carried:
        carried.rebuild(source, keep=range(len(many)))
        assert stages(carried) == stages(direct)      # (one step each)
        for e in (carried, direct):
            e.step(2)
            e.sync()
        for s in range(len(many)):
            a, b = carried.download(s), direct.download(s)
            for k in STATE:
                assert np.array_equal(a[k], b[k]), (s, k)

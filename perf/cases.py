"""Performance cases of the DEM step pipeline, through its public entry points.

A case is a dict of plain values; its "kind" says which user's program it stands for:

  scene   one scene held by an engine: `steps` steps, then the renderer's download of the state
          (ParticleSystem::update(dt) and getArray of the reference); "scene" picks the generator
  batch   many independent scenes in one engine, stepped with one launch per stage, then downloaded
  serve   one turn of a serving loop: the two oldest scenes of the resident set retire, two new scenes are
          admitted (arsim_engine_rebuild), the set steps, and the next two to retire are downloaded
  sis     the sequential-impulse model: stacked cubes on a static floor
  stages  the C ABI's stage functions on the caller's own device buffers, one whole step: the drop-in
          use, where ParticleSystem keeps its buffers and each wrapper call is replaced
  ar      one frame of the augmented-reality program through the stage functions: a depth image becomes
          the static scene, which is indexed, and the bodies' particles collide with it and each other

Every state goes on from pass to pass, as a running simulation does.
"""
import ctypes as C
import math
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

from diploma_thesis_amd import Engine, capi, scenes

METHODS = {"grid": capi.METHOD_GRID, "lbvh30": capi.METHOD_LBVH30, "lbvh63": capi.METHOD_LBVH63}
L = capi.lib
STATE = ("pos", "vel", "rb_pos", "rb_vel", "rb_ang", "rb_quat")


def listed():
    return [
        # an interactive frame: one step of the smallest benchmark scene (256 cubes), state read for the renderer
        dict(name="frame_16k_grid", kind="scene", scene="cubes", n=16384, method="grid", steps=1),
        # the headline scene: 8,192 cubes and as many grains, hashed 256^3 grid
        dict(name="headline_1m_grid", kind="scene", scene="headline", n=1048576, method="grid", steps=100),
        # the same scene on the 30-bit Morton tree
        dict(name="headline_1m_lbvh30", kind="scene", scene="headline", n=1048576, method="lbvh30", steps=40),
        # a mid-size ragged scene on the 63-bit tree
        dict(name="mix_50k_lbvh63", kind="scene", scene="mix", n=50021, method="lbvh63", steps=40),
        # the dense settled pile: ellipsoids of 33 to 2,145 particles in packed grains
        dict(name="pile_4m_grid", kind="scene", scene="pile", n=4194304, method="grid", steps=40),
        # many scenes at once (the batched benchmark's range of sizes), grid and LBVH forest
        dict(name="batch_128_grid", kind="batch", scenes=128, lo=1024, hi=65536, method="grid", steps=100),
        dict(name="batch_48_lbvh30", kind="batch", scenes=48, lo=1024, hi=65536, method="lbvh30", steps=40),
        # a turn of the serving loop over its range of scene sizes
        dict(name="serve_24_grid", kind="serve", scenes=24, lo=2048, hi=262144, method="grid", steps=50),
        # the reference's wired default step: two layers of 32 x 32 cubes resting on a scanned floor
        dict(name="sis_32x32x2", kind="sis", nx=32, nz=32, layers=2, steps=5),
        # drop-in stage calls on settled piles, uniform grid and LBVH with the per-step particle box
        dict(name="stages_300k_grid", kind="stages", scene="pile", n=300007, method="grid"),
        dict(name="stages_100k_lbvh30", kind="stages", scene="pile", n=100003, method="lbvh30"),
        # a frame of the augmented-reality program: a 640 x 480 depth image against 256 cubes landing on it
        dict(name="ar_640x480", kind="ar", width=640, height=480, n=16384),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["scene", "scene", "pile", "batch", "serve", "sis", "stages", "stages", "ar"])
    if kind == "scene":
        method = rng.choice(sorted(METHODS))
        return dict(kind="scene", scene="mix", n=log(4096, 1000000), method=method,
                    steps=rng.choice([1, 5, 20, 50]) if method == "grid" else rng.choice([1, 5, 20]))
    if kind == "pile":
        return dict(kind="scene", scene="pile", n=log(65536, 2000000), method=rng.choice(["grid", "lbvh30"]),
                    steps=rng.randint(2, 20))
    if kind in ("batch", "serve"):
        lo = log(1024, 8192)
        return dict(kind=kind, scenes=rng.randint(8, 48), lo=lo, hi=log(2 * lo, 65536),
                    method=rng.choice(["grid", "grid", "lbvh30"]), steps=rng.randint(5, 50))
    if kind == "sis":
        return dict(kind="sis", nx=rng.randint(4, 28), nz=rng.randint(4, 28), layers=rng.randint(1, 3),
                    steps=rng.randint(1, 5))
    if kind == "stages":
        n = log(2048, 600000)      # a pile's container holds its largest body from about 50,000 particles on
        return dict(kind="stages", scene="pile" if n >= 65536 else "mix", n=n, method=rng.choice(sorted(METHODS)))
    w = rng.randint(160, 1280)
    return dict(kind="ar", width=w, height=3 * w // 4, n=64 * log(16, 512))


# ------------------------------------------------------------------------------------------------ scenes
def _scene(case, seed):
    m, n = METHODS[case["method"]], case["n"]
    kind = case["scene"]
    if kind == "cubes":
        return scenes.config0(m, seed)
    if kind == "headline":
        return scenes.config1(m, seed)
    if kind == "pile":
        return scenes.config2(m, seed, scale=n / 4194304)
    return scenes.mix_scene(n, seed, m)


def _sizes(case):
    """Particle counts spread evenly over the logarithm of the range, so that the work is the case's own."""
    s, lo, hi = case["scenes"], case["lo"], case["hi"]
    return [int(round(lo * (hi / lo) ** ((k + 0.5) / s))) for k in range(s)]


def _many(case, seed):
    """The case's scenes, small and large ones mixed."""
    counts = np.random.default_rng(0).permutation(_sizes(case)).tolist()
    m = METHODS[case["method"]]
    with ThreadPoolExecutor(8) as pool:
        return list(pool.map(lambda k: scenes.mix_scene(counts[k], seed * 100003 + k, m), range(len(counts))))


def _host_state(n, b):
    return {k: np.zeros((b if k.startswith("rb") else n, 4), np.float32) for k in STATE}


def _row(a, start):
    return C.c_void_p(a.ctypes.data + 16 * start)


def _download(engine, s, out, p0=0, b0=0):
    """One scene's particle and body state into the caller's arrays, from rows p0 and b0 on."""
    capi.check(L.arsim_engine_download(engine.h, s, _row(out["pos"], p0), _row(out["vel"], p0), None, None, None,
                                       _row(out["rb_pos"], b0), _row(out["rb_vel"], b0), _row(out["rb_ang"], b0),
                                       _row(out["rb_quat"], b0), None), "engine_download")


def _depth_image(case, seed):
    """A room corner seen from above: a tilted plane with boxes on it, sensor noise and pixels without depth."""
    rng = np.random.default_rng(seed)
    w, h = case["width"], case["height"]
    y, x = np.mgrid[0:h, 0:w]
    d = 1.6 + 0.5 * (y / h) + 0.1 * np.sin(6.0 * x / w)
    for _ in range(6):
        cx, cy, s = rng.uniform(0, w), rng.uniform(0, h), rng.uniform(0.05, 0.15) * w
        d = np.where((abs(x - cx) < s) & (abs(y - cy) < s), d - rng.uniform(0.05, 0.3), d)
    d += rng.normal(scale=0.002, size=d.shape)
    d[rng.random(d.shape) < 0.03] = 0.0
    return np.round(np.clip(d, 0.0, 13.0) * 5000.0).astype(np.uint16)


def _accelerometer():
    g = np.array([0.478957, -8.010560, 4.166928])
    return g / np.sqrt((g * g).sum())


def _depth_points(depth):
    """Scene points of a depth image in 64 bits (identity camera), (H, W, 3); without depth at distance -1000."""
    h, w = depth.shape
    y, x = np.mgrid[0:h, 0:w].astype(np.float64)
    d = depth.astype(np.float64) / 5000.0
    d = np.where(d < 0.01, -1000.0, d)
    v = np.stack([d * (x - 318.6) / 517.3, d * (y - 255.3) / 516.5, d], -1)
    gx, gy, gz = _accelerometer().astype(np.float32).astype(np.float64)
    rot = np.array([[1.0, -gx, 0.0], [0.0, -gy, gz], [0.0, -gz, -gy]])
    u = v @ rot.T
    return u * np.array([1.0, -1.0, -1.0])


def _ar_bodies(case, seed, depth):
    """Cubes of 4^3 particles (radius 1/64) landing on scene points: host arrays and parameters."""
    rng = np.random.default_rng(seed + 1)
    r = np.float32(1.0 / 64.0)
    pts = _depth_points(depth).reshape(-1, 3)
    pts = pts[np.abs(pts).max(1) < 500.0]
    b = case["n"] // 64
    off = (np.stack(np.meshgrid(*[np.arange(4)] * 3, indexing="ij"), -1).reshape(-1, 3) - 1.5) * 2.0 * r
    at = pts[rng.integers(0, len(pts), b)] + rng.uniform(0.0, 4.0 * r, (b, 1)) * [0.0, 0.0, 1.0]
    pos = np.zeros((b * 64, 4), np.float32)
    rel = np.zeros_like(pos)
    rel[:, :3] = np.tile(off, (b, 1))
    pos[:, :3] = np.repeat(at, 64, 0) + rel[:, :3]
    vel = np.zeros_like(pos)
    vel[:, :3] = np.repeat(rng.normal(scale=0.3, size=(b, 3)), 64, 0)
    sc = scenes.mix_scene(1024, 0)
    p, cfg = sc.params, sc.cfg
    p.particleRadius = float(r)
    p.gridSize.x = p.gridSize.y = p.gridSize.z = 128
    p.numCells = 128 ** 3
    p.cellSize.x = p.cellSize.y = p.cellSize.z = float(2.0 * r)
    p.spring, p.damping, p.shear = 2000.0, 2.0, 0.5
    cfg.wallMask, cfg.dt = 0, 2e-5
    return dict(pos=pos, vel=vel, rel=rel, rb=np.repeat(np.arange(b, dtype=np.int32), 64)), p, cfg


# ------------------------------------------------------------------------------------------------ states
def prepare(case, seed):
    kind = case["kind"]
    if kind == "scene":
        sc = _scene(case, seed)
        return dict(case=case, engine=Engine(sc), out=_host_state(sc.n, sc.b))
    if kind == "batch":
        many = _many(case, seed)
        return dict(case=case, engine=Engine(many), out=_host_state(sum(s.n for s in many), sum(s.b for s in many)))
    if kind == "serve":
        many = _many(case, seed)
        return dict(case=case, active=Engine(many), idle=Engine(many[:1]), waiting=many)
    if kind == "sis":
        sc, points, normals = scenes.stacked_cubes(case["nx"], case["nz"], case["layers"], seed)
        e = Engine(sc)
        e.set_static(points, normals)
        return dict(case=case, engine=e, out=_host_state(sc.n, sc.b))
    if kind == "stages":
        return _stage_buffers(case, _scene(case, seed))
    depth = _depth_image(case, seed)
    arrays, p, cfg = _ar_bodies(case, seed, depth)
    st = dict(case=case, params=p, cfg=cfg)
    st.update({k: torch.from_numpy(v).cuda() for k, v in arrays.items()})
    st["depth"] = torch.from_numpy(depth.view(np.int16)).cuda()
    n, m = case["n"], depth.size
    st["force"], st["torque"] = _zeros(n, 4), _zeros(n, 4)
    st["static_pos"], st["static_norm"] = _zeros(m, 4), _zeros(m, 4)
    st["static_rb"] = torch.full((m,), -1, dtype=torch.int32, device="cuda")
    for name, k in (("dyn", n), ("sta", m)):
        st[name] = _index_buffers(k, p.numCells, 4)
    return st


def _zeros(*shape, dtype=torch.float32):
    return torch.zeros(shape, dtype=dtype, device="cuda")


def _index_buffers(n, cells, key_bytes):
    """Keys, indices, the sort's scratch, cell table and sorted copies of n points, as the stage functions take them."""
    key = torch.int32 if key_bytes == 4 else torch.int64
    ws = L.arsim_sort_workspace_bytes(n, key_bytes)
    d = dict(keys=_zeros(n, dtype=key), idx=_zeros(n, dtype=torch.int32), keys2=_zeros(n, dtype=key),
             idx2=_zeros(n, dtype=torch.int32), ws=_zeros(ws, dtype=torch.uint8), n=n, key_bytes=key_bytes,
             sorted_pos=_zeros(n, 4), sorted_vel=_zeros(n, 4))
    if cells:
        d["start"], d["end"] = _zeros(cells, dtype=torch.int32), _zeros(cells, dtype=torch.int32)
    return d


def _stage_buffers(case, sc):
    n, b = sc.n, sc.b
    st = dict(case=case, params=sc.params, cfg=sc.cfg, n=n, b=b)
    host = dict(pos=sc.pos, vel=sc.vel, rb=sc.rb, frame=sc.body_frame, rb_pos=sc.rb_pos, rb_vel=sc.rb_vel,
                rb_ang=sc.rb_ang, rb_quat=sc.rb_quat, inertia=sc.rb_inertia, mass=sc.rb_mass, ppo=sc.ppo,
                pstart=sc.pstart)
    st.update({k: torch.from_numpy(np.ascontiguousarray(v)).cuda() for k, v in host.items()})
    st["q_inc"], st["world_inertia"], st["rel"] = _zeros(b, 4), _zeros(b, 9), _zeros(n, 4)
    st["force"], st["torque"] = _zeros(n, 4), _zeros(n, 4)
    if case["method"] == "grid":
        st["index"] = _index_buffers(n, sc.params.numCells, 4)
        return st
    st["index"] = _index_buffers(n, 0, 4 if case["method"] == "lbvh30" else 8)
    st["box"], st["aabb_ws"] = _zeros(2, 4), _zeros(L.arsim_aabb_workspace_bytes(n), dtype=torch.uint8)
    for k in ("left", "right", "parent", "min_range", "max_range"):
        st[k] = _zeros(2 * n - 1, dtype=torch.int32)
    st["is_leaf"] = _zeros(2 * n - 1, dtype=torch.uint8)
    st["counter"], st["overflow"] = _zeros(n, dtype=torch.int32), _zeros(1, dtype=torch.int32)
    st["bounds"] = _zeros(2 * n - 1, 8)
    return st


# ------------------------------------------------------------------------------------------------ passes
def run(state):
    return {"scene": _run_scene, "sis": _run_scene, "batch": _run_batch, "serve": _run_serve, "stages": _run_stages,
            "ar": _run_ar}[state["case"]["kind"]](state)


def _run_scene(state):
    e = state["engine"]
    e.step(state["case"]["steps"])
    _download(e, 0, state["out"])
    return state["out"]


def _run_batch(state):
    e = state["engine"]
    e.step(state["case"]["steps"])
    p0 = b0 = 0
    for s, sc in enumerate(e.scenes):
        _download(e, s, state["out"], p0, b0)
        p0, b0 = p0 + sc.n, b0 + sc.b
    return state["out"]


def _run_serve(state):
    active, idle, waiting = state["active"], state["idle"], state["waiting"]
    idle.rebuild(active, range(2, len(active.scenes)), waiting[:2])
    state["active"], state["idle"] = idle, active
    state["waiting"] = waiting[2:] + waiting[:2]      # the requests to come have the sizes of those that retire
    idle.step(state["case"]["steps"])
    out = []
    for s in (0, 1):
        o = _host_state(idle.scenes[s].n, idle.scenes[s].b)
        _download(idle, s, o)
        out.append(o)
    return out


def _p(t):
    return C.c_void_p(t.data_ptr())


def _sort(d, bits):
    """Sorts d's (keys, idx) and returns the sorted arrays (the call exchanges the caller's pointers)."""
    ptrs = [_p(d[k]) for k in ("keys", "idx", "keys2", "idx2")]
    first = ptrs[0].value
    fn = L.arsim_sort_pairs_u32 if d["key_bytes"] == 4 else L.arsim_sort_pairs_u64
    capi.check(fn(*[C.byref(x) for x in ptrs], d["n"], 0, bits, _p(d["ws"]), d["ws"].numel(), None), "sort")
    return (d["keys"], d["idx"]) if ptrs[0].value == first else (d["keys2"], d["idx2"])


def _index_grid(d, pos, vel, rb, params):
    """Cell keys, sort, sorted copies and cell table of a point set; returns the sorted keys and index."""
    prm = C.byref(params)
    capi.check(L.arsim_calc_hash(_p(d["keys"]), _p(d["idx"]), _p(pos), d["n"], prm, None), "calc_hash")
    keys, idx = _sort(d, max(1, int(params.numCells - 1).bit_length()))
    capi.check(L.arsim_reorder_find_cell_start(_p(rb), _p(d["start"]), _p(d["end"]), _p(d["sorted_pos"]),
                                               _p(d["sorted_vel"]), _p(keys), _p(idx), _p(pos), _p(vel), d["n"],
                                               params.numCells, None), "reorder")
    return keys, idx


def _run_stages(st):
    n, b, prm, cfg, d = st["n"], st["b"], C.byref(st["params"]), C.byref(st["cfg"]), st["index"]
    P = {k: _p(v) for k, v in st.items() if isinstance(v, torch.Tensor)}
    ck = capi.check
    ck(L.arsim_integrate_bodies(P["rb_pos"], P["rb_vel"], P["rb_ang"], P["q_inc"], P["rb_quat"], P["inertia"],
                                P["world_inertia"], None, b, prm, cfg, None))
    ck(L.arsim_particle_pose(P["rb_pos"], P["rb_vel"], P["rb_ang"], P["rb_quat"], P["frame"], P["rb"], P["rel"],
                             P["pos"], P["vel"], n, None))
    ck(L.arsim_integrate_grains(P["pos"], P["vel"], P["rb"], n, prm, cfg, None))
    if st["case"]["method"] == "grid":
        keys, idx = _index_grid(d, st["pos"], st["vel"], st["rb"], st["params"])
        ck(L.arsim_dem_grid(P["rb"], P["force"], P["torque"], P["vel"], _p(d["sorted_pos"]), _p(d["sorted_vel"]),
                            P["rel"], _p(idx), _p(d["start"]), _p(d["end"]), n, prm, cfg, None))
    else:
        box, low, high = _p(st["box"]), _p(st["box"][0]), _p(st["box"][1])
        ck(L.arsim_aabb(P["pos"], n, low, high, P["aabb_ws"], st["aabb_ws"].numel(), None))
        morton = L.arsim_morton30 if d["key_bytes"] == 4 else L.arsim_morton63
        ck(morton(P["pos"], _p(d["keys"]), _p(d["idx"]), n, None, None, box, None))
        keys, idx = _sort(d, 30 if d["key_bytes"] == 4 else 63)
        ck(L.arsim_lbvh_build(_p(keys), d["key_bytes"], n, P["is_leaf"], P["left"], P["right"], P["parent"],
                              P["min_range"], P["max_range"], P["counter"], None))
        ck(L.arsim_lbvh_refit(_p(idx), P["pos"], P["vel"], P["rb"], float(st["params"].particleRadius), n,
                              P["is_leaf"], P["min_range"], P["max_range"], P["left"], P["right"], P["parent"],
                              _p(d["sorted_pos"]), _p(d["sorted_vel"]), P["bounds"], P["counter"], None))
        ck(L.arsim_dem_lbvh(P["rb"], P["force"], P["torque"], P["vel"], _p(d["sorted_vel"]), P["rel"], _p(idx),
                            P["left"], P["right"], _p(d["sorted_pos"]), P["bounds"], n, prm, cfg, P["overflow"],
                            None))
    ck(L.arsim_segmented_reduce_apply(P["force"], P["torque"], P["rel"], P["rb_vel"], P["rb_ang"], P["mass"],
                                      P["world_inertia"], P["pstart"], P["ppo"], b, prm, cfg, None))
    out = {k: st[k] for k in STATE}
    out.update(force=st["force"], torque=st["torque"], keys=keys, idx=idx)
    return out


def _run_ar(st):
    n, m, prm, cfg = st["case"]["n"], st["static_rb"].numel(), C.byref(st["params"]), C.byref(st["cfg"])
    w, h = st["case"]["width"], st["case"]["height"]
    P = {k: _p(v) for k, v in st.items() if isinstance(v, torch.Tensor)}
    camera = np.eye(4, dtype=np.float32).reshape(16)
    dyn, sta = st["dyn"], st["sta"]
    ck = capi.check
    ck(L.arsim_range_image_load(P["depth"], w, h, capi.ptr(camera), float(st["params"].particleRadius),
                                P["static_pos"], P["static_norm"], None, None, None))
    _, static_idx = _index_grid(sta, st["static_pos"], st["static_norm"], st["static_rb"], st["params"])
    keys, idx = _index_grid(dyn, st["pos"], st["vel"], st["rb"], st["params"])
    ck(L.arsim_dem_grid(P["rb"], P["force"], P["torque"], P["vel"], _p(dyn["sorted_pos"]), _p(dyn["sorted_vel"]),
                        P["rel"], _p(idx), _p(dyn["start"]), _p(dyn["end"]), n, prm, cfg, None))
    ck(L.arsim_dem_static_grid(P["force"], P["torque"], _p(dyn["sorted_pos"]), _p(dyn["sorted_vel"]), P["rel"],
                               _p(sta["sorted_pos"]), P["static_norm"], _p(idx), _p(static_idx), _p(sta["start"]),
                               _p(sta["end"]), n, prm, cfg, None))
    return dict(static_pos=st["static_pos"], static_norm=st["static_norm"], force=st["force"], torque=st["torque"],
                keys=keys, idx=idx, static_idx=static_idx)


# ------------------------------------------------------------------------------------------------ work
def work(case):
    """Compulsory traffic: per step each particle's position and velocity in and out and a body particle's frame in,
    each body's state in and out, its inertia in; the state once more for a download.  Operations: about 400 per
    particle (pose or integration, key, the tests and forces of its neighbours)."""
    kind = case["kind"]
    if kind == "ar":
        m, n = case["width"] * case["height"], case["n"]
        return {"bytes": m * (2 + 32 + 4) + n * (16 * 3 + 4 + 32 + 8), "flops": 60 * m + 600 * n}
    if kind == "sis":
        n = case["nx"] * case["nz"] * case["layers"] * 64
        body_n, bodies, steps, extra = n, n // 64, case["steps"], 32 * n
        flops = 18 * 300.0 * 0.37 * n      # 18 sweeps over the contacts
    else:
        if kind in ("batch", "serve"):
            n = sum(_sizes(case))
        else:
            n = case["n"]
        share = {"cubes": 1.0, "headline": 0.5, "pile": 0.68}.get(case.get("scene"), 0.75)
        body_n = int(share * n)
        bodies = body_n // (173 if case.get("scene") == "pile" else 64)
        steps = case.get("steps", 1)
        extra = {"stages": 32 * n + 8 * n, "serve": 64 * n}.get(kind, 32 * n)
        flops = 0.0
    per_step = 64 * n + 16 * body_n + (2 * 64 + 36 + 4) * bodies
    return {"bytes": steps * per_step + extra, "flops": steps * (400.0 * n + flops)}


# ------------------------------------------------------------------------------------------------ 64-bit results
class _Sim64:
    """The same step in 64 bits: independent scenes side by side, contacts from a cell list."""

    def __init__(self, many):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.dev = dev

        def cat(rows, width=None):
            a = np.concatenate([np.asarray(x, np.float64) for x in rows])
            return torch.from_numpy(a).to(dev)

        self.p, self.cfg = many[0].params, many[0].cfg
        self.count = [(s.n, s.b) for s in many]
        self.pos = cat([s.pos[:, :3] for s in many])
        self.vel = cat([s.vel[:, :3] for s in many])
        self.frame = cat([s.body_frame[:, :3] for s in many])
        self.x, self.v = cat([s.rb_pos[:, :3] for s in many]), cat([s.rb_vel[:, :3] for s in many])
        self.w, self.q = cat([s.rb_ang[:, :3] for s in many]), cat([s.rb_quat for s in many])
        self.inertia = cat([s.rb_inertia for s in many]).reshape(-1, 3, 3).transpose(1, 2).contiguous()
        self.mass = cat([s.rb_mass for s in many])
        b0 = np.cumsum([0] + [s.b for s in many])
        rb = np.concatenate([np.where(s.rb >= 0, s.rb + b0[k], -1) for k, s in enumerate(many)])
        self.rb = torch.from_numpy(rb.astype(np.int64)).to(dev)
        self.scene = torch.from_numpy(np.repeat(np.arange(len(many)), [s.n for s in many])).to(dev)
        for name in ("boxMin", "boxMax"):
            box = np.array([list(getattr(s.cfg, name)) for s in many], np.float64)
            setattr(self, name, torch.from_numpy(box).to(dev)[self.scene])
        self.r = float(self.p.particleRadius)
        self.dt = float(self.cfg.dt)
        self.g = torch.tensor([self.p.gravity.x, self.p.gravity.y, self.p.gravity.z], dtype=torch.float64, device=dev)

    def _rotation(self, q):
        x, y, z, w = q.unbind(1)
        return torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                            2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                            2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], 1).reshape(-1, 3, 3)

    @staticmethod
    def _mat_vec(m, v):
        return (m * v[:, None, :]).sum(2)

    def step(self):
        dt, p = self.dt, self.p
        # bodies: position by the old velocity, orientation by the angular velocity, gravity
        self.x = self.x + self.v * dt
        speed = self.w.norm(dim=1, keepdim=True)
        half = 0.5 * speed * dt
        turning = speed * dt > 1e-5
        axis = self.w / speed.clamp_min(1e-300)
        px, py, pz = torch.where(turning, torch.sin(half) * axis, torch.zeros_like(axis)).unbind(1)
        pw = torch.where(turning, torch.cos(half), torch.ones_like(half))[:, 0]
        qx, qy, qz, qw = self.q.unbind(1)
        q = torch.stack([pw * qx + px * qw + py * qz - pz * qy, pw * qy + py * qw + pz * qx - px * qz,
                         pw * qz + pz * qw + px * qy - py * qx, pw * qw - px * qx - py * qy - pz * qz], 1)
        self.q = q / q.norm(dim=1, keepdim=True)
        self.v = self.v + self.g * dt
        self.w = self.w * float(p.Wdamping)
        rot = self._rotation(self.q)
        tmp = (rot[:, :, :, None] * self.inertia[:, None, :, :]).sum(2)
        world = (tmp[:, :, :, None] * rot.transpose(1, 2)[:, None, :, :]).sum(2)
        # particles
        body = self.rb >= 0
        k = self.rb.clamp_min(0)
        grain_v = (self.vel + self.g * dt) * float(p.globalDamping)
        if self.x.shape[0]:
            rel = self._mat_vec(rot[k], self.frame)
            pos_b, vel_b = self.x[k] + rel, self.v[k] + torch.linalg.cross(self.w[k], rel)
        else:
            rel = pos_b = vel_b = torch.zeros_like(self.pos)
        self.pos = torch.where(body[:, None], pos_b, self.pos + grain_v * dt)
        self.vel = torch.where(body[:, None], vel_b, grain_v)
        self.rel = torch.where(body[:, None], rel, torch.zeros_like(rel))
        force = self._contacts() + self._walls()
        # bodies take the sums of their particles' forces, grains their own
        self.vel = torch.where(body[:, None], self.vel, self.vel + force * dt)
        self.force = torch.where(body[:, None], force, torch.zeros_like(force))
        self.torque = torch.linalg.cross(self.rel, self.force)
        if self.x.shape[0]:
            total = torch.zeros_like(self.v).index_add_(0, k, self.force)
            twist = torch.zeros_like(self.v).index_add_(0, k, self.torque)
            self.v = self.v + total * dt / self.mass[:, None]
            self.w = self.w + self._mat_vec(world, twist) * dt

    def _law(self, rel, normal, rv, overlap):
        p = self.p
        tangential = rv - (rv * normal).sum(1, keepdim=True) * normal
        return -p.spring * overlap * normal + p.damping * rv + p.shear * tangential + p.attraction * rel

    def _contacts(self):
        force = torch.zeros_like(self.pos)
        for a, b, rel, dist in _neighbours(self.pos, self.pos, 2.0 * self.r, self.scene, self.scene):
            keep = (a != b) & ((self.rb[a] != self.rb[b]) | (self.rb[a] < 0))
            a, b, rel, dist = a[keep], b[keep], rel[keep], dist[keep]
            f = self._law(rel, rel / dist, self.vel[b] - self.vel[a], 2.0 * self.r - dist)
            force.index_add_(0, a, f)
        return force

    def _walls(self):
        force = torch.zeros_like(self.pos)
        for bit in range(6):
            if not self.cfg.wallMask >> bit & 1:
                continue
            axis, high = bit >> 1, bool(bit & 1)
            d = self.boxMax[:, axis] - self.pos[:, axis] if high else self.pos[:, axis] - self.boxMin[:, axis]
            hit = torch.nonzero(d < self.r)[:, 0]
            normal = torch.zeros((hit.numel(), 3), dtype=torch.float64, device=self.dev)
            normal[:, axis] = 1.0 if high else -1.0
            d = d[hit, None]
            force[hit] += self._law(d * normal, normal, -self.vel[hit], self.r - d)
        return force

    def state(self, first=0, last=None):
        """pos, vel and the bodies' state of scenes first .. last as the engine lays them out."""
        last = len(self.count) if last is None else last
        ps = slice(sum(n for n, _ in self.count[:first]), sum(n for n, _ in self.count[:last]))
        bs = slice(sum(b for _, b in self.count[:first]), sum(b for _, b in self.count[:last]))
        return dict(pos=_pad(self.pos[ps]), vel=_pad(self.vel[ps]), rb_pos=_pad(self.x[bs]), rb_vel=_pad(self.v[bs]),
                    rb_ang=_pad(self.w[bs]), rb_quat=self.q[bs])


def _pad(v):
    return torch.cat([v, torch.zeros_like(v[:, :1])], 1)


def _neighbours(pa, pb, reach, sa, sb):
    """Yields (a, b, pb[b] - pa[a], distance) for the pairs of equal scenes closer than `reach`, in pieces."""
    low = torch.minimum(pa.min(0).values, pb.min(0).values)
    ca, cb = ((pa - low) / reach).floor().long() + 1, ((pb - low) / reach).floor().long() + 1
    size = torch.maximum(ca.max(0).values, cb.max(0).values) + 2

    def key(c, s):
        return ((s * size[2] + c[:, 2]) * size[1] + c[:, 1]) * size[0] + c[:, 0]

    keys, order = torch.sort(key(cb, sb))
    ka = key(ca, sa)
    for at in range(0, pa.shape[0], 1 << 19):
        some = torch.arange(at, min(at + (1 << 19), pa.shape[0]), device=pa.device)
        for dz in (-1, 0, 1):
            for dy in (-1, 0, 1):
                row = ka[some] + (dz * size[1] + dy) * size[0]
                begin = torch.searchsorted(keys, row - 1)
                count = torch.searchsorted(keys, row + 1, right=True) - begin
                a = torch.repeat_interleave(some, count)
                base = torch.repeat_interleave(begin - (count.cumsum(0) - count), count)
                b = order[base + torch.arange(a.numel(), device=pa.device)]
                rel = pb[b] - pa[a]
                dist = rel.norm(dim=1, keepdim=True)
                near = torch.nonzero(dist[:, 0] < reach)[:, 0]
                yield a[near], b[near], rel[near], dist[near]


def exact(case, seed):
    """What the first pass on a new state returns, in 64 bits.  The sequential impulses have no such value: cubes
    stacked face to face meet at equal depths, and which contact is the deepest is decided by rounding."""
    kind = case["kind"]
    if kind == "sis":
        return None
    if kind == "ar":
        return _exact_ar(case, seed)
    if kind in ("scene", "stages"):
        sim = _Sim64([_scene(case, seed)])
    else:
        many = _many(case, seed)
        sim = _Sim64(many[2:4] if kind == "serve" else many)
    for _ in range(case.get("steps", 1)):
        sim.step()
    if kind == "serve":
        return [sim.state(0, 1), sim.state(1, 2)]
    out = sim.state()
    if kind == "stages":
        out.update(force=_pad(sim.force), torque=_pad(sim.torque), keys=None, idx=None)
    return out


def _exact_ar(case, seed):
    depth = _depth_image(case, seed)
    arrays, p, cfg = _ar_bodies(case, seed, depth)
    w, h = case["width"], case["height"]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    pts = torch.from_numpy(_depth_points(depth)).to(dev)
    pts.reshape(-1, 3)[(w - 1) * (h - 1) + 1:] = 0.0        # pixels past (W-1)(H-1) are not written
    norm = torch.zeros_like(pts)
    n = torch.linalg.cross(pts[2:, 1:-1] - pts[:-2, 1:-1], pts[1:-1, 2:] - pts[1:-1, :-2])
    norm[1:-1, 1:-1] = n / n.norm(dim=2, keepdim=True)
    pts, norm = pts.reshape(-1, 3), norm.reshape(-1, 3)
    sim = object.__new__(_Sim64)
    sim.dev, sim.p, sim.cfg, sim.r = dev, p, cfg, float(p.particleRadius)
    for name, a in (("pos", "pos"), ("vel", "vel"), ("rel", "rel")):
        setattr(sim, name, torch.from_numpy(arrays[a][:, :3].astype(np.float64)).to(dev))
    sim.rb = torch.from_numpy(arrays["rb"].astype(np.int64)).to(dev)
    sim.scene = torch.zeros_like(sim.rb)
    force = sim._contacts()
    near = torch.nonzero(pts.abs().amax(1) < 500.0)[:, 0]
    at = pts[near]
    none = torch.zeros(at.shape[0], dtype=torch.int64, device=dev)
    for a, b, rel, dist in _neighbours(sim.pos, at, 2.0 * sim.r, sim.scene, none):
        force.index_add_(0, a, sim._law(rel, -norm[near[b]], -sim.vel[a], 2.0 * sim.r - dist))
    return dict(static_pos=_pad(pts), static_norm=_pad(norm), force=_pad(force),
                torque=_pad(torch.linalg.cross(sim.rel, force)), keys=None, idx=None, static_idx=None)

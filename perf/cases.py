"""Performance cases: the calls that a program using physkit_amd makes, at the sizes it
makes them.

A case names one `kind` of call and its sizes; the same kinds, with other sizes, are what
draw() returns.

  frame    a world set to the state that the program holds, one step, every body's state
           read back: the latency path (an environment's step, a frame replayed after a
           rollback)
  rollout  bodies set to a given state, `steps` steps in one call, every body's state read
           back: a planner, a trainer or an offline simulation. `scene` picks the bodies:
           pyramids (resting stacks), worlds (a batch of independent uneven worlds),
           granular (a dense lattice falling, far more broadphase pairs than contacts),
           hulls (deeply overlapping clusters, with solver and integration), chains
           (joints)
  collide  collision detection alone: overlapping pairs and contact counts of unmoving
           hulls, every leaf queried
  rays     closest hits of rays held in device memory
  queries  all hits of a batch of rays and the bodies of a batch of boxes, host arrays
  narrow   standalone GJK/EPA over shape pairs held in device memory
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import torch

import physkit_amd as pk

# EPA_GUARD: a degenerate polytope gives no contact instead of NaN that spreads
FP64, MIXED = pk.FLAG_EPA_GUARD, pk.FLAG_EPA_GUARD | pk.FLAG_MIXED


def listed():
    return [
        # a small world through the object API: launches and host waits count
        {"name": "frame_64", "kind": "frame", "bodies": 64, "api": "world"},
        # the 1,024-box scene two seconds in, piled up, stepped and read frame by frame
        {"name": "frame_1024", "kind": "frame", "bodies": 1024, "api": "bulk"},
        # 64 pyramids of 120 boxes at rest: long contact islands, 20 solver iterations
        {"name": "pyramids_64", "kind": "rollout", "scene": "pyramids", "count": 64, "mixed": False, "steps": 10},
        # about 14 independent worlds (10,000 bodies) in FP64, as a small planner batch runs them
        {"name": "worlds_10k_fp64", "kind": "rollout", "scene": "worlds", "count": 10000, "mixed": False, "steps": 20},
        # a training batch: about 1,000 worlds in the mixed-precision form
        {"name": "worlds_720k_mixed", "kind": "rollout", "scene": "worlds", "count": 720000, "mixed": True,
         "steps": 20},
        # a granular lattice: about 170 broadphase pairs to each body, nearly all culled
        {"name": "granular_131072_mixed", "kind": "rollout", "scene": "granular", "count": 131072, "mixed": True,
         "steps": 20},
        # overlapping hull clusters set free: islands too long for one workgroup
        {"name": "hulls_16384_fp64", "kind": "rollout", "scene": "hulls", "count": 16384, "mixed": False, "steps": 5},
        # jointed chains (hinges, ball sockets, sliders, distances, welds, springs)
        {"name": "chains_256", "kind": "rollout", "scene": "chains", "count": 256, "mixed": False, "steps": 20},
        # the narrowphase stress scene: 262,144 hulls, every pair through GJK, one detection
        {"name": "collide_262144", "kind": "collide", "bodies": 262144, "mixed": False},
        # closest-hit raycasts at the benchmark's size
        {"name": "rays_4m", "kind": "rays", "rays": 4194304, "bodies": 262144},
        # the queries that an application makes between steps
        {"name": "queries_4096", "kind": "queries", "rays": 4096, "boxes": 1024, "bodies": 32768},
        # a full batch of the entry point that allocates nothing
        {"name": "narrow_65536", "kind": "narrow", "pairs": 65536},
    ]


def _logint(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["frame", "frame", "rollout", "rollout", "rollout", "rollout", "collide", "rays", "queries",
                       "narrow"])
    if kind == "frame":
        return {"kind": kind, "bodies": _logint(rng, 8, 2048), "api": rng.choice(["world", "bulk", "bulk"])}
    if kind == "collide":
        return {"kind": kind, "bodies": _logint(rng, 1024, 200000), "mixed": rng.random() < 0.4}
    if kind == "rays":
        return {"kind": kind, "rays": _logint(rng, 1000, 3000000), "bodies": _logint(rng, 500, 150000)}
    if kind == "queries":
        return {"kind": kind, "rays": _logint(rng, 1, 16384), "boxes": _logint(rng, 1, 8192),
                "bodies": _logint(rng, 200, 32768)}
    if kind == "narrow":
        return {"kind": kind, "pairs": _logint(rng, 50, 60000)}
    scene = rng.choice(["pyramids", "worlds", "worlds", "granular", "hulls", "chains"])
    lo, hi = {"pyramids": (1, 64), "worlds": (500, 600000), "granular": (2000, 120000), "hulls": (1024, 16384),
              "chains": (4, 256)}[scene]
    return {"kind": kind, "scene": scene, "count": _logint(rng, lo, hi),
            "mixed": scene != "pyramids" and rng.random() < 0.5,
            "steps": rng.randint(2, 5) if scene == "hulls" else rng.randint(5, 20)}


# ---------------------------------------------------------------- scenes
def _take(s, idx):
    """Bodies idx (with repeats) of scene s, sharing its shapes."""
    out = {k: s[k][idx].copy() for k in ("is_static", "shape", "pos", "vel", "angvel", "quat", "mass", "inertia",
                                         "restitution", "friction")}
    out.update({k: s[k] for k in ("shape_offsets", "verts", "dt", "iterations", "flags")})
    return out


def _worlds(bodies, seed):
    """Independent worlds of `bodies` bodies in all: copies of 16 distinct uneven worlds (16
    to 4,096 bodies), each copy with velocities of its own, the last one cut to fit."""
    rng = np.random.default_rng(seed)
    base = pk.scene(pk.SCENE_BATCHED, seed, 16)
    fb = base["first_body"].astype(np.int64)
    size = fb[1:] - fb[:-1]
    which = np.arange(16 * (bodies // int(size.sum()) + 1)) % 16
    ends = np.cumsum(size[which])
    which = which[:int(np.searchsorted(ends, bodies)) + 1]
    s = _take(base, np.concatenate([np.arange(fb[w], fb[w + 1]) for w in which])[:bodies])
    s["first_body"] = np.concatenate([[0], ends[:len(which) - 1], [bodies]]).astype(np.uint32)
    dyn = s["is_static"] == 0
    s["vel"][dyn] += rng.normal(size=(int(dyn.sum()), 3)) * 0.5
    return s


def _granular(count, seed):
    """The granular generator's bodies (8 x 12 UV spheres and boxes of 1-3 cm, 0.07 m
    lattice, 64-box hopper) with their shapes drawn from 4,096."""
    rng = np.random.default_rng(seed)
    base = pk.scene(pk.SCENE_GRANULAR_LOW, seed, min(count, 4096))
    ns, n0 = int(base["n_static"]), len(base["shape"])
    s = _take(base, np.concatenate([np.arange(ns), rng.integers(ns, n0, count)]))
    side = int(np.ceil(count ** (1.0 / 3.0)))
    while side ** 3 < count:
        side += 1
    k = np.arange(count)
    grid = np.stack([k % side, k // (side * side), (k // side) % side], 1).astype(float)
    low = np.array([-0.035 * (side - 1), 10.0, -0.035 * (side - 1)])
    s["pos"][ns:] = low + 0.07 * grid + rng.uniform(-0.004, 0.004, (count, 3))
    return s


def _chains(count, seed):
    """`count` chains of 16 boxes hanging from a static box, the six joint types in turn."""
    rng = np.random.default_rng(seed)
    links, h = 16, (0.1, 0.2, 0.1)
    n = count * (links + 1)
    row, link = np.divmod(np.arange(n), links + 1)
    side = int(np.ceil(np.sqrt(count)))
    pos = np.stack([2.0 * (row % side), -0.5 * link, 2.0 * (row // side)], 1).astype(float)
    stat = link == 0
    mass = 1000.0 * 8.0 * h[0] * h[1] * h[2]
    inertia = np.diag([mass / 3 * (h[1] ** 2 + h[2] ** 2), mass / 3 * (h[0] ** 2 + h[2] ** 2),
                       mass / 3 * (h[0] ** 2 + h[1] ** 2)]).reshape(9)
    s = {"shape_offsets": np.array([0, 8], np.uint32), "verts": pk.mesh.box(h).vertices,
         "is_static": stat.astype(np.uint8), "shape": np.zeros(n, np.uint32), "pos": pos,
         "vel": rng.normal(size=(n, 3)) * 0.5 * ~stat[:, None], "angvel": np.zeros((n, 3)),
         "quat": np.tile([1.0, 0.0, 0.0, 0.0], (n, 1)), "mass": np.full(n, mass), "inertia": np.tile(inertia, (n, 1)),
         "restitution": np.full(n, 0.3), "friction": np.full(n, 0.5), "dt": 1.0 / 60.0, "iterations": 10, "flags": 0}
    types = [pk.JOINT_HINGE, pk.JOINT_BALL_SOCKET, pk.JOINT_DISTANCE, pk.JOINT_BALL_SOCKET, pk.JOINT_SLIDER,
             pk.JOINT_HINGE, pk.JOINT_SPRING, pk.JOINT_WELD]
    slots, joints = dict.fromkeys(types, 0), []
    for b in np.nonzero(~stat)[0].tolist():
        t = types[(b % (links + 1)) % len(types)]
        joints.append({"type": t, "slot": slots[t], "a": b - 1, "b": b, "local_a": (0.0, -0.25, 0.0),
                       "local_b": (0.0, 0.25, 0.0), "local_axis_a": (0.0, 0.0, 1.0), "local_axis_b": (0.0, 0.0, 1.0),
                       "anchor": tuple(pos[b] + (0.0, 0.25, 0.0)), "axis": (0.0, 1.0, 0.0), "distance": 0.05,
                       "stiffness": 2000.0, "damping": 20.0})
        slots[t] += 1
    s["joints"] = joints
    return s


def _load(s, flags):
    w = pk.GpuWorld(iterations=s["iterations"], flags=flags)
    w.load_scene(s)
    return w


def _random_rays(pos, n, seed):
    """Origins in the bodies' box grown by 10 m; half the rays aimed at a body, half of
    uniform direction; unbounded."""
    rng = np.random.default_rng(seed)
    o = rng.uniform(pos.min(0) - 10.0, pos.max(0) + 10.0, (n, 3))
    d = rng.normal(size=(n, 3))
    k = n // 2
    d[:k] = pos[rng.integers(len(pos), size=k)] - o[:k] + 0.05 * d[:k]
    return o, d, np.full(n, np.inf)


def _query_boxes(pos, n, seed):
    rng = np.random.default_rng(seed + 1)
    c = pos[rng.integers(len(pos), size=n)]
    h = rng.uniform(0.1, 1.0, (n, 3))
    return np.concatenate([c - h, c + h], 1)


def _shape_pairs(n, seed):
    """n pairs of AABBs, OBBs and box, pyramid, hull and UV-sphere meshes, about half of
    them overlapping, in the layout of pkg_gjk_epa_batch."""
    rng = np.random.default_rng(seed)
    meshes = [pk.mesh.box((0.4, 0.3, 0.5)).vertices, pk.mesh.pyramid(0.5, 0.7).vertices,
              pk.mesh.sphere(0.4, 16, 32).vertices]
    for k in (8, 13, 20, 32):
        v = rng.normal(size=(k, 3))
        meshes.append(v / np.linalg.norm(v, axis=1, keepdims=True) * rng.uniform(0.2, 0.5, 3))
    offs = np.cumsum([0] + [len(m) for m in meshes])
    sides = []
    for side in range(2):
        kind = np.where(rng.random(n) < 0.3, rng.integers(0, 3, n), 2).astype(np.int32)
        q = rng.normal(size=(n, 4))
        q /= np.linalg.norm(q, axis=1, keepdims=True)
        c = rng.normal(size=(n, 3)) * 0.35 + 0.4 * side
        h = rng.uniform(0.1, 0.6, (n, 3))
        m = rng.integers(0, len(meshes), n)
        prm = np.zeros((n, 10))
        prm[:, :3], prm[:, 3:7] = c, q
        prm[kind == 1, 7:] = h[kind == 1]
        flat = kind == 0
        prm[flat] = 0.0
        prm[flat, :3], prm[flat, 3:6] = (c - h)[flat], (c + h)[flat]
        mesh = kind == 2
        sides += [kind, prm, np.where(mesh, offs[m], 0).astype(np.int32),
                  np.where(mesh, offs[m + 1], 0).astype(np.int32)]
    return sides, np.concatenate(meshes)


def _cuda(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


# ---------------------------------------------------------------- prepare
def prepare(case, seed):
    st = {"case": case}
    kind = case["kind"]
    if kind == "frame":
        s = pk.scene(pk.SCENE_BOXES, seed, case["bodies"])
        if case["api"] == "bulk":
            w = gpu = _load(s, s["flags"] | FP64)
        else:
            off = s["shape_offsets"]
            w = pk.world(pk.world_desc.make().with_solver_iterations(s["iterations"]).with_epa_guard())
            for i, sh in enumerate(s["shape"].tolist()):
                d = pk.object_desc.stat() if s["is_static"][i] else pk.object_desc.dynam()
                w.create_rigid(d.with_mesh(pk.mesh.make(s["verts"][off[sh]:off[sh + 1]])).with_pos(s["pos"][i])
                               .with_vel(s["vel"][i]).with_orientation(s["quat"][i]).with_mass(s["mass"][i])
                               .with_inertia_tensor(s["inertia"][i].reshape(3, 3)))
            gpu = w.gpu
        gpu.step(s["dt"], 120)  # two seconds in: most boxes have landed
        b = gpu.bodies()
        st.update(w=w, gpu=gpu, dt=s["dt"], ids=np.arange(gpu.n, dtype=np.uint32),
                  start={k: b[k] for k in ("pos", "vel", "angvel", "quat")})
    elif kind == "rollout":
        scene, count, settle = case["scene"], case["count"], 0
        flags = MIXED if case["mixed"] else FP64
        if scene == "pyramids":
            s, settle = pk.scene(pk.SCENE_PYRAMIDS, seed, count), 30
        elif scene == "worlds":
            s, settle = _worlds(count, seed), 45
        elif scene == "granular":
            s, settle = _granular(count, seed), 3
        elif scene == "hulls":
            s = pk.scene(pk.SCENE_HULLS, seed, count)
            s["flags"] = 0  # the generator's own flags switch solver and integration off
        else:
            s, settle = _chains(count, seed), 30
        w = _load(s, s["flags"] | flags)
        if scene == "worlds":
            w.set_worlds(s["first_body"])
        if scene == "chains":
            w.add_joints(s["joints"])
        if settle:
            w.step(s["dt"], settle)
        b = w.bodies()
        st.update(w=w, dt=s["dt"], ids=np.arange(w.n, dtype=np.uint32),
                  start={k: b[k] for k in ("pos", "vel", "angvel", "quat")})
    elif kind == "collide":
        s = pk.scene(pk.SCENE_HULLS, seed, case["bodies"])
        st.update(w=_load(s, s["flags"] | (pk.FLAG_FP32_GJK | pk.FLAG_FP32_BROAD if case["mixed"] else 0)), dt=s["dt"])
        st["w"].step(s["dt"])
        # buffers of the caller's own, with room to spare (a hull has about 4 pairs)
        cap = 16 * case["bodies"] + 4096
        st.update(keys=np.zeros(cap, np.uint64), counts=np.zeros(cap, np.int32))
    elif kind == "rays":
        s = pk.scene(pk.SCENE_HULLS, seed, case["bodies"])
        o, d, m = _random_rays(s["pos"], case["rays"], seed)
        st.update(w=_load(s, 0), n=case["rays"], inp=[_cuda(o), _cuda(d), _cuda(m)],
                  ids=torch.zeros(case["rays"], dtype=torch.int32, device="cuda"),
                  dists=torch.zeros(case["rays"], dtype=torch.float64, device="cuda"))
    elif kind == "queries":
        s = pk.scene(pk.SCENE_HULLS, seed, case["bodies"])
        st.update(w=_load(s, 0), rays=_random_rays(s["pos"], case["rays"], seed),
                  boxes=_query_boxes(s["pos"], case["boxes"], seed))
        # where the program keeps its hits: room for 128 a ray and 256 a box
        st.update(ids=np.zeros(128 * case["rays"] + 4096, np.int64), dist=np.zeros(128 * case["rays"] + 4096),
                  box_ids=np.zeros(256 * case["boxes"] + 4096, np.int64))
    else:
        sides, verts = _shape_pairs(case["pairs"], seed)
        st.update(w=pk.GpuWorld(), n=case["pairs"], nv=len(verts), inp=[_cuda(a) for a in sides] + [_cuda(verts)],
                  out=torch.zeros(case["pairs"], 10, dtype=torch.float64, device="cuda"),
                  hit=torch.zeros(case["pairs"], dtype=torch.int32, device="cuda"))
        fn = pk.lib().pkg_gjk_epa_batch_device
        fn.argtypes = [C.c_void_p, C.c_uint32] + [C.c_void_p] * 9 + [C.c_uint32, C.c_void_p, C.c_void_p]
    return st


# ---------------------------------------------------------------- run
def _ok(w, status):
    if status != pk.PKG_OK:
        raise pk.PkgError(status, w.L.pkg_last_error(w.h))


def run(st):
    w, kind = st["w"], st["case"]["kind"]
    if kind == "frame":
        st["gpu"].set_state(st["ids"], **st["start"])
        w.step(st["dt"])
        return w.state() if st["case"]["api"] == "world" else w.bodies()
    if kind == "rollout":
        w.set_state(st["ids"], **st["start"])
        w.step(st["dt"], st["case"]["steps"])
        return w.bodies()
    if kind == "collide":
        w.step(st["dt"])
        keys, counts, n = st["keys"], st["counts"], C.c_size_t()
        _ok(w, w.L.pkg_get_pairs(w.h, keys.ctypes.data_as(pk.U64), len(keys), C.byref(n)))
        if n.value > len(keys):
            raise pk.PkgError(pk.PKG_INVALID_ARG, "more pairs than the buffers hold")
        _ok(w, w.L.pkg_get_manifolds(w.h, counts.ctypes.data_as(pk.I32), None, len(counts), C.byref(n)))
        return keys.view(np.int64), counts
    if kind == "rays":
        o, d, m = (t.data_ptr() for t in st["inp"])
        _ok(w, w.L.pkg_raycast_closest_device(w.h, st["n"], o, d, m, None, st["ids"].data_ptr(),
                                              st["dists"].data_ptr(), None))
        return st["ids"], st["dists"]
    if kind == "queries":
        off, ids, dist = w.raycast(*st["rays"])
        boff, bids = w.query_aabb(st["boxes"])
        st["ids"][:len(ids)], st["dist"][:len(dist)], st["box_ids"][:len(bids)] = ids, dist, bids
        return {"off": off.astype(np.int64), "ids": st["ids"], "dist": st["dist"], "box_off": boff.astype(np.int64),
                "box_ids": st["box_ids"]}
    p = [t.data_ptr() for t in st["inp"]]
    _ok(w, w.L.pkg_gjk_epa_batch_device(w.h, st["n"], *p, st["nv"], st["out"].data_ptr(), st["hit"].data_ptr()))
    return st["out"], st["hit"]


# ---------------------------------------------------------------- work
def work(case):
    """Inputs read once and outputs written once; a step reads and writes each body's state
    (589 bytes) and its pairs (24 bytes)."""
    kind = case["kind"]
    if kind == "frame":
        n = case["bodies"] + 1
        return {"bytes": n * (589 + 153 + 24 * 3), "flops": n * 3e4}
    if kind == "rollout":
        n, pairs, flops = {"pyramids": (120, 3, 3e4), "worlds": (1, 1, 8e3), "granular": (1, 170, 5e3),
                           "hulls": (1, 4, 3e4), "chains": (17, 2, 1e4)}[case["scene"]]
        n *= case["count"]
        return {"bytes": n * (case["steps"] * (589 + 24 * pairs) + 104 + 153), "flops": n * case["steps"] * flops}
    if kind == "collide":
        n = case["bodies"]
        return {"bytes": n * (20 * 24 + 56 + 4 * (24 + 12) + 6 * 8), "flops": n * 6e4}
    if kind == "rays":
        return {"bytes": 68 * case["rays"] + 89 * case["bodies"], "flops": 2e3 * case["rays"]}
    if kind == "queries":
        return {"bytes": 56 * case["rays"] + 48 * case["boxes"] + 89 * case["bodies"],
                "flops": 5e3 * (case["rays"] + case["boxes"])}
    return {"bytes": case["pairs"] * (2 * (92 + 24 * 20) + 84), "flops": 2e4 * case["pairs"]}


# ---------------------------------------------------------------- exact
def _bounds(s):
    """World bounds of freshly loaded bodies: the box of the rotated corners of each
    shape's local box."""
    off = s["shape_offsets"].astype(np.int64)
    lo, hi = np.minimum.reduceat(s["verts"], off[:-1])[s["shape"]], np.maximum.reduceat(s["verts"], off[:-1])[s["shape"]]
    w, x, y, z = s["quat"].T
    rot = np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                    2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                    2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], 1).reshape(-1, 3, 3)
    c = [np.einsum("nij,nj->ni", rot, np.stack([np.where(k >> a & 1, hi[:, a], lo[:, a]) for a in range(3)], 1))
         for k in range(8)]
    return s["pos"] + np.min(c, 0), s["pos"] + np.max(c, 0)


def _slabs(o, inv, lo, hi):
    """Entry distance of rays (rows) into boxes (columns), infinite where they miss."""
    tmin = torch.full((len(o), len(lo)), -torch.inf, dtype=torch.float64, device=o.device)
    tmax = -tmin
    for a in range(3):
        t0 = (lo[None, :, a] - o[:, None, a]) * inv[:, None, a]
        t1 = (hi[None, :, a] - o[:, None, a]) * inv[:, None, a]
        t0, t1 = torch.nan_to_num(t0, -torch.inf, torch.inf, -torch.inf), torch.nan_to_num(t1, torch.inf, torch.inf, -torch.inf)
        tmin, tmax = torch.maximum(tmin, torch.minimum(t0, t1)), torch.minimum(tmax, torch.maximum(t0, t1))
    return torch.where((tmax >= 0) & (tmin <= tmax), tmin.clamp(min=0.0), torch.inf)


def exact(case, seed):
    """Queries by brute force. A step's result is a long chain of contact decisions that
    amplify any difference, and GJK/EPA stops at a tolerance on a polytope of its own:
    neither has a value of its own outside that algorithm."""
    if case["kind"] not in ("rays", "queries") or case["rays"] * case["bodies"] > 3e10:
        return None
    s = pk.scene(pk.SCENE_HULLS, seed, case["bodies"])
    lo, hi = (torch.from_numpy(x).cuda() for x in _bounds(s))
    o, d, _ = (torch.from_numpy(x).cuda() for x in _random_rays(s["pos"], case["rays"], seed))
    inv = 1.0 / (d / d.norm(dim=1, keepdim=True))
    part = max(1, int(5e7) // case["bodies"])
    if case["kind"] == "rays":
        return None, torch.cat([_slabs(o[k:k + part], inv[k:k + part], lo, hi).min(1).values
                                for k in range(0, case["rays"], part)])
    dist = []
    for k in range(0, case["rays"], part):
        t = _slabs(o[k:k + part], inv[k:k + part], lo, hi).sort(1).values
        dist.append(t[torch.isfinite(t)])
    dist = torch.cat(dist)
    room = torch.zeros(128 * case["rays"] + 4096, dtype=torch.float64, device=dist.device)
    room[:len(dist)] = dist
    return {"off": None, "ids": None, "dist": room, "box_off": None, "box_ids": None}

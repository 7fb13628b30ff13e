"""The island solve where its chunks have edges: contact chains of 1 to 700 manifolds (around
the 256 manifolds of the two-lane form and of one chunk, the 512 of the one-lane form, and
past it: the per-pass kernel), alone and several together with short islands, bit for bit
against the oracle with the FP64 solve; the FP32 solve repeats itself and stays within the
mixed form's 1e-5 of the FP64 oracle over one step from the same state."""
import numpy as np
import pytest

from test_gpu_parity import _assert_same

pytestmark = pytest.mark.gpu


def _chains(oracle, lengths, seed):
    """Rows of slightly turned unit boxes, each overlapping the next by 2 cm: a row of m + 1
    boxes is an island of m manifolds; rows lie 5 m apart."""
    rng = np.random.default_rng(seed)
    pos, quat = [], []
    for r, m in enumerate(lengths):
        for k in range(m + 1):
            pos.append([0.98 * k, 2.0 + 0.01 * rng.normal(), 5.0 * r + 0.01 * rng.normal()])
            q = np.array([1.0, 0.0, 0.0, 0.0]) + 0.02 * rng.normal(size=4)
            quat.append(q / np.linalg.norm(q))
    n = len(pos)
    return {"shape_offsets": np.array([0, 8], np.uint32), "verts": oracle.box_verts((0.5, 0.5, 0.5)),
            "is_static": np.zeros(n, np.uint8), "shape": np.zeros(n, np.uint32), "pos": np.array(pos),
            "vel": 0.3 * rng.normal(size=(n, 3)), "angvel": np.zeros((n, 3)), "quat": np.array(quat), "mass": np.ones(n),
            "inertia": np.tile(np.eye(3).reshape(9) / 6.0, (n, 1)), "restitution": np.full(n, 0.2),
            "friction": np.full(n, 0.6)}


LENGTHS = [[1], [2], [33], [64], [255], [256], [257], [200, 57], [1] * 300, [120] * 5, [511], [512, 3], [513], [700, 20, 1]]


@pytest.mark.parametrize("lengths", LENGTHS, ids=lambda v: "+".join(map(str, v[:3])) + ("..." if len(v) > 3 else ""))
def test_island_sizes_bitexact(pk, oracle, lengths):
    s = _chains(oracle, lengths, 77)
    o = oracle.OracleWorld(iterations=6, solver_mode=1, flags=pk.FLAG_EPA_GUARD)
    o.load_scene(s)
    g = pk.GpuWorld(iterations=6, flags=pk.FLAG_EPA_GUARD)
    g.load_scene(s)
    mixed = [pk.GpuWorld(iterations=6, flags=pk.FLAG_EPA_GUARD | pk.FLAG_FP32_SOLVE) for _ in range(2)]
    for w in mixed:
        w.load_scene(s)
    rows = 0
    for k in range(4):
        o.step(1 / 120)
        g.step(1 / 120)
        gb, ob = g.bodies(), o.bodies()
        for f in ("pos", "vel", "angvel", "quat", "fat"):
            _assert_same(k, f, gb[f], ob[f])
        (gc, gd), (oc, od) = g.manifolds(), o.manifolds()
        _assert_same(k, "manifold counts", gc, oc)
        _assert_same(k, "manifold data", gd, od)
        _assert_same(k, "colours", g.colours(), o.colours())
        assert g.counters()["colours"] == o.counters()["colours"]
        rows += g.counters()["rows"]
        for w in mixed:
            w.step(1 / 120)
        a, b = (w.bodies() for w in mixed)
        for f in ("pos", "vel", "angvel", "quat"):
            _assert_same(k, "mixed " + f, a[f], b[f])
        if rows and rows == g.counters()["rows"]:  # the first solved step: the same state before it
            assert np.max(np.abs(a["pos"] - ob["pos"]) / np.maximum(np.abs(ob["pos"]), 1.0)) < 1e-5
    assert rows > 0
    for w in [g] + mixed:
        w.close()


def _join(*scenes):
    """Scenes in one, their bodies and shapes in that order."""
    out = {k: np.concatenate([s[k] for s in scenes])
           for k in ("is_static", "pos", "vel", "angvel", "quat", "mass", "inertia", "restitution", "friction", "verts")}
    shapes = np.cumsum([0] + [len(s["shape_offsets"]) - 1 for s in scenes])
    verts = np.cumsum([0] + [len(s["verts"]) for s in scenes])
    out["shape"] = np.concatenate([s["shape"] + np.uint32(k) for s, k in zip(scenes, shapes)]).astype(np.uint32)
    out["shape_offsets"] = np.concatenate([s["shape_offsets"][:-1] + np.uint32(v) for s, v in zip(scenes, verts)] +
                                          [[verts[-1]]]).astype(np.uint32)
    return out


def _turned(s, axis, angle):
    """The scene turned about an axis through the origin, so no contact normal is an axis."""
    u = np.asarray(axis, float) / np.linalg.norm(axis)
    w, v = np.cos(angle / 2), np.sin(angle / 2) * u

    def rot(x):
        t = 2.0 * np.cross(v, x)
        return x + w * t + np.cross(v, t)

    qw, qv = s["quat"][:, 0], s["quat"][:, 1:]
    quat = np.concatenate([(w * qw - qv @ v)[:, None], w * qv + qw[:, None] * v + np.cross(v, qv)], 1)
    return {**s, "pos": rot(s["pos"]), "quat": quat}


def _at(s, x):
    return {**s, "pos": s["pos"] + [x, 0.0, 0.0]}


def _star(oracle, m, seed):
    """A wide plate and m turned boxes on it, 2 cm deep: an island of m manifolds that all share
    the plate, so each has a colour of its own."""
    rng = np.random.default_rng(seed)
    side = int(np.ceil(np.sqrt(m)))
    k = np.arange(m)
    half = 0.8 * side
    pos = np.stack([1.5 * (k % side) - 0.75 * side + 0.75, np.full(m, 2.88), 1.5 * (k // side) - 0.75 * side + 0.75], 1)
    a = rng.uniform(-0.5, 0.5, m)
    quat = np.stack([np.cos(a), 0 * a, np.sin(a), 0 * a], 1)
    n = m + 1

    def part(verts, pos, quat, mass, inertia):
        c = len(pos)
        return {"shape_offsets": np.array([0, 8], np.uint32), "verts": verts, "is_static": np.zeros(c, np.uint8),
                "shape": np.zeros(c, np.uint32), "pos": pos, "vel": 0.2 * rng.normal(size=(c, 3)), "angvel": 0.1 * rng.normal(size=(c, 3)), "quat": quat,
                "mass": np.full(c, mass), "inertia": np.tile(np.eye(3).reshape(9) * inertia, (c, 1)),
                "restitution": np.full(c, 0.2), "friction": np.full(c, 0.6)}

    plate = part(oracle.box_verts((half, 0.5, half)), np.array([[0.0, 2.0, 0.0]]), np.array([[1.0, 0, 0, 0]]), 40.0, 60.0 * half)
    s = _join(plate, part(oracle.box_verts((0.4, 0.4, 0.4)), pos, quat, 1.0, 0.1))
    assert len(s["pos"]) == n
    return _turned(s, (1.0, 2.0, 3.0), 0.7)


@pytest.mark.parametrize("m", [63, 64, 65, 66, 130, 256, 257, 300])
def test_many_colours_bitexact(pk, oracle, m):
    """Islands of 63 to 300 colours: past 64 a colour's number comes from its round."""
    s = _star(oracle, m, m)
    o = oracle.OracleWorld(iterations=5, solver_mode=1, flags=pk.FLAG_EPA_GUARD)
    o.load_scene(s)
    g = pk.GpuWorld(iterations=5, flags=pk.FLAG_EPA_GUARD)
    g.load_scene(s)
    most = 0
    for k in range(4):
        o.step(1 / 120)
        g.step(1 / 120)
        gb, ob = g.bodies(), o.bodies()
        for f in ("pos", "vel", "angvel", "quat"):
            _assert_same(k, f, gb[f], ob[f])
        (gc, gd), (oc, od) = g.manifolds(), o.manifolds()
        _assert_same(k, "manifold counts", gc, oc)
        _assert_same(k, "manifold data", gd, od)
        _assert_same(k, "colours", g.colours(), o.colours())
        assert g.counters()["colours"] == o.counters()["colours"]
        most = max(most, g.counters()["colours"])
    assert most >= m
    g.close()


def _mixed_run(pk, s, steps=4):
    g = pk.GpuWorld(iterations=6, flags=pk.FLAG_EPA_GUARD | pk.FLAG_FP32_SOLVE)
    g.load_scene(s)
    out, colours = [], []
    for _ in range(steps):
        g.step(1 / 120)
        colours.append(g.counters()["colours"])
        b = g.bodies()
        out.append({f: b[f] for f in ("pos", "vel", "angvel", "quat")})
    g.close()
    return out, colours


@pytest.mark.parametrize("stars", [[64], [66], [100], [256], [80] * 5], ids=str)
def test_fp32_rows_of_many_colours(pk, oracle, stars):
    """The FP32 solve keeps the rows of an island of more than 64 colours as they are computed in FP64
    and rounded, in the island kernel as in the per-colour launches, which a long chain far
    away sends the whole scene to; short islands next to it go their own way."""
    parts = [_at(_star(oracle, m, 10 * m + k), 100.0 * (k + 1)) for k, m in enumerate(stars)]
    n = sum(len(p["pos"]) for p in parts)
    got, colours = _mixed_run(pk, _join(*parts))
    if min(stars) > 64:
        assert colours[0] == 0 and colours[1] > 64  # contacts start in the second step
        want, c = _mixed_run(pk, _join(*parts, _at(_chains(oracle, [300], 5), -2000.0)))
        assert c == colours
        # as long as the scene takes the per-colour launches
        for k in range(next((k for k in range(1, 4) if c[k] <= 64), 4)):
            for f in got[k]:
                _assert_same(k, f, got[k][f], want[k][f][:n])
    chains = _chains(oracle, [3] * 40, 6)
    alone, _ = _mixed_run(pk, chains)
    beside, _ = _mixed_run(pk, _join(chains, *parts))
    for k, (a, b) in enumerate(zip(alone, beside)):
        for f in a:
            _assert_same(k, "beside " + f, b[f][:len(a[f])], a[f])

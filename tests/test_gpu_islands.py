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

"""Ray and box queries whose threads share a query's leaves (up to 16,384 rays, 8,192 boxes) and
whose hits are sorted by counting (up to 512 a query) or by radix passes: the oracle's hits
with fewer bodies than threads a query and in worlds of one body, and the same hits on
either side of each line."""
import numpy as np
import pytest

import batched_util as bu
from test_gpu_queries import _random_rays

pytestmark = pytest.mark.gpu


def _scene(pk, n, seed):
    s = pk.scene(pk.SCENE_BOXES, seed, max(n - 1, 1))  # the ground and n - 1 boxes
    if n == 1:
        s = bu.body_range(s, 0, 1)
    rng = np.random.default_rng(seed)
    s["pos"][1:] = rng.uniform(0, 10, size=(n - 1, 3))
    return s, rng


def _boxes(rng, n, half):
    c = rng.uniform(0, 10, size=(n, 3))
    return np.concatenate([c - half, c + half], 1)


@pytest.mark.parametrize("sizes", [[1], [2], [31], [32], [33], [1, 1, 2, 31, 33, 65, 1]], ids=str)
def test_few_bodies(pk, oracle, sizes):
    s, rng = _scene(pk, sum(sizes), 9)
    s["first_body"] = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint32)
    g = pk.GpuWorld(iterations=s["iterations"], flags=s["flags"])
    g.load_scene(s)
    world = None
    if len(sizes) > 1:
        g.set_worlds(s["first_body"])
        world = np.arange(96, dtype=np.uint32) % len(sizes)
    o, d, m = _random_rays(rng, -2.0, 12.0, 96, s["pos"])
    boxes = _boxes(rng, 96, 3.0)
    off, ids, dist = g.raycast(o, d, m, world)
    boff, bids = g.query_aabb(boxes, world)
    g.close()
    for w in range(len(sizes)):
        ws, b0, b1 = bu.world_slice(s, w)
        ow = oracle.OracleWorld(iterations=ws["iterations"], solver_mode=1, flags=ws["flags"])
        ow.load_scene(ws)
        for r in range(w, 96, len(sizes)):
            oi, od = ow.raycast(o[r], d[r], m[r])
            np.testing.assert_array_equal(ids[off[r]:off[r + 1]].astype(np.int64) - b0, oi)
            np.testing.assert_array_equal(dist[off[r]:off[r + 1]], od)
            ob = ow.query_aabb(boxes[r, :3], boxes[r, 3:])
            np.testing.assert_array_equal(bids[boff[r]:boff[r + 1]].astype(np.int64) - b0, ob)


@pytest.mark.parametrize("extra", [0, 1])
@pytest.mark.parametrize("most", ["few", "many"])
def test_either_side_of_the_lines(pk, extra, most):
    s, rng = _scene(pk, 700, 10)
    g = pk.GpuWorld(iterations=s["iterations"], flags=s["flags"])
    g.load_scene(s)
    o, d, m = _random_rays(rng, -2.0, 12.0, 16384 + extra, s["pos"])
    boxes = _boxes(rng, 8192 + extra, 1.0)
    if most == "many":
        boxes[77] = [-50, -50, -50, 50, 50, 50]
    off, ids, dist = g.raycast(o, d, m)
    boff, bids = g.query_aabb(boxes)
    assert (np.diff(boff).max() > 512) == (most == "many")
    for k in range(0, 16384 + extra, 3000):
        e = min(k + 3000, 16384 + extra)
        f, i, t = g.raycast(o[k:e], d[k:e], m[k:e])
        np.testing.assert_array_equal(f, off[k:e + 1] - off[k])
        np.testing.assert_array_equal(i, ids[off[k]:off[e]])
        np.testing.assert_array_equal(t, dist[off[k]:off[e]])
    for k in range(0, 8192 + extra, 3000):
        e = min(k + 3000, 8192 + extra)
        f, i = g.query_aabb(boxes[k:e])
        np.testing.assert_array_equal(f, boff[k:e + 1] - boff[k])
        np.testing.assert_array_equal(i, bids[boff[k]:boff[e]])
    g.close()


@pytest.mark.parametrize("n", [33, 700, 5000])
def test_bodies_without_a_finite_box(pk, n):
    """Bodies whose pose is NaN or infinite and flat static bodies are hits of the same rays and boxes
    whether a query's threads share its leaves or, with more queries, one thread walks the tree
    from its root."""
    s, rng = _scene(pk, n, 11)
    bad = rng.choice(np.arange(1, n), 8, replace=False)
    s["pos"][bad[0]] = np.nan
    s["pos"][bad[1], 1] = np.nan
    s["pos"][bad[2], 0] = np.inf
    s["pos"][bad[3], 2] = -np.inf
    s["quat"][bad[4]] = np.nan
    # flat: a square in the plane y = 0 of the body
    s["shape_offsets"] = np.append(s["shape_offsets"], s["shape_offsets"][-1] + 4).astype(np.uint32)
    s["verts"] = np.concatenate([s["verts"], [[-1.0, 0, -1], [1, 0, -1], [1, 0, 1], [-1, 0, 1]]])
    flat = bad[5:]
    s["shape"][flat] = len(s["shape_offsets"]) - 2
    s["is_static"][flat] = 1
    s["quat"][flat] = [1.0, 0, 0, 0]
    g = pk.GpuWorld(iterations=s["iterations"], flags=s["flags"])
    g.load_scene(s)
    o, d, m = _random_rays(rng, -2.0, 12.0, 2000, s["pos"][np.setdiff1d(np.arange(n), bad)])
    o[:200] = s["pos"][flat[0]] + rng.normal(size=(200, 3)) * [3.0, 0.0, 3.0]
    d[:200] = rng.normal(size=(200, 3))
    d[:200, 1] = rng.choice([0.0, -0.0], 200)
    m[:200] = np.inf
    boxes = _boxes(rng, 1000, 2.0)
    boxes[:10] = [-np.inf, -np.inf, -np.inf, np.inf, np.inf, np.inf]
    boxes[10] = np.nan
    rep, brep = 9, 9  # 18,000 rays and 9,000 boxes: past the lines
    off, ids, dist = g.raycast(np.tile(o, (rep, 1)), np.tile(d, (rep, 1)), np.tile(m, rep))
    boff, bids = g.query_aabb(np.tile(boxes, (brep, 1)))
    f, i, t = g.raycast(o, d, m)
    np.testing.assert_array_equal(f, off[:2001])
    np.testing.assert_array_equal(i, ids[:f[-1]])
    np.testing.assert_array_equal(t, dist[:f[-1]])
    bf, bi = g.query_aabb(boxes)
    np.testing.assert_array_equal(bf, boff[:1001])
    np.testing.assert_array_equal(bi, bids[:bf[-1]])
    g.close()

"""The wavefront-per-pair narrowphase against the oracle, bit for bit, where its layout has
edges: vertex counts around the 32 lanes that search one shape (one vertex per lane up to
32, strides above), equal supports and equal plane distances (axis-aligned boxes on a
grid: heap ties), polytopes past the first stores' faces, and values that are not finite."""
import numpy as np
import pytest

from test_gpu_parity import _assert_same, _oracle_shape

pytestmark = pytest.mark.gpu


def _hull(rng, n):
    v = rng.normal(size=(n, 3))
    return v / np.linalg.norm(v, axis=1, keepdims=True) * rng.uniform(0.3, 0.6, 3)


def _quat(rng):
    q = rng.normal(size=4)
    return q / np.linalg.norm(q)


def _cases(oracle, rng, what):
    if isinstance(what, int):  # meshes of `what` vertices against meshes of 1-70
        return [((2, np.concatenate([rng.normal(size=3) * 0.1, _quat(rng)]), _hull(rng, what)),
                 (2, np.concatenate([rng.normal(size=3) * 0.25, _quat(rng)]), _hull(rng, int(rng.integers(1, 71)))))
                for _ in range(96)]
    box = oracle.box_verts((0.5, 0.5, 0.5))
    out = []
    if what == "grid":
        for d in np.ndindex(4, 4, 4):
            c = np.array(d) * 0.25
            out.append(((2, [0, 0, 0, 1, 0, 0, 0], box), (2, np.concatenate([c, [1, 0, 0, 0]]), box)))
            out.append(((0, [-0.5, -0.5, -0.5, 0.5, 0.5, 0.5], None), (1, np.concatenate([c, [1, 0, 0, 0], [0.5, 0.5, 0.5]]), None)))
    elif what == "faces":  # dense spheres without the generator's vertex order: full scans, long solves
        sph = oracle.sphere_verts(0.5, 16, 32)[::-1].copy()
        for _ in range(24):
            u = rng.normal(size=3)
            out.append(((2, np.concatenate([[0, 0, 0], _quat(rng)]), sph),
                        (2, np.concatenate([u / np.linalg.norm(u) * rng.uniform(0.0, 0.6), _quat(rng)]), sph)))
    else:
        for bad in (np.nan, np.inf, 1e200, 1e308):
            for k in range(3):
                p = np.zeros(3)
                p[k] = bad
                out.append(((2, np.concatenate([p, [1, 0, 0, 0]]), box), (2, [0.1, 0, 0, 1, 0, 0, 0], box)))
                v = box.copy()
                v[k, k] = bad
                out.append(((2, [0, 0, 0, 1, 0, 0, 0], v), (2, [0.1, 0.2, 0, 1, 0, 0, 0], box)))
    return out


@pytest.mark.parametrize("what", [1, 2, 5, 31, 32, 33, 64, 65, "grid", "faces", "not finite"])
def test_batch_edges_bitexact(pk, oracle, what):
    rng = np.random.default_rng(4711)
    cases = _cases(oracle, rng, what)
    print(f"[wave] {what}: {len(cases)} pairs", flush=True)
    g = pk.GpuWorld()
    hit, out = g.gjk_epa_batch([c[0] for c in cases], [c[1] for c in cases])
    g.close()
    for i, (a, b) in enumerate(cases):
        with np.errstate(all="ignore"):
            r = oracle.gjk_epa(_oracle_shape(oracle, a), _oracle_shape(oracle, b))
        if r is None:
            assert hit[i] == 0, i
        elif r == "degenerate":
            assert hit[i] == 2, i
        else:
            assert hit[i] == 1, i
            _assert_same(i, "gjk_epa", out[i], np.concatenate([r["normal"], r["world_a"], r["world_b"], [r["depth"]]]))


@pytest.mark.parametrize("kind, n, steps, flags", [(0, 2, 40, 0), (0, 300, 90, 0), (1, 900, 4, 0), (1, 6000, 3, 0),
                                                   (5, 3000, 12, 0), (3, 8, 30, 96)],
                         ids=["boxes2", "boxes300", "hulls900", "hulls6000", "granular", "batched fp32 filters"])
def test_fused_and_separate_stages_agree(pk, kind, n, steps, flags):
    """Launch shapes that were set keep GJK and EPA in separate kernels; the defaults run a
    wavefront per pair through both where the list is expected to be short. Every step's
    bodies, pairs, manifolds and hit counts are equal, with lists that grow past what the
    step before suggested and lists on both sides of the line."""
    s = pk.scene(kind, 4712, n)
    worlds = []
    for tuned in (False, True):
        g = pk.GpuWorld(iterations=s["iterations"], flags=flags | pk.FLAG_EPA_GUARD)
        g.load_scene(s)
        if len(s["first_body"]) > 2:
            g.set_worlds(s["first_body"])
        if tuned:
            g.set_tuning(2, 64, 0)
        worlds.append(g)
    hits = 0
    for k in range(steps):
        got = []
        for g in worlds:
            g.step(s["dt"])
            b, (c, d) = g.bodies(), g.manifolds()
            got.append([b[f] for f in ("pos", "vel", "angvel", "quat", "fat")] + [g.pairs(), c, d, g.counters()["gjk_hits"]])
        for i, (a, b) in enumerate(zip(*got)):
            _assert_same(k, i, a, b)
        hits += got[0][-1]
    for g in worlds:
        g.close()
    assert hits > 0 or n == 2  # two boxes may not have met yet


def test_list_that_grows_at_once(pk):
    """A step that lists many pairs after one that listed hardly any (bodies set back to a dense
    state): the same contacts as with separate kernels set, in at most twice their time."""
    s = pk.scene(pk.SCENE_HULLS, 4713, 65536)
    ids = np.arange(65536, dtype=np.uint32)
    rest = {"vel": np.zeros((65536, 3)), "angvel": np.zeros((65536, 3)), "quat": s["quat"]}
    ms, out = [], []
    for tuned in (False, True):
        g = pk.GpuWorld(iterations=4, flags=pk.FLAG_EPA_GUARD)
        g.load_scene(s)
        if tuned:
            g.set_tuning(4, 64, 1 << 20)
        took = []
        for _ in range(4):
            g.set_state(ids, pos=30.0 * s["pos"], **rest)
            g.step(s["dt"], 2)
            assert g.counters()["gjk_listed"] < 1000
            g.set_state(ids, pos=s["pos"], **rest)
            t = g.step_timed(s["dt"], 1)
            took.append(t["gjk"] + t["epa"])
        c = g.counters()
        assert c["gjk_listed"] > 50000
        out.append((g.pairs(), *g.manifolds(), g.bodies()["pos"], c["gjk_hits"]))
        ms.append(min(took))
        g.close()
    for i, (a, b) in enumerate(zip(*out)):
        _assert_same("dense", i, a, b)
    print(f"[wave] dense step: default {ms[0]:.3f} ms, separate kernels {ms[1]:.3f} ms", flush=True)
    assert ms[0] <= 2.0 * ms[1]


def test_lists_longer_than_a_launch(pk, monkeypatch):
    """Lists of more wavefronts than one launch can count (2^25) go in several: with 97 a launch (read
    from PKG_WAVE_LAUNCH when a context is created) the batch and a step's EPA, reruns of
    overflows among them, give what single launches give."""
    rng = np.random.default_rng(4714)
    pairs = [((2, np.concatenate([rng.normal(size=3) * 0.1, _quat(rng)]), _hull(rng, int(rng.integers(1, 40)))),
              (2, np.concatenate([rng.normal(size=3) * 0.3, _quat(rng)]), _hull(rng, int(rng.integers(1, 40)))))
             for _ in range(400)]
    sph = pk.mesh.sphere(0.5, 16, 32).vertices
    n = 400  # deep pairs of spheres, each far from the others: all hit, some past 192 faces
    u = rng.normal(size=(n // 2, 3))
    u *= rng.uniform(0.05, 0.6, (n // 2, 1)) / np.linalg.norm(u, axis=1, keepdims=True)
    a = np.stack([5.0 * (np.arange(n // 2) % 20), np.zeros(n // 2), 5.0 * (np.arange(n // 2) // 20)], 1)
    s = {"shape_offsets": np.array([0, len(sph)], np.uint32), "verts": sph, "is_static": np.zeros(n, np.uint8),
         "shape": np.zeros(n, np.uint32), "pos": np.stack([a, a + u], 1).reshape(n, 3), "vel": np.zeros((n, 3)),
         "angvel": np.zeros((n, 3)), "quat": np.array([_quat(rng) for _ in range(n)]), "mass": np.ones(n),
         "inertia": np.tile(np.eye(3).reshape(9) * 0.1, (n, 1)), "restitution": np.full(n, 0.5), "friction": np.full(n, 0.5)}
    got = []
    for per in (None, "97", "1"):
        if per:
            monkeypatch.setenv("PKG_WAVE_LAUNCH", per)
        g = pk.GpuWorld(iterations=4, flags=pk.FLAG_ALL_MOVED | pk.FLAG_NO_SOLVER | pk.FLAG_NO_INTEGRATE)
        g.load_scene(s)
        g.set_tuning(2, 64, 1 << 20)
        g.step(1 / 60)
        c = g.counters()
        assert c["gjk_hits"] == n // 2 and c["epa_overflow"] > 0
        got.append((*g.manifolds(), *g.gjk_epa_batch([p[0] for p in pairs], [p[1] for p in pairs])))
        g.close()
    for other in got[1:]:
        for i, (x, y) in enumerate(zip(got[0], other)):
            _assert_same("launches", i, y, x)

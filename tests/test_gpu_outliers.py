"""Bodies far outside the bulk of a scene (which the LBVH's Morton grid cuts off) change
neither pairs nor bodies nor manifolds: bit for bit against the oracle, with body counts
around the grid's 1,024-body sample and outliers up to infinity and NaN."""
import numpy as np
import pytest

from test_gpu_parity import _assert_same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, far", [(1, 1e4), (63, 1e6), (64, 1e13), (300, -1e4), (1023, 1e9), (1024, np.inf), (1500, np.nan),
                                    (2500, 1e300)])
def test_outliers_bitexact(pk, oracle, n, far):
    s = pk.scene(pk.SCENE_BOXES, 515, n)
    rng = np.random.default_rng(n)
    s["pos"][:, 1] *= 0.2  # denser: contacts in the first steps
    out = rng.choice(np.arange(1, n + 1), size=max(1, n // 100), replace=False)
    s["pos"][out, rng.integers(0, 3, len(out))] = far
    o = oracle.OracleWorld(iterations=s["iterations"], solver_mode=1, flags=s["flags"] | pk.FLAG_EPA_GUARD)
    o.load_scene(s)
    g = pk.GpuWorld(iterations=s["iterations"], flags=s["flags"] | pk.FLAG_EPA_GUARD)
    g.load_scene(s)
    for k in range(6):
        o.step(s["dt"])
        g.step(s["dt"])
        gb, ob = g.bodies(), o.bodies()
        for f in ("pos", "vel", "angvel", "quat", "fat"):
            _assert_same(k, f, gb[f], ob[f])
        _assert_same(k, "pairs", g.pairs(), o.pairs())
        (gc, gd), (oc, od) = g.manifolds(), o.manifolds()
        _assert_same(k, "manifold counts", gc, oc)
        _assert_same(k, "manifold data", gd, od)
    g.close()

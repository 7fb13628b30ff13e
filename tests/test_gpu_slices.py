"""The pair query, whose threads share a query's leaves in scenes of up to 24,576 bodies:
the same pairs, bit for bit, as the oracle, with fewer leaves than threads a query, worlds
of one body, and either side of that line."""
import numpy as np
import pytest

import batched_util as bu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[2], [3], [15], [16], [17], [33], [1, 1, 2, 15, 16, 17, 1, 33, 100], [24576], [24577],
                                   [24500, 1, 2, 73], [24500, 1, 2, 74]], ids=str)
def test_pairs_equal_the_oracle(pk, oracle, sizes):
    n = sum(sizes)
    s = pk.scene(pk.SCENE_BOXES, 61, n - 1)
    s["flags"] |= pk.FLAG_NO_SOLVER
    s["first_body"] = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint32)
    rng = np.random.default_rng(n)
    side = 0.8 * n ** (1 / 3)
    s["pos"][1:] = rng.uniform(0, side, size=(n - 1, 3)) + [0, 0.5, 0]
    g = pk.GpuWorld(iterations=s["iterations"], flags=s["flags"])
    g.load_scene(s)
    if len(sizes) > 1:
        g.set_worlds(s["first_body"])
    worlds = []
    for w in range(len(sizes)):
        ws, b0, b1 = bu.world_slice(s, w)
        o = oracle.OracleWorld(iterations=ws["iterations"], solver_mode=1, flags=ws["flags"])
        o.load_scene(ws)
        worlds.append((o, b0, b1))
    found = 0
    for k in range(2):
        g.step(s["dt"])
        keys = g.pairs()
        for o, b0, b1 in worlds:
            o.step(s["dt"])
            local, _ = bu.keys_in(keys, b0, b1)
            np.testing.assert_array_equal(local, o.pairs(), err_msg=f"step {k} bodies {b0}..{b1}")
            found += len(local)
    g.close()
    assert found > 0 or n < 16

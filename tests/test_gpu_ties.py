"""EPA where several live faces are equally near: the face taken is the one that the order of
the heap's operations gives, from the first tetrahedron or many expansions on. Unrotated
spheres and boxes on a grid, bit for bit against the oracle."""
import numpy as np
import pytest

from test_gpu_parity import _assert_same, _oracle_shape

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stacks, sectors", [(2, 4), (4, 4), (4, 8), (8, 8), (8, 16), (16, 32)])
def test_equal_distances_bitexact(pk, oracle, stacks, sectors):
    one = [1, 0, 0, 0]
    sph = oracle.sphere_verts(0.5, stacks, sectors)
    box = oracle.box_verts((0.5, 0.5, 0.5))
    cases = []
    for d in np.ndindex(4, 4, 4):
        c = np.concatenate([np.array(d) * 0.2, one])
        cases.append(((2, [0, 0, 0] + one, sph), (2, c, sph)))
        cases.append(((2, [0, 0, 0] + one, box), (2, c, sph)))
    g = pk.GpuWorld()
    hit, out = g.gjk_epa_batch([c[0] for c in cases], [c[1] for c in cases])
    g.close()
    for i, (a, b) in enumerate(cases):
        r = oracle.gjk_epa(_oracle_shape(oracle, a), _oracle_shape(oracle, b))
        if r is None:
            assert hit[i] == 0, i
        elif r == "degenerate":
            assert hit[i] == 2, i
        else:
            assert hit[i] == 1, i
            _assert_same(i, "gjk_epa", out[i], np.concatenate([r["normal"], r["world_a"], r["world_b"], [r["depth"]]]))

"""The FP64 M2L's two tile shapes against each other, and rows that a launch
does not hold at once (the shapes and parts by the rules of csrc/m2l_plan.hpp)."""
import numpy as np
import pytest

import m2l_plan
from scalfmm_amd import Engine
from scalfmm_amd.distributions import plummer, uniform_cube

pytestmark = pytest.mark.gpu
CENTER = (0.5, 0.5, 0.5)


@pytest.mark.parametrize("p", [5, 6, 7, 8])
def test_tile_shapes_same_bits(p):
    """Sets alone (one column tile per workgroup) and together (two): the same
    bits, since a target's terms are added in the same order."""
    x, y, z, q = uniform_cube(25503, 23)
    off = [0, 8001, 16502, 25503]
    e = Engine(6, 1.0, CENTER, p)
    e.set_particle_sets(off, x, y, z, q)
    e.build_tree()
    assert m2l_plan.two_tiles(sum(e.tree_info().n_cells))
    e.evaluate()
    got = e.results()
    e.close()
    e = Engine(6, 1.0, CENTER, p)
    for a, b in zip(off, off[1:]):
        e.set_particles(x[a:b], y[a:b], z[a:b], q[a:b])
        e.build_tree()
        assert not m2l_plan.two_tiles(sum(e.tree_info().n_cells))
        e.evaluate()
        for g, r in zip(got, e.results()):
            assert np.array_equal(g[a:b], r)
    e.close()


@pytest.mark.parametrize("order", [6, 7, 8])
@pytest.mark.parametrize("dist,n,h,two", [(uniform_cube, 3001, 4, False), (plummer, 2003, 5, False), (uniform_cube, 20003, 5, True)])
def test_rows_in_parts(oracle, dist, n, h, two, order):
    """At epsilon 5e-9 the ranks sum to more rows than a launch holds: the second
    part continues from the partial locals of the first.  Against the oracle with
    the same epsilon, 1e-12 relative L2 (the FP64 path's bound)."""
    eps = 5e-9
    x, y, z, q = dist(n, 37)
    e = Engine(h, 1.0, CENTER, order, epsilon=eps)
    e.set_particles(x, y, z, q)
    e.build_tree()
    assert m2l_plan.two_tiles(sum(e.tree_info().n_cells)) == two
    rank = []  # per offset |pos|; its operator is that of the sorted offset
    for v in np.ndindex(4, 4, 4):
        if max(v) > 1:
            a, b, c = sorted(v, reverse=True)
            rank.append(e.operator(((a + 3) * 7 + b + 3) * 7 + c + 3)[0].shape[1])
    assert len(m2l_plan.rows(rank)[3]) - 1 > 116
    e.evaluate()
    ref = oracle.fmm(x, y, z, q, CENTER, 1.0, h, order, epsilon=eps)
    for a, b in zip(e.results(), ref[:4]):
        assert np.linalg.norm(a - b) < 1e-12 * np.linalg.norm(b)
    e.close()

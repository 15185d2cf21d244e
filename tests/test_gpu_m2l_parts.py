"""The FP64 M2L's two tile shapes against each other (which one a tree takes is
csrc/m2l_plan.hpp's rule)."""
import numpy as np
import pytest

import m2l_plan
from scalfmm_amd import Engine
from scalfmm_amd.distributions import uniform_cube

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

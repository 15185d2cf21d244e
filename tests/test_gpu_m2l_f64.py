"""The FP64 M2L at the edges of its tiles against the oracle: fewer cells than a
column tile, partly filled tiles, both tile shapes (by the number of
cells), every order, and sparse trees whose tiles skip offsets.  Locals and
results to 1e-12 relative L2, the bound of the FP64 path."""
import numpy as np
import pytest

from oracle import pyoracle
from scalfmm_amd import Engine
from scalfmm_amd.distributions import plummer, uniform_cube

pytestmark = pytest.mark.gpu
CENTER = (0.5, 0.5, 0.5)

CASES = [
    (uniform_cube, 9, 3, 5),  # a handful of cells
    (uniform_cube, 700, 4, 6),  # 585 cells at most: one partly filled tile of the last workgroup
    (uniform_cube, 701, 4, 7),
    (uniform_cube, 3001, 4, 8),
    (plummer, 20011, 6, 5),  # sparse: tiles without some of the offsets
    (plummer, 20011, 7, 7),
    (uniform_cube, 45001, 6, 5),  # 18,000 cells and more: two column tiles per workgroup
    (uniform_cube, 45001, 6, 6),
    (uniform_cube, 45001, 6, 7),
    (uniform_cube, 45001, 6, 8),
]


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("dist,n,h,p", CASES)
def test_m2l_tiles(dist, n, h, p):
    x, y, z, q = dist(n, 17)
    e = Engine(h, 1.0, CENTER, p)
    e.set_particles(x, y, z, q)
    e.build_tree()
    e.evaluate()
    ref = pyoracle.fmm(x, y, z, q, CENTER, 1.0, h, p)
    for got, want in zip(e.results(), ref[:4]):
        assert rel(got, want) < 1e-12
    e.close()


def test_m2l_tile_shapes_agree():
    """A set alone (one column tile per workgroup) and among others (two): the
    same bits, since a target's terms are added in the same order."""
    x, y, z, q = uniform_cube(36003, 23)
    for p in (5, 7):
        e = Engine(6, 1.0, CENTER, p)
        off = [0, 12001, 24002, 36003]
        e.set_particle_sets(off, x, y, z, q)
        e.build_tree()
        e.evaluate()
        got = e.results()
        e.close()
        e = Engine(6, 1.0, CENTER, p)
        for a, b in zip(off, off[1:]):
            e.set_particles(x[a:b], y[a:b], z[a:b], q[a:b])
            e.build_tree()
            assert sum(e.tree_info().n_cells) < 16384  # the other tile shape
            e.evaluate()
            for g, r in zip(got, e.results()):
                assert np.array_equal(g[a:b], r)
        e.close()


@pytest.mark.parametrize("p", [7, 8])
def test_m2l_wide_addresses_agree(p):
    """Compressed expansions within 4 GB (each set alone) and beyond (64-bit
    addresses): the same bits."""
    x, y, z, q = uniform_cube(130003, 29)
    off = [0, 35001, 75002, 130003]
    e = Engine(7, 1.0, CENTER, p)
    e.set_particle_sets(off, x, y, z, q)
    e.build_tree()
    e.evaluate()
    got = e.results()
    a, b = off[0], off[1]
    e.close()
    e = Engine(7, 1.0, CENTER, p)
    e.set_particles(x[a:b], y[a:b], z[a:b], q[a:b])
    e.build_tree()
    e.evaluate()
    for g, r in zip(got, e.results()):
        assert np.array_equal(g[a:b], r)
    e.close()

"""The device tree at the edges of its tiles (2,048 particles, 32 cells), on
shallow, deep and clustered sets, and on levels above and below the dense key
tables: keys, permutation, cells, leaf ranges and lists equal the oracle's bit
for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,h,spread", [(1, 3, 1.0), (31, 4, 1.0), (2047, 5, 1.0), (2048, 6, 0.1), (2049, 4, 1.0),
                                        (4097, 8, 0.01), (20481, 10, 0.3), (3000, 12, 0.001)])
def test_tree_tiles(oracle, n, h, spread):
    from scalfmm_amd import Engine
    rng = np.random.default_rng(n)
    p = 0.5 + (rng.random((3, n)) - 0.5) * spread
    p[:, : n // 3] = rng.random((3, n // 3))
    x, y, z = (p[d].copy() for d in range(3))
    e = Engine(h, 1.0, (0.5, 0.5, 0.5), 5)
    e.set_particles(x, y, z, np.ones(n))
    e.build_tree()
    t = oracle.Tree(x, y, z, [0.5, 0.5, 0.5], 1.0, h)
    for a, b in zip(e.sorted_keys(), t.sorted()):
        assert np.array_equal(a, b)
    for a, b in zip(e.leaf_ranges(), t.leaf_ranges()):
        assert np.array_equal(a, b)
    for a, b in zip(e.p2p_list(), t.p2p_list()):
        assert np.array_equal(a, b)
    for level in range(2, h):
        assert np.array_equal(e.cell_keys(level), t.cell_keys(level)), level
        for a, b in zip(e.m2l_list(level), t.m2l_list(level)):
            assert np.array_equal(a, b), level
    e.close()

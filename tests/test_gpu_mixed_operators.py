"""Which operators a mixed context holds: from order 6 the FP64 products run
unless a tile shape is set, and the bfloat16 tiles' operators (a position's planes,
tens of MB) are made where one is."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _free():
    from scalfmm_amd import _abi
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert _abi.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("hilo", [False, True])
@pytest.mark.parametrize("order", [6, 8])
def test_tiles_operators_where_a_shape_is_set(tmp_path, order, hilo):
    from scalfmm_amd import PRECISION_MIXED, PRECISION_MIXED_HILO, Engine
    from scalfmm_amd.distributions import uniform_cube
    x, y, z, q = uniform_cube(3000, 8)
    planes = 316 * 6 * 16 * order ** 3 * 2  # at rank 16 for every position: less than there are

    def engine():
        return Engine(4, 1.0, (0.5, 0.5, 0.5), order, precision=PRECISION_MIXED_HILO if hilo else PRECISION_MIXED)

    def results(e):
        e.set_particles(x, y, z, q)
        e.build_tree()
        e.evaluate()
        return e.results()

    results(engine())  # whatever the process takes once
    before = _free()
    e = engine()
    products = results(e)
    used = before - _free()
    e.set_m2l_variant(0)
    assert before - _free() >= used + planes
    tiles = results(e)
    # a shape set first, operators loaded again, and back to the products
    f = engine()
    f.set_m2l_variant(0)
    for a, b in zip(results(f), tiles):
        assert np.array_equal(a, b)
    f.save_operators(tmp_path / "ops")
    f.load_operators(tmp_path / "ops")
    for a, b in zip(results(f), products):
        assert np.array_equal(a, b)
    f.set_m2l_variant(0)
    for a, b in zip(results(f), tiles):
        assert np.array_equal(a, b)
    e.set_m2l_variant(-1)
    for a, b in zip(results(e), products):
        assert np.array_equal(a, b)
    e.close()
    f.close()

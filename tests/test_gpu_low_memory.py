"""Evaluations where other programs hold the device's memory."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
CENTER = (0.5, 0.5, 0.5)


def test_products_prepared_again_after_a_failure():
    """The FP64 products' operators (15 MB at order 8) find no memory on their
    first use: that evaluation fails, and the next one, with the memory back,
    prepares them again."""
    from device_memory import all_but
    from scalfmm_amd import PRECISION_MIXED, Engine, FmmError, _abi
    from scalfmm_amd.distributions import uniform_cube
    x, y, z, q = uniform_cube(3001, 5)

    def engine():
        e = Engine(4, 1.0, CENTER, 8, precision=PRECISION_MIXED)
        e.set_particles(x, y, z, q)
        e.build_tree()
        return e

    ref = engine()
    ref.set_m2l_variant(4)
    ref.evaluate()
    e = engine()
    e.set_m2l_variant(0)
    e.evaluate()  # every other buffer
    e.synchronize()
    e.set_m2l_variant(4)
    with all_but(0) as left:
        print("left", left, flush=True)
        with pytest.raises(FmmError) as err:
            e.evaluate()
        assert err.value.code == _abi.ERR_NOMEM
    e.evaluate()
    for a, b in zip(e.results(), ref.results()):
        assert np.array_equal(a, b)
    e.close()
    ref.close()


@pytest.mark.parametrize("n,h,order,cells,left", [(60000, 6, 7, (28000, 37449), 900 << 20), (9000, 6, 8, (8193, 12288), 300 << 20),
                                                  (60000, 6, 5, (28000, 37449), 400 << 20)])
def test_fp64_m2l_with_little_memory(n, h, order, cells, left):
    """The compressed expansions (0.6 to 1.3 GB here) find less memory than
    they would take: the rows run in parts, with the same bits, and all at once
    again when the memory is back."""
    from device_memory import all_but
    from scalfmm_amd import Engine, FFmmM2L, FFmmNearAndFarFields
    from scalfmm_amd.distributions import uniform_cube
    x, y, z, q = uniform_cube(n, 7)

    def engine():
        e = Engine(h, 1.0, CENTER, order)
        e.set_particles(x, y, z, q)
        e.build_tree()
        assert cells[0] <= sum(e.tree_info().n_cells) <= cells[1]  # the tile shape
        return e

    e = engine()
    e.evaluate()
    ref = e.results()
    e.close()
    e = engine()
    e.evaluate(FFmmNearAndFarFields & ~FFmmM2L)  # every other buffer
    e.synchronize()
    with all_but(left) as free:
        print("left", free, flush=True)
        for _ in range(2):
            e.evaluate()
            for a, b in zip(e.results(), ref):
                assert np.array_equal(a, b)
    e.build_tree()
    e.evaluate()
    for a, b in zip(e.results(), ref):
        assert np.array_equal(a, b)
    e.close()


def test_near_field_leaves_room_for_the_expansions():
    """The slots of the near field (80 MB) would fit a quarter of the free
    memory, but not beside the expansions (270 MB) and what the M2L needs at the
    least (160 MB): the pairs are taken one way instead, within the FP64 path's 1e-12."""
    from device_memory import all_but
    from scalfmm_amd import Engine
    from scalfmm_amd.distributions import uniform_cube
    x, y, z, q = uniform_cube(90000, 7)
    for a in (x, y, z):  # eight leaves of 3,750 particles
        a[:30000] = 0.5 + (a[:30000] - 0.5) / 16

    def engine(h):
        e = Engine(h, 1.0, CENTER, 8)
        e.set_particles(x, y, z, q)
        return e

    e = engine(6)
    e.build_tree()
    e.evaluate()
    ref = e.results()
    e.close()
    e = engine(6)
    e.synchronize()
    with all_but(490 << 20) as left:
        print("left", left, flush=True)
        e.build_tree()
        e.evaluate()
        got = e.results()
    for a, b in zip(got, ref):
        assert np.linalg.norm(a - b) <= 1e-12 * np.linalg.norm(b)
    e.close()

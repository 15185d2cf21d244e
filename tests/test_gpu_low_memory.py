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
    with all_but(4 << 20) as left:
        print("left", left, flush=True)
        with pytest.raises(FmmError) as err:
            e.evaluate()
        assert err.value.code == _abi.ERR_NOMEM
    e.evaluate()
    for a, b in zip(e.results(), ref.results()):
        assert np.array_equal(a, b)
    e.close()
    ref.close()

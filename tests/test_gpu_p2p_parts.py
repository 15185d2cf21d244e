"""The FP64 near field of the big leaves with work items in 1 to 32 parts beside
each other, one or several charge vectors: against the oracle's near field (1e-12
relative L2, the bound of the FP64 path), and the same bits again."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nrhs", [1, 3])
@pytest.mark.parametrize("sizes", [[70, 5000, 300, 2000, 64, 1, 9000, 700], [65, 0, 0, 0, 0, 0, 0, 0], [4097, 0, 66, 0, 0, 0, 0, 257]])
def test_items_in_parts(oracle, sizes, nrhs):
    from scalfmm_amd import Engine, FFmmNearField
    rng = np.random.default_rng(9)
    pts = []
    for m, cnt in enumerate(sizes):  # the eight leaves of a cell of height 3
        ix, iy, iz = oracle.demorton(m)
        pts.append((np.array([ix, iy, iz]) + 0.01 + 0.98 * rng.random((cnt, 3))) / 4.0)
    p = np.concatenate(pts)
    x, y, z = (p[:, d].copy() for d in range(3))
    q = 2.0 * rng.random((nrhs, len(x))) - 1.0
    e = Engine(3, 1.0, (0.5, 0.5, 0.5), 5)
    e.set_particle_sets([0, len(x)], x, y, z, q)
    for _ in range(2):
        e.build_tree()
        e.evaluate(FFmmNearField)
        got = [np.atleast_2d(a).copy() for a in e.results()]
        e.evaluate(FFmmNearField)
        assert all(np.array_equal(a, np.atleast_2d(b)) for a, b in zip(got, e.results()))
        for r in range(nrhs):
            ref = oracle.fmm(x, y, z, q[r], (0.5, 0.5, 0.5), 1.0, 3, 5, ops=FFmmNearField)
            for a, b in zip(got, ref[:4]):
                assert np.linalg.norm(a[r] - b) <= 1e-12 * np.linalg.norm(b)
    e.close()

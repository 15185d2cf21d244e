"""The FP64 near field of the big leaves, each unordered pair once, at the edges
of its work items: leaves of one to four targets per lane, one particle past an
item or a chunk of 64 sources, small leaves between them.  Against the oracle's
near field (1e-12 relative L2, the bound of the FP64 path) and the ordered-pair
kernel; the same bits on repeated evaluations."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

H = 3
SIZES = [65, 64, 128, 129, 1, 191, 192, 193, 255, 256, 257, 3, 300, 511, 513, 70, 66, 64, 127, 1, 320, 2, 0, 100]


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("ops", ["near", "all"])
def test_f64_mutual_p2p(oracle, ops):
    from scalfmm_amd import Engine, FFmmNearAndFarFields, FFmmNearField
    rng = np.random.default_rng(5)
    pts = []
    for m, cnt in enumerate(SIZES):  # consecutive Morton leaves of width 1/4
        ix, iy, iz = oracle.demorton(m)
        pts.append((np.array([ix, iy, iz]) + 0.01 + 0.98 * rng.random((cnt, 3))) / 4.0)
    p = np.concatenate(pts)
    x, y, z = (p[:, d].copy() for d in range(3))
    q = 2.0 * rng.random(len(x)) - 1.0
    bits = FFmmNearField if ops == "near" else FFmmNearAndFarFields
    ref = oracle.fmm(x, y, z, q, (0.5, 0.5, 0.5), 1.0, H, 5, ops=bits)
    out = {}
    for mutual in (True, False):
        e = Engine(H, 1.0, (0.5, 0.5, 0.5), 5)
        e.set_p2p_mutual(mutual)
        e.set_particles(x, y, z, q)
        e.build_tree()
        e.evaluate(bits)
        out[mutual] = e.results()
        for a, b in zip(out[mutual], ref[:4]):
            assert _rel(a, b) <= 1e-12
        e.evaluate(bits)
        assert all(np.array_equal(a, b) for a, b in zip(e.results(), out[mutual]))
        e.close()
    for a, b in zip(out[True], out[False]):
        assert _rel(a, b) <= 1e-12


def test_last_leaf_reads_clean_padding(oracle):
    """The masked sources past a big last leaf read the padding of the sorted
    arrays: finite results also where that memory held NaN before."""
    from scalfmm_amd import Engine, FFmmNearField
    rng = np.random.default_rng(6)
    n = 1021
    x, y, z = 0.75 + 0.24 * rng.random((3, n))  # one leaf
    q = 2.0 * rng.random(n) - 1.0
    ref = oracle.fmm(x, y, z, q, (0.5, 0.5, 0.5), 1.0, H, 5, ops=FFmmNearField)
    for mutual in (True, False):
        for charges in (np.full(n, np.nan), q):
            e = Engine(H, 1.0, (0.5, 0.5, 0.5), 5)
            e.set_p2p_mutual(mutual)
            # the arrays of 4 more particles hold NaN where the next ones have their padding
            extra = 4 if np.isnan(charges[0]) else 0
            e.set_particles(*(np.concatenate([a, a[:extra]]) for a in (x, y, z)), np.concatenate([charges, charges[:extra]]))
            e.build_tree()
            e.evaluate(FFmmNearField)
            got = e.results()
            if extra:  # the same context again, on the buffers it has
                e.set_particles(x, y, z, q)
                e.build_tree()
                e.evaluate(FFmmNearField)
                got = e.results()
            e.close()
            for a, b in zip(got, ref[:4]):
                assert _rel(a, b) <= 1e-12

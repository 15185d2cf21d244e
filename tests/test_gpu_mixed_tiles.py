"""The bfloat16 M2L tiles at orders 7 and 8 on the reference's fixture and on
clustered sets.  A context that sets no shape runs the FP64 products there, so the
shapes are set; tolerances as in test_gpu_mixed.py."""
import numpy as np
import pytest

from test_gpu_mixed import FORCE_TOL, POT_TOL, _check, _mixed, _rel, _say, plummer100k  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", [0, 3])
@pytest.mark.parametrize("ops_name", ["far", "all"])
def test_tiles_fixture_order7(oracle, fixture20k, ops_name, variant):
    from scalfmm_amd import FFmmFarField, FFmmNearAndFarFields
    ops = {"far": FFmmFarField, "all": FFmmNearAndFarFields}[ops_name]
    f = fixture20k
    x, y, z, q = (f["data"][:, k].copy() for k in range(4))
    e = _mixed(5, 7)
    e.set_m2l_variant(variant)
    e.set_particles(x, y, z, q)
    e.build_tree()
    e.evaluate(ops)
    assert e.m2l_variant()[0] == variant
    _check(e.results(), oracle.fmm(x, y, z, q, f["center"], f["width"], 5, 7, ops=ops))
    e.close()


@pytest.mark.parametrize("ops_name", ["far", "all"])
def test_tiles_plummer_order8(oracle, plummer100k, ops_name):  # noqa: F811
    from scalfmm_amd import FFmmFarField, FFmmNearAndFarFields
    ops = {"far": FFmmFarField, "all": FFmmNearAndFarFields}[ops_name]
    d = plummer100k
    x, y, z, q = d["xyzq"]
    ref = oracle.fmm(x, y, z, q, (0.5, 0.5, 0.5), 1.0, d["h"], d["p"], ops=ops)
    for variant in (0, 3):
        e = _mixed(d["h"], d["p"])
        e.set_m2l_variant(variant)
        e.set_particles(x, y, z, q)
        e.build_tree()
        e.evaluate(ops)
        got = e.results()
        _check(got, ref)
        if ops_name == "all":
            t = np.sort(np.random.default_rng(3).choice(d["n"], 500, replace=False))
            assert _rel(got[0][t], oracle.direct(x, y, z, q, targets=t)[0]) <= 1e-6
        e.close()


def test_tiles_plummer10m_order8():
    """Ten million clustered particles, shape 0, against the FP64 form."""
    from scalfmm_amd import Engine
    from scalfmm_amd.distributions import plummer
    _say("plummer 10M: generating (seed 2)")
    x, y, z, q = plummer(10_000_000, 2)
    out = []
    for variant in (None, 0):
        e = Engine(8, 1.0, (0.5, 0.5, 0.5), 8) if variant is None else _mixed(8, 8)
        if variant is not None:
            e.set_m2l_variant(variant)
        e.set_particles(x, y, z, q)
        e.build_tree()
        e.evaluate()
        out.append(e.results())
        e.close()
        _say(f"  evaluated: shape {variant}")
    d = [_rel(a, b) for a, b in zip(out[1], out[0])]
    _say(f"  pot {d[0]:.3e} F {max(d[1:]):.3e}")
    assert d[0] <= POT_TOL and max(d[1:]) <= FORCE_TOL, d

"""The equispaced (Fourier space) M2L where parents have few children, many, and
both in one tree, against the oracle (1e-12 relative L2, as test_gpu_uniform.py)."""
import functools

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
C = (0.5, 0.5, 0.5)


def points(kind, n):
    rng = np.random.default_rng(n)
    if kind == "sphere":
        v = rng.normal(size=(3, n))
        p = 0.5 + 0.49 * v / np.linalg.norm(v, axis=0)
    elif kind == "line":
        p = np.stack((rng.random(n), 0.5 + 1e-3 * rng.random(n), 0.5 + 1e-3 * rng.random(n)))
    else:
        p = rng.random((3, n))
    return (*(a.copy() for a in p), 2 * rng.random(n) - 1)


@functools.lru_cache(maxsize=1)
def operators(oracle, order):
    return oracle.ChebGlobal(order, uniform=True)


CASES = [("uniform", 1, 4, False), ("uniform", 300, 6, False), ("sphere", 1003, 6, False), ("line", 700, 7, False),
         ("uniform", 2501, 5, False), ("uniform", 5001, 5, True), ("uniform", 5003, 6, False)]


@pytest.mark.parametrize("order,kind,n,h,many", [(p, *c) for p in (5, 6, 7, 8) for c in CASES if c[1] <= (6000, 6000, 1100, 800)[p - 5]])
def test_few_and_many_children(oracle, order, kind, n, h, many):
    from scalfmm_amd import Engine, _abi
    x, y, z, q = points(kind, n)
    e = Engine(h, 1.0, C, order)
    e.set_m2l_scheme(_abi.M2L_UNIFORM)
    e.set_particles(x, y, z, q)
    e.build_tree()
    cells = e.tree_info().n_cells
    assert (cells[h - 1] >= 5 * cells[h - 2]) == many
    e.evaluate()
    ref = oracle.fmm_global(operators(oracle, order), x, y, z, q, C, 1.0, h)
    for a, b in zip(e.results(), ref[:4]):
        assert np.linalg.norm(a - b) <= 1e-12 * np.linalg.norm(b)
    e.close()

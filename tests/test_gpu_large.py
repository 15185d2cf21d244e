"""Sizes at which a kernel needs more threads than one dimension of a launch
holds (2^32)."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu

N, H = (1 << 29) + 4099, 9


def test_near_field_beyond_2_29_particles():
    """Eight lanes per particle.  The near field of a few targets, the last of the
    Morton order among them, against sums over their 27 leaves (1e-12, the FP64
    path's bound)."""
    import torch
    from scalfmm_amd import Engine, FFmmNearField
    if torch.cuda.mem_get_info()[0] < 220 << 30:
        pytest.skip("needs 220 GiB of device memory")
    g = torch.Generator(device="cuda")
    g.manual_seed(11)
    pos = [torch.rand(N, generator=g, device="cuda", dtype=torch.float64) for _ in range(3)]
    q = torch.rand(N, generator=g, device="cuda", dtype=torch.float64)
    for d in range(3):  # some in the last leaf of the Morton order
        pos[d][N - 3:] = 1 - torch.tensor([1e-3, 2e-3, 3e-3], dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    e = Engine(H, 1.0, (0.5, 0.5, 0.5), 5)
    e.set_particles_device(N, *(a.data_ptr() for a in (*pos, q)))
    e.build_tree()
    e.evaluate(FFmmNearField)
    e.synchronize()
    p = ctypes.c_void_p()
    assert e._L.hfmm_get_results_device(e.h, ctypes.byref(p), None, None, None) == 0

    class Block:
        __cuda_array_interface__ = {"data": (p.value, False), "shape": (N,), "typestr": "<f8", "version": 3}

    got = torch.as_tensor(Block(), device="cuda")
    leaves = 1 << (H - 1)
    for i in (0, N // 2, N - 4, N - 3, N - 2, N - 1):
        near = torch.ones(N, dtype=torch.bool, device="cuda")
        for a in pos:
            near &= (torch.floor(a * leaves) - torch.floor(a[i] * leaves)).abs() <= 1
        near[i] = False
        at = near.nonzero()[:, 0]
        r2 = sum((a[at] - a[i]) ** 2 for a in pos)
        want = (q[at] / r2.sqrt()).sum()
        assert len(at) > 100
        assert abs(float(got[i] - want)) <= 1e-12 * float(want), i
    e.close()
    del got, pos, q, near, at
    torch.cuda.empty_cache()


def test_mixed_multipoles_beyond_2_32():
    """52 million cells of 128 multipoles at order 5 in the hi/lo form: potentials
    of targets at both ends of the Morton order against direct sums, within the
    order's interpolation error (1e-3, as on the smaller sets, and a factor of ten)."""
    import torch
    from scalfmm_amd import PRECISION_MIXED_HILO, Engine
    if torch.cuda.mem_get_info()[0] < 240 << 30:
        pytest.skip("needs 240 GiB of device memory")
    n, h = 40_000_003, 10
    g = torch.Generator(device="cuda")
    g.manual_seed(12)
    pos = [torch.rand(n, generator=g, device="cuda", dtype=torch.float64) for _ in range(3)]
    q = 2 * torch.rand(n, generator=g, device="cuda", dtype=torch.float64) - 1
    for d in range(3):
        pos[d][:32] *= 0.01
        pos[d][32:64] = 1 - 0.01 * pos[d][32:64]
    torch.cuda.synchronize()
    e = Engine(h, 1.0, (0.5, 0.5, 0.5), 5, precision=PRECISION_MIXED_HILO)
    e.set_m2l_variant(2)
    e.set_particles_device(n, *(a.data_ptr() for a in (*pos, q)))
    e.build_tree()
    e.evaluate()
    e.synchronize()
    p = ctypes.c_void_p()
    assert e._L.hfmm_get_results_device(e.h, ctypes.byref(p), None, None, None) == 0

    class Block:
        __cuda_array_interface__ = {"data": (p.value, False), "shape": (n,), "typestr": "<f8", "version": 3}

    got = torch.as_tensor(Block(), device="cuda")
    for t in (range(32), range(32, 64)):
        want = []
        for i in t:
            r2 = sum((a - a[i]) ** 2 for a in pos)
            r2[i] = float("inf")
            want.append((q * r2.rsqrt()).sum())
        want = torch.stack(want)
        err = float((got[t.start:t.stop] - want).norm() / want.norm())
        print(f"targets {t}: {err:.2e}", flush=True)
        assert err <= 1e-2
    e.close()
    del got, pos, q, r2
    torch.cuda.empty_cache()

"""More than 2^29 particles: eight lanes each are more threads than one dimension
of a launch holds.  The near field of a few targets, the last of the sorted order
among them, against sums over their 27 leaves (1e-12, the FP64 path's bound)."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu

N, H = (1 << 29) + 4099, 9


def test_near_field_beyond_2_29_particles():
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

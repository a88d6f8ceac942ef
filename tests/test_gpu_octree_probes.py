"""gk_octree_probes (each corner once) against gk_octree_points (nine probes a
voxel): the map gives the same positions, bit for bit, with no point twice, for
lattices of odd sizes, few voxels, one voxel and all of them."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("res", [(1, 1, 1), (3, 5, 7), (10, 10, 10), (31, 2, 65)])
@pytest.mark.parametrize("share", [0.0, 0.3, 1.0])
def test_probes(gpu, res, share):
    from gempy_amd import _lib
    from gempy_amd.engine import _ptr, _stream, handle
    lib, total = _lib.load(), res[0] * res[1] * res[2]
    g = torch.Generator().manual_seed(total)
    vox = torch.randperm(total, generator=g)[:max(1, int(share * total))].sort().values.cuda()
    n = vox.numel()
    ext, cres = (C.c_double * 6)(-3.0, 10.0, 0.1, 0.7, 100.0, 1000.0), (C.c_int64 * 3)(*res)
    want = torch.empty((9 * n, 3), dtype=torch.float64, device="cuda")
    _lib.check("gk_octree_points", lib.gk_octree_points(handle(0), ext, cres, _ptr(vox), n, 0, _ptr(want), _stream()))
    xyz = torch.full((9 * n, 3), -9.0, dtype=torch.float64, device="cuda")
    probe = torch.full((9 * n,), -1, dtype=torch.int32, device="cuda")
    count = C.c_int64(0)
    _lib.check("gk_octree_probes", lib.gk_octree_probes(handle(0), ext, cres, _ptr(vox), n, _ptr(xyz), _ptr(probe),
                                                        C.byref(count), _stream()))
    assert torch.equal(xyz[probe.long()], want)
    assert torch.equal(probe[0::9].cpu(), torch.arange(n, dtype=torch.int32))
    assert torch.unique(xyz[:count.value], dim=0).shape[0] == count.value == torch.unique(want, dim=0).shape[0]
    assert bool((xyz[count.value:] == -9.0).all())

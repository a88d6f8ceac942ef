"""gk_octree_probes refuses voxel indices outside the level, and writes nothing
for them."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bad", [-1, 3 * 5 * 7, 10 ** 12, -10 ** 12])
def test_voxel_outside_the_level(gpu, bad):
    from gempy_amd import _lib
    from gempy_amd.engine import _ptr, _stream, handle
    lib = _lib.load()
    vox = torch.tensor([0, bad, 104], dtype=torch.int64, device="cuda")
    ext, cres = (C.c_double * 6)(0.0, 1.0, 0.0, 1.0, 0.0, 1.0), (C.c_int64 * 3)(3, 5, 7)
    xyz = torch.full((27, 3), -9.0, dtype=torch.float64, device="cuda")
    probe = torch.full((27,), -1, dtype=torch.int32, device="cuda")
    count = C.c_int64(-1)
    print(f"[gpu-case] probes with voxel {bad}", flush=True)
    rc = lib.gk_octree_probes(handle(0), ext, cres, _ptr(vox), 3, _ptr(xyz), _ptr(probe), C.byref(count), _stream())
    assert _lib.GK_ERR[rc] == "GK_ERR_ARG" and count.value == 0
    assert bool((probe[9:18] == -1).all()) and bool((xyz[1] == -9.0).all())


def test_level_too_large(gpu):
    from gempy_amd import _lib
    from gempy_amd.engine import _ptr, _stream, handle
    vox = torch.zeros(1, dtype=torch.int64, device="cuda")
    xyz, probe = torch.empty((9, 3), dtype=torch.float64, device="cuda"), torch.empty(9, dtype=torch.int32, device="cuda")
    ext, count = (C.c_double * 6)(0.0, 1.0, 0.0, 1.0, 0.0, 1.0), C.c_int64(-1)
    for res in ((2 ** 31, 2 ** 31, 2 ** 31), (2 ** 62, 3, 3), (1290, 1290, 1290)):
        rc = _lib.load().gk_octree_probes(handle(0), ext, (C.c_int64 * 3)(*res), _ptr(vox), 1, _ptr(xyz), _ptr(probe),
                                          C.byref(count), _stream())
        assert _lib.GK_ERR[rc] == "GK_ERR_ARG"

"""Data that hold a position which is no number: the neighbour search finds fewer
neighbours than it should, nothing is read at the missing ones, the solve
reports an error and the next one is as before."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _stack(oris):
    from gempy_amd import synthetic
    m = synthetic.config3(seed=6, n_points=300, n_ori=max(oris, 1), n_surfaces=3, resolution=(8, 8, 8))
    s = m.stacks[0]
    if oris == 0:
        s.ori_xyz, s.ori_grad, s.ori_nugget = s.ori_xyz[:0], s.ori_grad[:0], s.ori_nugget[:0]
    return m, s


@pytest.mark.parametrize("oris,bad", [(60, "point"), (60, "orientation"), (0, "point")])
def test_nan_position(gpu, oris, bad):
    from gempy_amd import _lib
    from gempy_amd.engine import DeviceStack, _ptr, _stream
    import ctypes as C
    m, s = _stack(oris)
    (s.sp_xyz if bad == "point" else s.ori_xyz)[7, 1] = np.nan
    ds = DeviceStack(s, m.options.kernel_options, [500.0] * 3)
    print(f"[gpu-case] NaN {bad}, {oris} orientations", flush=True)
    n = ds.sys.n_ori + ds.sys.n_rest
    idx = torch.empty((n, 32), dtype=torch.int32, device=gpu)
    hk = torch.empty(n, dtype=torch.float32, device=gpu)
    _lib.check("knn", _lib.load().gk_test_knn_local(ds.h, C.byref(ds.sys), _ptr(idx), _ptr(hk), _stream()))
    none = (idx == 0x7fffffff).all(1)
    assert int(none.sum()) == 1 and bool(((idx < n) | none[:, None]).all())
    with pytest.raises(Exception):
        ds.solve(_lib.GK_SOLVE_FP32_REFINE)
    torch.cuda.synchronize()
    m, s = _stack(60)
    good = DeviceStack(s, m.options.kernel_options, [500.0] * 3)
    w, info = good.solve(_lib.GK_SOLVE_FP32_REFINE)
    assert bool(w.isfinite().all()) and info["fallback"] == 0

"""Explicit points whose pairs all lie within the range are summed without the
mask: the same bits as gk_eval_noalloc, which always tests it, for point sets
and sources inside, across and outside half the range around the centre, with
centres away from the data, and for the sizes at which the flags of the source
groups change (1,024 rest points or orientations each)."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _eval(name, ds, w, X, precision, gradient):
    from gempy_amd import _lib
    from gempy_amd.engine import _ptr, _stream
    n = X.shape[0]
    S = torch.full((n,), -1.0, dtype=torch.float64, device="cuda")
    G = torch.full((n, 3), -1.0, dtype=torch.float64, device="cuda") if gradient else None
    d = _lib.GkEvalDesc()
    d.kind, d.precision, d.n_points = _lib.GK_POINTS_EXPLICIT, precision, n
    d.xyz, d.scalar, d.gradient = _ptr(X), _ptr(S), _ptr(G)
    _lib.check(name, getattr(_lib.load(), name)(ds.h, C.byref(ds.sys), _ptr(w), C.byref(d), _stream()))
    return S, G


@pytest.mark.parametrize("range_,center", [(1732.06, 500.0), (1732.06, 400.0), (900.0, 500.0), (4000.0, 0.0)])
@pytest.mark.parametrize("points,oris", [(1030, 5), (1029, 1025), (60, 20)])
@pytest.mark.parametrize("gradient", [False, True])
def test_same_bits_as_masked(gpu, range_, center, points, oris, gradient):
    from gempy_amd import _lib, synthetic
    from gempy_amd.data import KernelOptions
    from gempy_amd.engine import DeviceStack
    m = synthetic.config3(seed=2, n_points=points, n_ori=oris, n_surfaces=3, resolution=(8, 8, 8))
    ds = DeviceStack(m.stacks[0], KernelOptions(range=range_, c_o=range_ ** 2 / 42.0, uni_degree=1), [center] * 3)
    w = torch.randn(ds.N, dtype=torch.float64, generator=torch.Generator().manual_seed(5)).cuda()
    r = np.random.default_rng(3)
    for lo, hi in ((0.0, 1000.0), (-500.0, 1500.0), (1600.0, 1700.0)):
        X = torch.tensor(r.uniform(lo, hi, (2100, 3)), device="cuda")
        X[7] = ds.ref_xyz[0]
        X[8] = ds.ori_xyz[0]
        for precision in (_lib.GK_F64, _lib.GK_F32):
            a, b = _eval("gk_eval", ds, w, X, precision, gradient), _eval("gk_eval_noalloc", ds, w, X, precision, gradient)
            assert torch.equal(a[0], b[0])
            assert not gradient or torch.equal(a[1], b[1])

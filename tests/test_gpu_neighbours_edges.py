"""The neighbour search and the exact local inverse where their waves are
partly filled: exactly as many data points as neighbours, one more, a lane or a
workgroup more, all points but a few in one cell, coincident points.
Neighbours: distances against brute force in float64, to the rounding of
float32 positions (coordinates below 1, 2^-24 each, 8 of them per distance)."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _stack(n, kind):
    from gempy_amd import synthetic
    m = synthetic.config3(n_points=n + 2 - 8, n_ori=8, n_surfaces=2, resolution=(8, 8, 8))
    st = m.stacks[0]
    r = np.random.default_rng(n)
    if kind == "cluster":                        # nine of ten points within a thousandth of the model
        k = r.random(len(st.sp_xyz)) < 0.9
        st.sp_xyz[k] = 500.0 + r.uniform(-0.5, 0.5, (int(k.sum()), 3))
    if kind == "same":
        st.sp_xyz[3:20] = st.sp_xyz[2]
    return m, st


@pytest.mark.parametrize("n,kind", [(32, "fold"), (33, "fold"), (63, "fold"), (65, "fold"), (257, "fold"),
                                    (700, "cluster"), (100, "cluster"), (130, "same")])
def test_neighbours(gpu, n, kind):
    from gempy_amd import _lib
    from gempy_amd.engine import DeviceStack, _ptr, _stream
    m, st = _stack(n, kind)
    ko, center, K = m.options.kernel_options, [500.0] * 3, _lib.GK_LOCAL_NEIGHBOURS
    ds = DeviceStack(st, ko, center)
    assert ds.sys.n_ori + ds.sys.n_rest == n
    idx = torch.full((n * K,), -7, dtype=torch.int32, device="cuda")
    hk = torch.empty(n, dtype=torch.float32, device="cuda")
    _lib.check("gk_test_knn_local", _lib.load().gk_test_knn_local(ds.h, C.byref(ds.sys), _ptr(idx), _ptr(hk), _stream()))
    idx = idx.cpu().numpy().reshape(n, K)
    rest = np.concatenate([st.sp_xyz[o + 1:o + c] for o, c in zip(np.cumsum([0] + st.counts[:-1]), st.counts)])
    X = (np.concatenate([st.ori_xyz, rest]) - np.asarray(center)) / ko.range
    D = np.sqrt(((X[:, None] - X[None]) ** 2).sum(-1))
    got = np.take_along_axis(D, idx.astype(np.int64), 1)
    want = np.sort(D, 1)[:, :K]
    assert all(len(set(row)) == K for row in idx.tolist())
    assert np.abs(got - want).max() <= 8 * 2.0 ** -24
    assert np.abs(hk.cpu().numpy() - want[:, -1]).max() <= 8 * 2.0 ** -24


@pytest.mark.parametrize("n", [32, 33, 127, 515])
def test_solve_with_local_inverse(gpu, n):
    """FP32 form (factor, local inverse, FP64 refinement) against the direct FP64 form: fields to the residual."""
    from gempy_amd import _lib
    from gempy_amd.engine import DeviceStack
    m, st = _stack(n, "fold")
    ds = DeviceStack(st, m.options.kernel_options, [500.0] * 3)
    w, info = ds.solve(_lib.GK_SOLVE_FP32_REFINE, tol=1e-9)
    _, s = ds.surface_thresholds(w)
    w2, _ = ds.solve(_lib.GK_SOLVE_FP64_LU)
    _, s2 = ds.surface_thresholds(w2)
    assert info["fallback"] == 0                 # the residual may end at the floor of the FP64 operator
    assert float((s - s2).abs().max()) <= 1e-6 * float(s2.max() - s2.min())

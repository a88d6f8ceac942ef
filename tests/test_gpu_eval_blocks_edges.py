"""Lattice evaluations in blocks at the edges of their grouping, against the
explicit-point path, which has no blocks."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _ds(points, oris, range_, degree=1, seed=5):
    from gempy_amd import synthetic
    from gempy_amd.data import KernelOptions
    from gempy_amd.engine import DeviceStack
    m = synthetic.config3(seed=seed, n_points=points, n_ori=oris, n_surfaces=4, resolution=(8, 8, 8))
    ds = DeviceStack(m.stacks[0], KernelOptions(range=range_, c_o=range_ * range_ / 42.0, uni_degree=degree), [500.0] * 3)
    w = torch.randn(ds.N, dtype=torch.float64, generator=torch.Generator().manual_seed(seed))
    return ds, w.cuda()


@pytest.mark.parametrize("weight", [float("inf"), -float("inf"), 1e308])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_infinite_orientation_weight(gpu, weight, prec):
    """An orientation with an infinite weight makes the field infinite, with the
    sign of the plain sum, at every point (1e308 times 2 c_o / a, 82
    here, is infinite once packed)."""
    from gempy_amd import _lib, synthetic
    from gempy_amd.data import RegularGrid
    ds, w = _ds(3000, 600, 1732.05)
    g = RegularGrid(synthetic.EXTENT, (100, 101, 102))
    w[17] = weight
    p = _lib.GK_F64 if prec == "f64" else _lib.GK_F32
    print(f"[gpu-case] weight {weight} {prec}", flush=True)
    S, _, _ = ds.evaluate_lattice(g, w, p)
    S2, _, _ = ds.evaluate_points(torch.tensor(g.values(), device="cuda"), w, p)
    assert int(S2.isinf().sum()) > 0.99 * S2.numel()
    assert bool(((S == S2) | (S.isnan() & S2.isnan())).all())


@pytest.mark.parametrize("prec,depth", [("f64", 0.01), ("f32", 0.05)])
def test_blocks_many_ranges_wide(gpu, prec, depth):
    """A lattice whose blocks are thousands of ranges wide, orientations just
    within the range of its points: none is taken for beyond the range.  The
    reference is the plain lattice sum with the same runs of points
    (gk_eval_noalloc), so that both see the same rounded positions.

    Bound: a point has some ten sources within the range, each a polynomial with
    terms up to 14 times the packed weight 2, some ten roundings; in FP64 the
    runs start at other points (4 and 8 long), so positions differ by two
    roundings of 2.4e5, times 105 depth^2, the slope of C'/r."""
    import ctypes as C
    from gempy_amd import _lib
    from gempy_amd.data import KernelOptions, RegularGrid, StackInput
    from gempy_amd.engine import DeviceStack, _ptr, _stream
    n, h, no = 96, 5000.123, 3000
    g = RegularGrid((0.0, n * h) * 3, (n,) * 3)
    r = np.random.default_rng(11)
    ijk, axis, ang = r.integers(0, n, (no, 3)), r.integers(0, 3, no), r.uniform(0, np.pi / 2, no)
    off = -(1.0 - depth * r.random(no))[:, None] * np.stack([np.cos(ang), np.sin(ang)], 1)
    q = ijk.astype(float)
    for a in range(3):                       # beside the three edges of the lattice at its origin, where blocks start
        u, v, i = (a + 1) % 3, (a + 2) % 3, axis == a
        q[i, u], q[i, v] = 0.0, 0.0
    q = (q + 0.5) * h
    for a in range(3):
        u, v, i = (a + 1) % 3, (a + 2) % 3, axis == a
        q[i, u] += off[i, 0]
        q[i, v] += off[i, 1]
    st = StackInput("wide", np.array([[0.0, 0, 0], [h, h, h]]), [2], np.zeros(2), q, np.ones((no, 3)), np.zeros(no))
    ds = DeviceStack(st, KernelOptions(range=1.0, c_o=1.0, uni_degree=0), [n * h / 2] * 3)
    w = torch.zeros(ds.N, dtype=torch.float64)
    w[:3 * no] = 1.0
    w = w.cuda()
    out = []
    for name in ("gk_eval", "gk_eval_noalloc"):
        d = _lib.GkEvalDesc()
        d.kind, d.precision = _lib.GK_POINTS_LATTICE, _lib.GK_F64 if prec == "f64" else _lib.GK_F32
        for k in range(3):
            d.origin[k], d.spacing[k], d.res[k] = g.origin[k], g.spacing[k], n
        S = torch.full((g.n_points,), -1.0, dtype=torch.float64, device=gpu)
        d.scalar = _ptr(S)
        print(f"[gpu-case] wide blocks {prec} {name}", flush=True)
        _lib.check(name, getattr(_lib.load(), name)(ds.h, C.byref(ds.sys), _ptr(w), C.byref(d), _stream()))
        out.append(S)
    eps = 2.0 ** -53 if prec == "f64" else 2.0 ** -24
    bound = 24 * 2 * 14 * 10 * eps
    if prec == "f64":
        bound += 24 * 2 * 105 * depth ** 2 * 4 * 2.4e5 * eps
    assert int((out[1].abs() > 8 * bound).sum()) > n
    assert float((out[0] - out[1]).abs().max()) <= bound


def _bound(points, oris, range_, prec, gradient=False):
    """As in test_gpu_eval_blocks.py."""
    from test_gpu_eval_blocks import _bound as b
    return b(points, oris, range_, prec, gradient)


@pytest.mark.parametrize("prec,ny", [("f64", 24), ("f32", 16)])
def test_slab(gpu, prec, ny):
    from gempy_amd import _lib, synthetic
    from gempy_amd.data import RegularGrid
    ds, w = _ds(3000, 600, 1732.05)
    g = RegularGrid(synthetic.EXTENT, (150, ny, 170))
    S, _, _ = ds.evaluate_lattice(g, w, _lib.GK_F64 if prec == "f64" else _lib.GK_F32)
    S2, _, _ = ds.evaluate_points(torch.tensor(g.values(), device="cuda"), w)
    assert float((S - S2).abs().max()) <= _bound(3000, 600, 1732.05, prec)


@pytest.mark.parametrize("range_,gradient", [(1732.05, False), (450.0, True)])
def test_negative_spacing(gpu, range_, gradient):
    """Axes that run downwards: the same field, reversed."""
    from gempy_amd.data import RegularGrid
    n = (3000, 600) if not gradient else (2000, 500)
    ds, w = _ds(*n, range_)
    g = RegularGrid((1000.0, 0.0, 0.0, 1000.0, 1000.0, 0.0), (100, 101, 102))
    S, G, _ = ds.evaluate_lattice(g, w, gradient=gradient)
    S2, G2, _ = ds.evaluate_points(torch.tensor(g.values(), device="cuda"), w, gradient=gradient)
    assert float((S - S2).abs().max()) <= _bound(*n, range_, "f64")
    if gradient:
        assert float((G - G2).abs().max()) <= _bound(*n, range_, "f64", True)


@pytest.mark.parametrize("degree", [0, 2])
@pytest.mark.parametrize("faults", [0, 2])
def test_drift_and_fault_columns(gpu, degree, faults):
    """Drift of degree 0 and 2 and fault columns, on a ragged lattice, with ids.
    The drift's terms reach 2 x 10^6 times weights up to 5: 16 roundings of their
    sum more than the pairs have."""
    from gempy_amd import synthetic
    from gempy_amd.data import KernelOptions, RegularGrid
    from gempy_amd.engine import DeviceStack
    m = synthetic.config3(seed=5, n_points=2500, n_ori=500, n_surfaces=4, resolution=(8, 8, 8)).stacks[0]
    step = np.stack([np.where(m.sp_xyz[:, 0] > 400.0, 2.0, 1.0), np.where(m.sp_xyz[:, 1] > 300.0, 1.0, 2.0)], 1)
    ds = DeviceStack(m, KernelOptions(range=1732.05, c_o=1732.05 ** 2 / 42.0, uni_degree=degree), [500.0] * 3,
                     fault_sp=step[:, :faults] if faults else None)
    assert ds.n_fault == faults
    w = torch.randn(ds.N, dtype=torch.float64, generator=torch.Generator().manual_seed(9)).cuda()
    g = RegularGrid(synthetic.EXTENT, (101, 99, 97))
    X = torch.tensor(g.values(), device="cuda")
    fv = None
    if faults:
        fv = torch.stack([(X[:, 0] > 400.0).double() + 1.0, (X[:, 1] <= 300.0).double() + 1.0], 1).contiguous()
    thr = [3e6, 0.0, -3e6]
    S, _, ids = ds.evaluate_lattice(g, w, thresholds=thr, fault_values=fv)
    S2, _, _ = ds.evaluate_points(X, w, fault_values=fv)
    drift = 16 * 2.0 ** -53 * 2 * 5 * 6e6 if degree == 2 else 0.0
    assert float((S - S2).abs().max()) <= _bound(2500, 500, 1732.05, "f64") + drift
    assert bool((ids == 1 + sum((S < t).int() for t in thr)).all())
    if faults:                                # the columns do reach the field
        S0, _, _ = ds.evaluate_lattice(g, w, fault_values=torch.zeros_like(fv))
        assert float((S - S0).abs().min()) > 0.0

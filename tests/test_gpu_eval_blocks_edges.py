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

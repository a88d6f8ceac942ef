"""The one launch that prepares sources and operator rows, at the edges of its
workgroups (1,024 rest points or orientations each), for every drift degree and
with fault columns: the matrix-free product against the assembled matrix.
Bound per row: terms of at most 16 c_o each (four covariances of an increment,
or a drift function), 16 roundings of 2^-53 each, over all unknowns."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rest,oris,surfaces", [(1, 1, 1), (5, 1024, 1), (1023, 2, 3), (1024, 1025, 2), (1025, 33, 10),
                                                (2049, 64, 1)])
@pytest.mark.parametrize("degree,faults", [(0, 0), (1, 0), (2, 0), (1, 2), (0, 1)])
def test_product_matches_matrix(gpu, rest, oris, surfaces, degree, faults):
    from gempy_amd import synthetic
    from gempy_amd.data import KernelOptions
    from gempy_amd.engine import DeviceStack
    m = synthetic.config3(seed=7, n_points=rest + surfaces, n_ori=oris, n_surfaces=surfaces, resolution=(8, 8, 8))
    st, a = m.stacks[0], synthetic.RANGE
    f = None
    if faults:
        f = np.random.default_rng(1).integers(1, 3, (len(st.sp_xyz), faults)).astype(float)
        f[0], f[1] = 1.0, 2.0                    # no column without a step
    ds = DeviceStack(st, KernelOptions(range=a, c_o=a * a / 42.0, uni_degree=degree), [500.0] * 3, fault_sp=f)
    assert (ds.sys.n_rest, ds.sys.n_ori) == (rest, oris) and (faults == 0 or ds.n_fault == faults)
    A, _, _ = ds.assemble()
    A = A[:ds.N, :ds.N]
    A = torch.tril(A) + torch.tril(A, -1).T
    x = torch.randn(ds.N, dtype=torch.float64, generator=torch.Generator().manual_seed(rest)).cuda()
    y = ds.matvec(x)
    tol = 2.0 ** -53 * 16 * 16 * a * a / 42.0 * float(x.abs().sum())
    assert float((y - (A @ x)).abs().max()) <= tol

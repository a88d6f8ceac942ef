"""FP64 and FP32 Cholesky at the edges of the 16-column panels, the 128-column
diagonal blocks, the 256-column block columns and the identity padding:
L L^T = A, the stored inverses of the diagonal blocks, the triangular solves.

Tolerances: a Cholesky factor of a well-conditioned matrix of unit diagonal
scale satisfies |L L^T - A| <= (n + 1) u |L| |L|^T entrywise (u = 2^-53 or
2^-24); the inverses and solves add their own n u times the condition number
(below 5 here)."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _spd(n, seed):
    g = np.random.default_rng(seed)
    m = g.standard_normal((n, n))
    return 0.3 * m @ m.T / n + np.eye(n)


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 127, 128, 129, 255, 256, 257, 385, 640, 1025, 2304])
def test_cholesky_edges(gpu, dtype, n):
    from gempy_amd import _lib as L
    from gempy_amd.engine import _ptr, _stream, handle
    lib = L.load()
    tdt, u = (torch.float64, 2.0 ** -53) if dtype == "f64" else (torch.float32, 2.0 ** -24)
    print(f"[gpu-case] cholesky {dtype} n={n}", flush=True)
    lda = -(-n // 256) * 256
    A = _spd(n, n)
    t = torch.full((lda, lda), 7.0, dtype=tdt, device=gpu)       # padding is the library's to reset
    t[:n, :n] = torch.tensor(A, dtype=tdt)
    A = t[:n, :n].double().cpu().numpy()
    dinv = torch.empty(L.GK_CHOL_PLANES * lda * 256, dtype=tdt, device=gpu)
    info = C.c_int32(-1)
    fn = lib.gk_cholesky_f64 if dtype == "f64" else lib.gk_cholesky_f32
    L.check("chol", fn(handle(0), _ptr(t), n, lda, _ptr(dinv), C.byref(info), _stream()))
    assert info.value == 0
    full = torch.tril(t).double().cpu().numpy()
    lo = full[:n, :n]
    assert np.array_equal(full[n:, n:], np.eye(lda - n)) and not full[n:, :n].any()
    # the factorization reads A's lower triangle only (m m^T need not be
    # symmetric to the last bit)
    assert np.tril(np.abs(lo @ lo.T - A) <= 2 * (n + 1) * u * (np.abs(lo) @ np.abs(lo).T)).sum() == n * (n + 1) // 2
    d = dinv[:lda * 256].reshape(lda // 256, 256, 256).double().cpu().numpy()
    for k in range(lda // 256):
        blk = full[k * 256:(k + 1) * 256, k * 256:(k + 1) * 256]
        assert not np.triu(d[k], 1).any()
        assert np.abs(d[k] @ blk - np.eye(256)).max() <= 256 * 5 * u * 4
    b = np.random.default_rng(n + 1).standard_normal(n)
    x = torch.zeros(lda, dtype=tdt, device=gpu)
    x[:n] = torch.tensor(b, dtype=tdt)
    b = x[:n].double().cpu().numpy()
    fs = lib.gk_cholesky_solve_f64 if dtype == "f64" else lib.gk_cholesky_solve_f32
    L.check("solve", fs(handle(0), _ptr(t), _ptr(dinv), lda, _ptr(x), _stream()))
    xs = x.double().cpu().numpy()
    assert not xs[n:].any()
    r = np.abs(A @ xs[:n] - b).max()
    assert r <= 8 * (n + 256) * u * (np.abs(A).sum(1).max() * np.abs(xs).max() + np.abs(b).max())


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("bad", [0, 20, 140, 300])
def test_cholesky_reports_the_failed_pivot(gpu, dtype, bad):
    """A negative diagonal entry fails at its own column (1-based)."""
    from gempy_amd import _lib as L
    from gempy_amd.engine import _ptr, _stream, handle
    lib = L.load()
    tdt = torch.float64 if dtype == "f64" else torch.float32
    print(f"[gpu-case] cholesky {dtype} failing pivot {bad}", flush=True)
    t = torch.eye(512, dtype=tdt, device=gpu)
    t[bad, bad] = -1.0
    dinv = torch.empty(L.GK_CHOL_PLANES * 512 * 256, dtype=tdt, device=gpu)
    info = C.c_int32(-1)
    fn = lib.gk_cholesky_f64 if dtype == "f64" else lib.gk_cholesky_f32
    assert fn(handle(0), _ptr(t), 500, 512, _ptr(dinv), C.byref(info), _stream()) == -3
    assert info.value == bad + 1

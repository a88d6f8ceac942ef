"""The diagonal-block Cholesky kernel run on the CPU with its waves in
different orders between barriers (tests/host/potrf_waves.cpp): no order may
change a bit, so nothing that one wave reads is written by another one in the
same interval, and L L^T = A, X L = I in each.

Tolerances: |L L^T - A| <= (n + 1) u |L| |L|^T entrywise for a Cholesky factor
(u = 2^-53 or 2^-24), twice that for the reciprocal pivots in place of
divisions; the inverse n u times the condition number (below 5)."""
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(os.path.dirname(HERE), "gempy_amd", "csrc", "gk_dense.hip")
ORDERS = ["01234567", "76543210", "21034567", "60715243"]


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    cxx = next((c for c in ("/opt/rocm/llvm/bin/clang++", shutil.which("clang++")) if c and os.path.exists(c)), None)
    if cxx is None:
        pytest.skip("needs clang++ (vector types)")
    d = tmp_path_factory.mktemp("potrf")
    text = open(SRC).read()
    beg = text.index("// Blocked Cholesky + inverse of a DB x DB block")
    end = text.index("// FP32:", text.index("__device__ void potrf_blocked"))
    (d / "kernel.inc").write_text(text[beg:end])
    exe = d / "potrf_waves"
    subprocess.run([cxx, "-std=c++17", "-O1", "-ffp-contract=off", "-Wno-everything",
                    f'-DKERNEL_SRC="{d / "kernel.inc"}"', "-o", str(exe), os.path.join(HERE, "host", "potrf_waves.cpp")],
                   check=True)
    return str(exe)


def _run(exe, A, live, order):
    bits = A.dtype.itemsize * 8
    r = subprocess.run([exe, str(bits), str(live), order], input=A.tobytes(), capture_output=True, timeout=60)
    assert r.returncode == 0, f"harness status {r.returncode} in order {order}"
    n = 128 * 128
    out = np.frombuffer(r.stdout[:2 * n * A.dtype.itemsize], dtype=A.dtype).reshape(2, 128, 128)
    return np.tril(out[0]), out[1], int(np.frombuffer(r.stdout[-4:], dtype=np.int32)[0])


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("live", [1, 16, 17, 100, 128])
def test_no_wave_order_changes_the_factor(harness, dtype, live):
    u = 2.0 ** -53 if dtype is np.float64 else 2.0 ** -24
    g = np.random.default_rng(live)
    m = g.standard_normal((128, 128))
    A = np.eye(128)
    A[:live, :live] += 0.3 * (m @ m.T)[:live, :live] / 128
    A = A.astype(dtype)
    first = None
    for order in ORDERS:
        L, X, info = _run(harness, A, live, order)
        assert info == 0
        lo = L.astype(np.float64)
        assert (np.tril(np.abs(lo @ lo.T - A)) <= 2 * 129 * u * (np.abs(lo) @ np.abs(lo).T)).all(), order
        assert np.abs(X.astype(np.float64) @ lo - np.eye(128)).max() <= 128 * 5 * u * 4, order
        if first is not None:
            assert np.array_equal(L, first[0]) and np.array_equal(X, first[1]), order
        first = first or (L, X)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("bad", [0, 20, 100])
def test_failed_pivot_in_every_order(harness, dtype, bad):
    A = np.eye(128, dtype=dtype)
    A[bad, bad] = -1.0
    assert [_run(harness, A, 128, o)[2] for o in ORDERS] == [bad + 1] * len(ORDERS)

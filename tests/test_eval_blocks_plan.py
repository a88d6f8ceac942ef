"""Which lattice evaluations run in blocks (launches recorded on the CPU, see
fake_hip.py): those that test_gpu_eval_blocks*.py compare with the explicit
points must not quietly be two plain sums, and a few stay plain on purpose."""
import os

import pytest

import fake_hip

LIB_PY = os.path.join(os.path.dirname(fake_hip.LIB), "_lib.py")

BODY = """
import importlib.util
spec = importlib.util.spec_from_file_location("gk_lib", LIB_PY)
L = importlib.util.module_from_spec(spec)
spec.loader.exec_module(L)
buf = device(256)

def plan(res, n_rest, n_ori, range_, prec, gradient, lo, hi, box):
    s = L.GkSystem()
    s.n_ori, s.n_rest, s.n_surf = n_ori, n_rest, 4
    s.range, s.c_o, s.i_res, s.gi_res = range_, 1.0, 4.0, 2.0
    for f in ("ori_xyz", "ori_grad", "ori_nugget", "rest_xyz", "rest_surf", "rest_nugget", "ref_xyz"):
        setattr(s, f, buf)
    d = L.GkEvalDesc()
    d.kind, d.precision = L.GK_POINTS_LATTICE, L.GK_F64 if prec == "f64" else L.GK_F32
    for k in range(3):
        s.center[k] = 500.0
        d.spacing[k] = (box[2 * k + 1] - box[2 * k]) / res[k]
        d.origin[k], d.res[k] = box[2 * k] + d.spacing[k] / 2, res[k]
    d.scalar = buf
    d.gradient = buf if gradient else None
    b = f64(*lo, *hi)
    fake.fake_d2h(b, C.c_size_t(48))
    fake.fake_clear()
    assert lib.gk_eval(h, C.byref(s), buf, C.byref(d), None) == 0, lib.gk_last_error()
    names = launched()
    if any("far_nodes" in n for n in names):
        return "nodes"
    if any("near_kernel" in n for n in names):
        return "near"
    assert any("eval_kernel" in n for n in names), names
    return "plain"

bad = []
for name, want, args in CASES:
    got = plan(*args)
    if got != want:
        bad.append((name, want, got))
assert not bad, bad
"""

EXTENT = (0.0, 1000.0) * 3
LO, HI = (1.0, 1.0, 40.0), (999.0, 999.0, 960.0)


def _case(want, res, n_rest, n_ori, range_, prec, gradient, lo=LO, hi=HI, box=EXTENT):
    return (f"{res} {n_rest} {n_ori} {range_} {prec} {gradient}", want,
            (res, n_rest, n_ori, range_, prec, gradient, lo, hi, box))


CASES = [
    # as in test_gpu_eval_blocks.py
    _case("nodes", (101, 97, 103), 1996, 400, 1732.05, "f64", False),
    _case("nodes", (130, 64, 90), 2996, 30, 1732.05, "f64", False),
    _case("nodes", (128, 128, 128), 596, 200, 1732.05, "f64", False),
    _case("plain", (200, 3, 200), 5996, 1500, 1732.05, "f64", False),
    _case("plain", (1, 300, 301), 8996, 2000, 1732.05, "f64", False),
    _case("nodes", (100, 100, 100), 2996, 600, 1732.05, "f32", False),
    _case("nodes", (61, 157, 73), 4996, 1000, 1732.05, "f32", False),
    _case("near", (96, 97, 98), 2996, 700, 450.0, "f64", False),
    _case("nodes", (96, 97, 98), 2996, 700, 1300.0, "f64", False),
    _case("near", (96, 97, 98), 1996, 500, 450.0, "f64", True),
    _case("nodes", (96, 97, 98), 2996, 700, 300.0, "f32", False),
    _case("near", (96, 97, 98), 1996, 500, 450.0, "f32", True),
    _case("near", (80, 81, 300), 1996, 600, 60.0, "f64", False),
    _case("nodes", (90, 91, 92), 2996, 600, 4000.0, "f64", False, box=(2000.0, 2600.0, -50.0, 300.0, 400.0, 500.0)),
    _case("nodes", (90, 91, 92), 2996, 600, 4000.0, "f64", False, box=(0.0, 1000.0, 0.0, 1000.0, 499.0, 500.0)),
    _case("nodes", (101, 99, 97), 2496, 500, 1732.05, "f64", False),
    _case("nodes", (100, 101, 102), 2996, 600, 1732.05, "f64", False),
    _case("near", (100, 101, 102), 2996, 600, 450.0, "f64", False),
    # as in test_gpu_eval_blocks_edges.py
    _case("nodes", (150, 24, 170), 2996, 600, 1732.05, "f64", False),
    _case("nodes", (150, 16, 170), 2996, 600, 1732.05, "f32", False),
    _case("nodes", (100, 101, 102), 2996, 600, 1732.05, "f32", False),
    _case("nodes", (100, 101, 102), 2996, 600, 1732.05, "f64", False, box=(1000.0, 0.0, 0.0, 1000.0, 1000.0, 0.0)),
    _case("near", (100, 101, 102), 1996, 500, 450.0, "f64", True, box=(1000.0, 0.0, 0.0, 1000.0, 1000.0, 0.0)),
    # below 0.2 ms of pairs, and gradients without a range mask
    _case("plain", (50, 50, 50), 2996, 600, 1732.05, "f64", False),
    _case("plain", (101, 128, 90), 1596, 320, 1732.05, "f64", True),
    # sources with no box (all NaN) and lattices without extent
    _case("plain", (100, 101, 102), 2996, 600, 450.0, "f64", False, lo=(1e300,) * 3, hi=(-1e300,) * 3),
    _case("plain", (100, 101, 102), 2996, 600, 450.0, "f64", False, box=(0.0, 1000.0, 5.0, 5.0, 0.0, 1000.0)),
]


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return fake_hip.build(tmp_path_factory.mktemp("fake"))


def test_plans(fake):
    fake_hip.run(fake, f"CASES = {CASES}\nLIB_PY = {LIB_PY!r}\n" + BODY)

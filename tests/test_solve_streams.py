"""Work that a solve puts on another stream is waited for also where the solve
fails (on the CPU, see fake_hip.py): the next call uses the same buffers."""
import os

import pytest

import fake_hip

LIB_PY = os.path.join(os.path.dirname(fake_hip.LIB), "_lib.py")

BODY = """
import importlib.util
spec = importlib.util.spec_from_file_location("gk_lib", LIB_PY)
L = importlib.util.module_from_spec(spec)
spec.loader.exec_module(L)
buf = device(1 << 16)
s = L.GkSystem()
s.n_ori, s.n_rest, s.n_surf, s.uni_degree = 20, 100, 3, 1
s.range, s.c_o, s.i_res, s.gi_res = 1000.0, 1.0, 4.0, 2.0
for f in ("ori_xyz", "ori_grad", "ori_nugget", "rest_xyz", "rest_surf", "rest_nugget", "ref_xyz"):
    setattr(s, f, buf)
fake.fake_d2h(f64(0, 0, 0, 1000, 1000, 1000), C.c_size_t(48))
fake.fake_d2h((C.c_int32 * 1)(5), C.c_size_t(4))             # every factorization fails at its fifth pivot
fake.fake_clear()
info = L.GkSolveInfo()
rc = lib.gk_solve(h, C.byref(s), L.GK_SOLVE_FP32_REFINE, C.c_double(1e-6), 300, buf, C.byref(info), None)
assert L.GK_ERR[rc] == "GK_ERR_NOT_SPD", (rc, lib.gk_last_error())
log = [l.split() for l in fake.fake_log().decode().splitlines()]
at = [i for i, l in enumerate(log) if l[0] == "launch" and "local_inverse" in l[2]]
assert len(at) == 1
other = log[at[0]][1]
assert other != "stream0"
done = [l[2] for l in log[at[0]:] if l[0] == "record" and l[1] == other][0]
assert ["wait", "stream0", done] in log[at[0]:], "the caller's stream does not wait for the local inverses"
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return fake_hip.build(tmp_path_factory.mktemp("fake"))


def test_failed_solve_waits_for_its_other_stream(fake):
    fake_hip.run(fake, f"LIB_PY = {LIB_PY!r}\n" + BODY)

"""The isosurface's case tables under a workspace that grows (on the CPU, see
fake_hip.py): every launch is handed intact tables, also when the larger
workspace comes back at the smaller one's address."""
import pytest

import fake_hip

BODY = """
fake.fake_watch(C.c_size_t(2048))                 # the tables are the only large upload
field = device(8 * 64 ** 3)
nv, nf = C.c_int64(), C.c_int64()
for n in (8, 8, 40, 16, 64):
    fake.fake_clear()
    rc = lib.gk_marching_cubes(h, field, i64(n, n, n), None, C.c_double(0.0), f64(0, 0, 0), f64(1, 1, 1), None,
                               C.c_int64(0), None, C.c_int64(0), C.byref(nv), C.byref(nf), None)
    assert rc == 0, lib.gk_last_error()
    names = launched()
    assert len(names) >= 4 and all("mc_" in s for s in names), names
    assert all(fake.fake_intact(i) for i in range(len(names))), f"lattice {n}: launches without the case tables"
lib.gk_destroy(h)
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return fake_hip.build(tmp_path_factory.mktemp("fake"))


def test_tables_survive_a_growing_workspace(fake):
    fake_hip.run(fake, BODY)

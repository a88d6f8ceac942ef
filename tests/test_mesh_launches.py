"""The isosurface's passes take as many workgroups as the points need, however
few layers the lattice has (launches recorded on the CPU, see fake_hip.py)."""
import pytest

import fake_hip

BODY = """
field, buf = device(8 << 23), device(64)
nv, nf = C.c_int64(), C.c_int64()
for res in ((200, 200, 200), (2000, 2000, 2), (2, 2000, 2000), (1000, 1000, 5), (3, 3, 3)):
    fake.fake_clear()
    rc = lib.gk_marching_cubes(h, field, i64(*res), None, C.c_double(0.0), f64(0, 0, 0), f64(1, 1, 1), buf,
                               C.c_int64(0), buf, C.c_int64(0), C.byref(nv), C.byref(nf), None)
    assert rc == 0, lib.gk_last_error()
    points = res[0] * res[1] * res[2]
    grid = {n: fake.fake_grid(i, 0) for i, n in enumerate(launched())}
    bits = [g for n, g in grid.items() if "mc_bits" in n]
    assert bits == [-(-points // (64 * 32))], (res, grid)
    assert max(grid.values()) <= points // 128 + 1, (res, grid)
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return fake_hip.build(tmp_path_factory.mktemp("fake"))


def test_workgroups_follow_the_points(fake):
    fake_hip.run(fake, BODY)

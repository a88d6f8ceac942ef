"""Which tiles an FP64 product takes (launches recorded on the CPU, see
fake_hip.py): small ones where 128 x 128 tiles leave the chip idle, the large
ones where they fill their rounds of 256 CUs and the product is long."""
import pytest

import fake_hip

BODY = """
buf = device(64)
for lower, m, n, k, large in CASES:
    fake.fake_clear()
    rc = lib.gk_gemm_f64(h, C.c_int64(m), C.c_int64(n), C.c_int64(k), buf, C.c_int64(k), buf, C.c_int64(k),
                         C.c_int32(1), C.c_double(1.0), buf, C.c_int64(n), C.c_int32(lower), None)
    assert rc == 0, lib.gk_last_error()
    t = m // 128
    tiles = t * (t + 1) // 2 if lower else t * (n // 128)
    grid = [fake.fake_grid(i, 0) for i in range(fake.fake_launches())]
    assert len(grid) == 1 and (grid[0] == tiles) == large, (lower, m, n, k, grid, tiles)
"""

CASES = [
    (0, 128, 128, 4096, False), (0, 1024, 1024, 4096, False), (0, 2048, 2048, 256, False), (0, 2048, 2048, 4096, True),
    (0, 3328, 1024, 4096, False), (0, 4352, 1024, 4096, False), (0, 2560, 2560, 4096, False), (0, 2816, 2816, 128, False),
    (0, 2816, 2816, 256, True), (0, 4096, 4096, 128, True), (1, 2048, 2048, 4096, False), (1, 2816, 2816, 256, False),
    (1, 2560, 2560, 2048, True), (1, 3712, 3712, 256, False), (1, 3840, 3840, 256, True), (1, 4096, 4096, 128, True),
]


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return fake_hip.build(tmp_path_factory.mktemp("fake"))


def test_tiles_of_fp64_products(fake):
    fake_hip.run(fake, f"CASES = {CASES}\n" + BODY)

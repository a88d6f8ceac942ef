"""gk_marching_cubes on lattices of few layers (words of 64 points span many
rows) against plain NumPy, and its two writing kernels (small and large
lattices) against each other.  Positions: two units in the last place, as in
test_gpu_mesh_words.py."""
import numpy as np
import pytest
from test_gpu_mesh_words import _mesh, _reference, cube_faces  # noqa: F401 (a fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(2, 2, 2), (9, 11, 2), (2, 40, 3), (13, 2, 5), (3, 3, 33), (5, 7, 31), (2, 2, 129)])
@pytest.mark.parametrize("masked", [False, True])
def test_thin_lattices(gpu, cube_faces, shape, masked):  # noqa: F811
    r = np.random.default_rng(sum(shape) + masked)
    F = r.standard_normal(shape)
    F[r.random(shape) < 0.03] = np.nan
    mask = (r.random(shape) < 0.7).astype(np.uint8) if masked else None
    print(f"[gpu-case] thin mesh {shape} masked {masked}", flush=True)
    V, T = _reference(F, mask, cube_faces)
    rc, v, t, nv, nf = _mesh(F, mask)
    assert rc == 0 and nv == len(V) and nf == len(T)
    assert np.abs(v[:nv] - V).max(initial=0.0) <= 2 * 2.0 ** -52 * max(shape)
    assert np.array_equal(t[:nf], T)


def test_large_lattice_equals_its_slabs(gpu):
    """70 x 70 x 75 (5,742 words) takes the kernel of 16 words a block, slabs of
    it that of 2; the slabs' triangles are the whole's in order."""
    r = np.random.default_rng(4)
    F = r.standard_normal((70, 70, 75))
    F[r.random(F.shape) < 0.01] = np.nan
    rc, v, t, nv, nf = _mesh(F)
    assert rc == 0
    whole = v[t[:nf]]
    parts = []
    for x in range(0, 69, 23):
        rc, v, t, _, n = _mesh(np.ascontiguousarray(F[x:x + 24]))
        assert rc == 0
        parts.append(v[t[:n]] + np.array([x, 0.0, 0.0]))
    parts = np.concatenate(parts)
    assert parts.shape == whole.shape
    assert np.abs(parts - whole).max() <= 2 * 2.0 ** -52 * 75

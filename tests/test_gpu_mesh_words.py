"""gk_marching_cubes at the edges of its 64-point words: rows shorter than a
word, exactly one, one point more, several words; with masks and NaN.  Vertices
are compared in their order (by point, then axis) with plain NumPy, faces with
the triangles of each cube alone (a 2 x 2 x 2 lattice of its corner signs) in
cube order.  Vertex positions are one division, one sum and one product-sum
each: two units in the last place of coordinates up to 130."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _mesh(F, mask=None, cap=None):
    from gempy_amd import _lib
    from gempy_amd.engine import _ptr, _stream, handle
    lib, n = _lib.load(), F.shape
    f = torch.tensor(F, dtype=torch.float64, device="cuda")
    m = None if mask is None else torch.tensor(mask, dtype=torch.uint8, device="cuda")
    most = 3 * F.size if cap is None else cap
    v = torch.full((most, 3), -1.0, dtype=torch.float64, device="cuda")
    t = torch.full((5 * F.size, 3), -1, dtype=torch.int32, device="cuda")
    nv, nf = C.c_int64(0), C.c_int64(0)
    rc = lib.gk_marching_cubes(handle(0), _ptr(f), (C.c_int64 * 3)(*n), _ptr(m), 0.0, (C.c_double * 3)(0, 0, 0),
                               (C.c_double * 3)(1, 1, 1), _ptr(v), v.shape[0], _ptr(t), t.shape[0], C.byref(nv),
                               C.byref(nf), _stream())
    return rc, v.cpu().numpy(), t.cpu().numpy(), nv.value, nf.value


def _offsets(e):
    axis, k, o, j = e // 4, e % 4, [0, 0, 0], 0
    for d in range(3):
        if d != axis:
            o[d] = (k >> j) & 1
            j += 1
    return axis, o


def _reference(F, mask, cube_faces):
    """Vertices (by point, then axis) and faces (by cube) of the meshed cubes."""
    n = F.shape
    used, cubes = {}, []
    for x in range(n[0] - 1):
        for y in range(n[1] - 1):
            for z in range(n[2] - 1):
                c = F[x:x + 2, y:y + 2, z:z + 2]
                if np.isnan(c).any() or (mask is not None and not mask[x + 1, y + 1, z + 1]):
                    continue
                case = sum(int(c[k & 1, (k >> 1) & 1, k >> 2] > 0) << k for k in range(8))
                if case in (0, 255):
                    continue
                edges = []
                for e in range(12):
                    axis, o = _offsets(e)
                    p = np.array([x, y, z]) + o
                    q = p.copy()
                    q[axis] += 1
                    if (F[tuple(p)] > 0) != (F[tuple(q)] > 0):
                        key = 3 * ((p[0] * n[1] + p[1]) * n[2] + p[2]) + axis
                        used[key] = (p, axis, (0.0 - F[tuple(p)]) / (F[tuple(q)] - F[tuple(p)]))
                        edges.append(key)
                cubes.append((case, sorted(edges)))
    order = {k: i for i, k in enumerate(sorted(used))}
    V = np.zeros((len(used), 3))
    for k, i in order.items():
        p, axis, t = used[k]
        V[i] = p
        V[i, axis] += t
    faces = [[order[edges[j]] for j in tri] for case, edges in cubes for tri in cube_faces[case]]
    return V, np.array(faces, dtype=np.int32).reshape(-1, 3)


@pytest.fixture(scope="module")
def cube_faces(gpu):
    """Triangles of each corner case, as ranks of the cube's edges in vertex order."""
    out = {}
    for case in range(1, 255):
        F = np.array([1.0 if (case >> k) & 1 else -1.0 for k in range(8)]).reshape(2, 2, 2).transpose(2, 1, 0)
        rc, _, t, _, nf = _mesh(np.ascontiguousarray(F))
        assert rc == 0 and 1 <= nf <= 5
        out[case] = t[:nf].tolist()
    return out


@pytest.mark.parametrize("n", [(2, 2, 2), (3, 2, 63), (2, 4, 64), (3, 3, 65), (2, 3, 66), (4, 3, 128), (3, 5, 130)])
@pytest.mark.parametrize("masked,nans", [(False, False), (True, False), (True, True)])
def test_words(gpu, cube_faces, n, masked, nans):
    r = np.random.default_rng(n[2])
    F = r.standard_normal(n) + 0.4
    mask = (r.random(n) < 0.8).astype(np.uint8) if masked else None
    if nans:
        F[tuple(r.integers(0, k, 3) for k in n)] = np.nan
    V, T = _reference(F, mask, cube_faces)
    rc, v, t, nv, nf = _mesh(F, mask)
    assert rc == 0 and (nv, nf) == (len(V), len(T))
    np.testing.assert_allclose(v[:nv], V, rtol=0, atol=2 * np.spacing(130.0))
    np.testing.assert_array_equal(t[:nf], T)
    assert (v[nv:] == -1.0).all() and (t[nf:] == -1).all()


def test_small_buffer_stays_untouched(gpu):
    F = np.random.default_rng(0).standard_normal((4, 5, 70))
    rc, v, t, nv, nf = _mesh(F, cap=10)
    assert rc != 0 and nv > 10 and (v == -1.0).all() and (t == -1).all()

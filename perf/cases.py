"""Timing cases of the co-kriging engine: what a user's program has it do,
from one small model to the 200^3 grid of a 25,000-datum stack.

The data are the folded and faulted stacks of gempy_amd.synthetic (positions,
nuggets, range and c_o as there).  Every kind of case goes through a public
entry point:

  model     compute_model of one folded stack (assemble, solve, thresholds,
            dense grid, ids): what a script calls after each edit of a model
  faulted   compute_model of the fault + 3 stacks workload with octree levels
  solve     DeviceStack.solve and the field at the surface points, in the FP64
            (Cholesky or LU) or the FP32-factor form
  grid      DeviceStack.evaluate_lattice with weights at hand: FP64 or FP32
            pair sums, with or without gradient and ids, full or short range
  points    DeviceStack.evaluate_points at scattered points (custom grids,
            wells, probes)
  operator  DeviceStack.matvec, the matrix-free product of iterative solves
  adjoint   forward and backward of a misfit at observation points
  mesh      gk_marching_cubes of one surface of a dense grid into buffers that the
            program keeps

The weights of the evaluation kinds are drawn at the size a solve leaves them
(a few units per datum); solved systems are compared through their field, as
programs use them (the weights themselves carry the system's condition
number).  Solves stop at about 4,000 unknowns here: the FP64 residual floor of
the system grows with its size (3e-9 relative at 2,500 unknowns, 1e-7 at
35,000), and two correct solutions of the larger ones differ by more than a
comparison of double-precision fields may allow.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from gempy_amd import GemPyEngineConfig, _lib, compute_model, synthetic
from gempy_amd.autodiff import scalar_field_at
from gempy_amd.data import KernelOptions, RegularGrid, SolverForm
from gempy_amd.engine import DeviceStack, _ptr, _stream, handle

CENTER = [500.0, 500.0, 500.0]
FORMS = {"fp64": _lib.GK_SOLVE_FP64_CHOL, "fp64_lu": _lib.GK_SOLVE_FP64_LU, "fp32": _lib.GK_SOLVE_FP32_REFINE}


# --------------------------------------------------------------------- cases
def listed():
    return [
        # the smallest call: a three-surface sketch on a 50^3 grid, recomputed after every edit
        dict(name="model_sketch", kind="model", points=24, oris=6, surfaces=3, nx=50, ny=50, nz=50, dtype="float64",
             gradient=False),
        # a whole structural model: one fault, three stacks of 1,600 points, four octree levels
        dict(name="model_faulted_octree", kind="faulted", scale=1.0, n=128, levels=4, dtype="float64"),
        # the double-precision solve of a densely sampled stack
        dict(name="solve_fp64", kind="solve", points=2400, oris=400, surfaces=10, form="fp64"),
        # the single-precision factor with FP64 refinement on the same data
        dict(name="solve_fp32", kind="solve", points=2400, oris=400, surfaces=10, form="fp32"),
        # the largest evaluation: 8,000,000 cells of a 25,000-datum stack, field and ids
        dict(name="grid_large", kind="grid", points=20000, oris=5000, surfaces=10, nx=200, ny=200, nz=200, prec="f64",
             gradient=False, ids=True, range=synthetic.RANGE),
        # field and gradient of an ordinary stack on a box of unequal sides
        dict(name="grid_gradient", kind="grid", points=1600, oris=320, surfaces=3, nx=101, ny=128, nz=90, prec="f64",
             gradient=True, ids=False, range=synthetic.RANGE),
        # FP32 pair sums, as previews ask for: the field is kept in float32
        dict(name="grid_fp32", kind="grid", points=5000, oris=1000, surfaces=10, nx=100, ny=100, nz=100, prec="f32",
             gradient=False, ids=False, range=synthetic.RANGE),
        # a kernel range shorter than the model: most pairs are beyond it
        dict(name="grid_short_range", kind="grid", points=5000, oris=1000, surfaces=10, nx=150, ny=133, nz=61,
             prec="f64", gradient=False, ids=True, range=450.0),
        # ids at a ragged set of scattered points
        dict(name="points_ids", kind="points", points=5000, oris=1000, surfaces=10, n=100003, gradient=False, ids=True),
        # one matrix-free product at the size of the headline solve
        dict(name="operator_large", kind="operator", points=20000, oris=5000, surfaces=10),
        # one step of an inversion: the misfit at 10,000 observations and its gradient
        dict(name="adjoint_step", kind="adjoint", points=800, oris=160, surfaces=3, n=10000),
        # one surface's mesh of a dense grid
        dict(name="mesh_surface", kind="mesh", nx=200, ny=200, nz=200, masked=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _axes(rng, most, lo=20, hi=220):
    while True:
        n = [_log(rng, lo, hi) for _ in range(3)]
        if n[0] * n[1] * n[2] <= most:
            return dict(nx=n[0], ny=n[1], nz=n[2])


def draw(rng):
    kind = rng.choice(["model", "faulted", "solve", "solve", "grid", "grid", "grid", "points", "operator", "adjoint",
                       "mesh"])
    s = rng.randint(2, 10)
    if kind == "model":
        p = _log(rng, 24, 800)
        return dict(kind=kind, points=p, oris=max(4, p // 5), surfaces=min(s, 4), dtype=rng.choice(["float32", "float64"]),
                    gradient=rng.random() < 0.3, **_axes(rng, 1_000_000))
    if kind == "faulted":
        levels = rng.randint(2, 4)
        return dict(kind=kind, scale=round(rng.uniform(0.1, 1.0), 2), n=rng.randint(4, 12) * 2 ** (levels - 1),
                    levels=levels, dtype="float64")
    if kind == "solve":
        p = _log(rng, 60, 2400)
        return dict(kind=kind, points=p, oris=max(4, int(p * rng.uniform(0.1, 0.2))), surfaces=s,
                    form=rng.choice(["fp64", "fp32", "fp32", "fp64_lu"]))
    if kind == "grid":
        p = _log(rng, 30, 12000)
        prec = rng.choice(["f64", "f64", "f64", "f32"])
        c = dict(kind=kind, points=p, oris=max(2, int(p * rng.uniform(0.05, 0.3))), surfaces=s, prec=prec,
                 gradient=rng.random() < 0.3, ids=prec == "f64" and rng.random() < 0.7,
                 range=rng.choice([synthetic.RANGE, synthetic.RANGE, round(rng.uniform(300.0, 1500.0), 1)]))
        return dict(c, **_axes(rng, min(4_000_000, int(3e10 / p))))
    if kind == "points":
        p = _log(rng, 30, 20000)
        return dict(kind=kind, points=p, oris=max(2, int(p * rng.uniform(0.05, 0.3))), surfaces=s,
                    n=min(_log(rng, 100, 500_000), int(5e9 / p)), gradient=rng.random() < 0.3, ids=rng.random() < 0.7)
    if kind == "operator":
        p = _log(rng, 200, 20000)
        return dict(kind=kind, points=p, oris=max(2, int(p * rng.uniform(0.1, 0.25))), surfaces=s)
    if kind == "adjoint":
        p = _log(rng, 60, 800)
        return dict(kind=kind, points=p, oris=max(4, p // 5), surfaces=min(s, 4), n=_log(rng, 500, 20000))
    return dict(kind=kind, masked=rng.random() < 0.5, **_axes(rng, 8_000_000, 30, 250))


# -------------------------------------------------------------------- inputs
def _fold(case, seed, res=(8, 8, 8)):
    return synthetic.config3(seed=seed, n_points=case["points"], n_ori=case["oris"], n_surfaces=case["surfaces"],
                             resolution=res)


def _res(case):
    return (case["nx"], case["ny"], case["nz"])


def _kernel(case):
    a = case.get("range", synthetic.RANGE)
    return KernelOptions(range=a, c_o=a * a / 42.0, uni_degree=1)


def _unknowns(case):
    return 3 * case["oris"] + case["points"] - case["surfaces"] + 3


def _weights(case, seed):
    """Weights of the size a solve leaves: a few units per datum, the drift near 0.5."""
    g = torch.Generator().manual_seed(seed + 77)
    w = torch.randn(_unknowns(case), dtype=torch.float64, generator=g)
    w[:-3] *= 4.0
    w[-3:] *= 0.5
    return w


def _levels(case):
    """Decreasing values across the bulk of the field of _weights."""
    sd = 1.6 * _kernel(case).c_o * math.sqrt(case["points"])
    return np.linspace(1.0, -1.0, case["surfaces"]) * sd


def _grid(case):
    return RegularGrid(synthetic.EXTENT, _res(case))


def _points(n, seed):
    return np.random.default_rng(seed + 31).uniform(0.0, 1000.0, (n, 3))


def _mesh_input(case, seed, dev="cuda"):
    r = np.random.default_rng(seed)
    amp, ph, k = r.uniform(30, 80, 3), r.uniform(0, 2 * np.pi, 3), r.uniform(0.5, 2.0, (3, 2))
    g = _grid(case)
    x, y, z = (torch.tensor(g.origin[d] + g.spacing[d] * np.arange(_res(case)[d]), dtype=torch.float64, device=dev)
               for d in range(3))
    top = 500.0 + torch.zeros((len(x), len(y)), dtype=torch.float64, device=dev)
    for a, p, (kx, ky) in zip(amp, ph, k):
        top = top + a * torch.sin(2 * np.pi * (kx * x[:, None] + ky * y[None, :]) / 1000.0 + p)
    f = (z[None, None, :] - top[:, :, None]).reshape(-1)
    m = (z[None, None, :] > (top - 30.0 + 0.08 * x[:, None])[:, :, None]).to(torch.uint8).reshape(-1)
    return f.contiguous(), (m if case["masked"] else None)


def _most_vertices(case):
    """A bound on the crossings of a surface z = top(x, y) of bounded variation."""
    nx, ny, nz = _res(case)
    return 6 * (nx * ny + ny * nz + nx * nz)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "model":
        m = _fold(case, seed, _res(case))
        m.options.solver = SolverForm.FP64_CHOL
        m.options.evaluation_options.compute_scalar_gradient = case["gradient"]
        return dict(kind=kind, model=m, cfg=GemPyEngineConfig(dtype=case["dtype"]))
    if kind == "faulted":
        m = synthetic.config2(seed=seed, scale=case["scale"], resolution=(case["n"],) * 3, octree_levels=case["levels"])
        m.options.solver = SolverForm.FP64_CHOL
        return dict(kind=kind, model=m, cfg=GemPyEngineConfig(dtype=case["dtype"]))
    if kind == "mesh":
        f, m = _mesh_input(case, seed)
        most = _most_vertices(case)
        return dict(kind=kind, field=f, mask=m, grid=_grid(case),
                    vertices=torch.zeros((most, 3), dtype=torch.float64, device="cuda"),
                    faces=torch.zeros((2 * most, 3), dtype=torch.int32, device="cuda"))
    if kind == "adjoint":
        st = _fold(case, seed).stacks[0]
        obs = torch.tensor(_points(case["n"], seed), device="cuda")
        return dict(kind=kind, stack=st, kopts=_kernel(case), obs=obs, target=_target(obs))
    ds = DeviceStack(_fold(case, seed).stacks[0], _kernel(case), CENTER)
    s = dict(kind=kind, ds=ds)
    if kind == "solve":
        return dict(s, form=FORMS[case["form"]])
    s.update(w=_weights(case, seed).cuda())
    if kind == "operator":
        return s
    s.update(gradient=case["gradient"], thr=_levels(case) if case["ids"] else None)
    if kind == "grid":
        return dict(s, grid=_grid(case), prec=_lib.GK_F32 if case["prec"] == "f32" else _lib.GK_F64)
    return dict(s, xyz=torch.tensor(_points(case["n"], seed), device="cuda"))


def _target(obs):
    """Observed field of the misfit: planar layers of the stacks' scale."""
    return 2.0 * obs[:, 2] + 0.1 * obs[:, 0]


# ----------------------------------------------------------------------- run
def _level_volume(level):
    """An octree level as the volume a viewer draws: ids at its voxels, 0 where coarser."""
    v = torch.zeros(math.prod(level.resolution), dtype=torch.int32, device="cuda")
    v[level.voxel_index] = level.ids
    return v


def run(state):
    kind = state["kind"]
    if kind in ("model", "faulted"):
        sol = compute_model(state["model"], state["cfg"])
        out = {"lith": sol.lith_block, "scalar": sol.scalar_field_matrix,
               "thresholds": sol.scalar_field_at_surface_points}
        if kind == "model":
            out["gradient"] = sol.stacks[0].gradient
        else:
            out["fault"] = sol.fault_blocks[0]
            out["octree"] = [_level_volume(o) for o in sol.octrees_output]
        return out
    if kind == "solve":
        # to the rounding floor of the FP64 operator
        w, _ = state["ds"].solve(state["form"], tol=1e-10)
        thr, s = state["ds"].surface_thresholds(w)
        return {"thresholds": thr, "scalar": s}
    if kind == "grid":
        s, g, i = state["ds"].evaluate_lattice(state["grid"], state["w"], state["prec"], state["gradient"], state["thr"])
        if state["prec"] == _lib.GK_F32:
            s, g = s.float(), None if g is None else g.float()
        return {"scalar": s, "gradient": g, "ids": i}
    if kind == "points":
        s, g, i = state["ds"].evaluate_points(state["xyz"], state["w"], _lib.GK_F64, state["gradient"], state["thr"])
        return {"scalar": s, "gradient": g, "ids": i}
    if kind == "operator":
        return {"y": state["ds"].matvec(state["w"])}
    if kind == "adjoint":
        st = state["stack"]
        sp = torch.tensor(st.sp_xyz, dtype=torch.float64, requires_grad=True)
        g = torch.tensor(st.ori_grad, dtype=torch.float64, requires_grad=True)
        s = scalar_field_at(sp, g, st, state["kopts"], state["obs"], CENTER)
        loss = ((s - state["target"]) ** 2).mean()
        loss.backward()
        return {"field": s.detach(), "loss": loss.detach(), "d_points": sp.grad, "d_gradients": g.grad}
    g, lib = state["grid"], _lib.load()
    nv, nf = C.c_int64(0), C.c_int64(0)
    v, f = state["vertices"], state["faces"]
    _lib.check("gk_marching_cubes", lib.gk_marching_cubes(
        handle(0), _ptr(state["field"]), (C.c_int64 * 3)(*g.resolution), _ptr(state["mask"]), 0.0,
        (C.c_double * 3)(*g.origin), (C.c_double * 3)(*g.spacing), _ptr(v), v.shape[0], _ptr(f), f.shape[0],
        C.byref(nv), C.byref(nf), _stream()))
    return {"n_vertices": nv.value, "n_faces": nf.value, "vertices": v, "faces": f}


# ---------------------------------------------------------------------- work
def _pair_flops(points, oris, gradient):
    """Flops of the kernel sums at one point, each pair once: 21 per interface
    source and 24 per orientation, 34 and 46 with the gradient."""
    return points * (34 if gradient else 21) + oris * (46 if gradient else 24)


def work(case):
    kind = case["kind"]
    if kind == "mesh":
        n = case["nx"] * case["ny"] * case["nz"]
        return {"bytes": n * 8 + (n if case["masked"] else 0), "flops": 0}
    if kind == "faulted":
        per = (int(200 * case["scale"]), int(40 * case["scale"])), (int(1600 * case["scale"]), int(320 * case["scale"]))
        n, stacks = case["n"] ** 3, [per[0]] + [per[1]] * 3
        flops = sum((3 * o + p) ** 3 / 3 + n * _pair_flops(p, o, False) for p, o in stacks)
        return {"bytes": n * (4 * 8 + 3 * 4), "flops": flops}
    p, o = case["points"], case["oris"]
    n_unk = _unknowns(case)
    data = 8 * (4 * p + 7 * o)
    if kind == "model":
        n = case["nx"] * case["ny"] * case["nz"]
        return {"bytes": data + n * (12 + (24 if case["gradient"] else 0)),
                "flops": n_unk ** 3 / 3 + n * _pair_flops(p, o, case["gradient"])}
    if kind == "solve":
        k = 2 if case["form"] == "fp64_lu" else 1
        return {"bytes": data + 8 * p, "flops": k * n_unk ** 3 / 3 + p * _pair_flops(p, o, False)}
    if kind == "operator":
        return {"bytes": data + 16 * n_unk, "flops": p * _pair_flops(p, o, False) + o * _pair_flops(p, o, True)}
    if kind == "adjoint":
        n = case["n"]
        return {"bytes": 2 * data + 40 * n,
                "flops": n_unk ** 3 / 3 + n * _pair_flops(p, o, False) + (p + o) * 34 * n +
                2 * p * _pair_flops(p, o, True)}
    n = case["n"] if kind == "points" else case["nx"] * case["ny"] * case["nz"]
    # a kernel range inside the box: only the pairs within it count
    share = min(1.0, 4.19 * (case.get("range", synthetic.RANGE) / 1000.0) ** 3)
    return {"bytes": data + n * (8 + (24 if kind == "points" else 0) + (24 if case["gradient"] else 0) +
                                 (4 if case["ids"] else 0)),
            "flops": share * n * _pair_flops(p, o, case["gradient"])}


# --------------------------------------------------------------------- exact
# The same results from dense FP64 torch: covariance C, its radial derivatives,
# the saddle-point matrix, its direct solution, the sums over the sources.
def _d1(t):                                            # (C'/r) a^2 / c_o
    rho = t.sqrt()
    v = ((5.25 * t - 17.5) * t + 26.25) * rho - 14.0
    return torch.where(t < 1, v, torch.zeros_like(v))


def _c(t):                                             # C / c_o
    rho = t.sqrt()
    v = (((0.75 * t - 3.5) * t + 8.75) * rho - 7.0) * t + 1.0
    return torch.where(t < 1, v, torch.zeros_like(v))


def _diff(x, y, a):
    return (x[:, None, :] - y[None, :, :]) / a


def _sq(h):
    t = (h * h).sum(-1)
    return torch.where(t > 0, t, torch.full_like(t, 1e-280))


def _split(counts):
    starts = np.concatenate([[0], np.cumsum(counts)[:-1]])
    rest = np.setdiff1d(np.arange(int(np.sum(counts))), starts)
    return starts, rest, np.repeat(np.arange(len(counts)), counts)[rest]


class _Exact:
    """One stack's interpolant (i_res 4, gi_res 2, degree-1 drift)."""

    def __init__(self, stack, kopts, dev="cuda", sp=None, grad=None, fault_sp=None):
        t = lambda v: torch.as_tensor(v, dtype=torch.float64, device=dev)   # noqa: E731
        self.a, self.c_o = kopts.range, kopts.c_o
        sp = t(stack.sp_xyz) if sp is None else sp
        self.q, self.qn = t(stack.ori_xyz), t(stack.ori_nugget)
        self.g = t(stack.ori_grad) if grad is None else grad
        ref, rest, surf = _split(stack.counts)
        self.ref, self.rest = sp[torch.as_tensor(ref, device=dev)], sp[torch.as_tensor(rest, device=dev)]
        self.surf = torch.as_tensor(surf, device=dev)
        nug = t(stack.sp_nugget)
        self.nug = nug[torch.as_tensor(rest, device=dev)] + nug[torch.as_tensor(ref, device=dev)][self.surf]
        self.fault = None
        if fault_sp is not None:
            f = t(fault_sp)
            self.fault = (f[torch.as_tensor(rest, device=dev)] - f[torch.as_tensor(ref, device=dev)][self.surf])[:, None]

    def solve(self):
        a, c_o, q, p, p0 = self.a, self.c_o, self.q, self.rest, self.ref[self.surf]
        no, r = q.shape[0], p.shape[0]
        h = _diff(q, q, a)
        tt = _sq(h)
        d1 = _d1(tt)
        d2 = torch.where(tt < 1, 26.25 * (1 - tt) ** 2 / tt.sqrt(), torch.zeros_like(tt))
        d2 = torch.where(tt > 1e-200, d2, torch.zeros_like(tt))
        gg = torch.cat([torch.cat([-(h[..., u] * h[..., v] * d2 + (d1 if u == v else 0.0)) for v in range(3)], 1)
                        for u in range(3)], 0) * (c_o / a ** 2)
        gg = gg + torch.diag(self.qn.repeat(3))
        h1, h2 = _diff(q, p, a), _diff(q, p0, a)
        k1, k2 = _d1(_sq(h1)), _d1(_sq(h2))
        gi = torch.cat([h1[..., u] * k1 - h2[..., u] * k2 for u in range(3)], 0) * (2.0 * c_o / a)
        cc = _c(_sq(_diff(p, p, a))) - _c(_sq(_diff(p, self.ref, a)))[:, self.surf]
        rr = _c(_sq(_diff(self.ref, p, a))) - _c(_sq(_diff(self.ref, self.ref, a)))[:, self.surf]
        ii = 4.0 * c_o * (cc - rr[self.surf]) + torch.diag(self.nug)
        ug = torch.eye(3, dtype=q.dtype, device=q.device).repeat_interleave(no, 0)
        ui = 2.0 * (p - p0)
        if self.fault is not None:
            ug = torch.cat([ug, torch.zeros_like(ug[:, :1])], 1)
            ui = torch.cat([ui, 2.0 * self.fault], 1)
        z = torch.zeros((ui.shape[1],) * 2, dtype=q.dtype, device=q.device)
        m = torch.cat([torch.cat([gg, gi, ug], 1), torch.cat([gi.T, ii, ui], 1), torch.cat([ug.T, ui.T, z], 1)], 0)
        b = torch.cat([self.g.T.reshape(-1), torch.zeros(r + z.shape[0], dtype=q.dtype, device=q.device)])
        return torch.linalg.solve(m, b)

    def field(self, x, w, gradient=False, fault_x=None, chunk=1 << 23):
        """S (and grad S) at x (n, 3), the sources in blocks."""
        no, r = self.q.shape[0], self.rest.shape[0]
        wi = w[3 * no:3 * no + r]
        wr = torch.zeros(self.ref.shape[0], dtype=w.dtype, device=w.device).index_add(0, self.surf, wi)
        src, sw = torch.cat([self.rest, self.ref]) / self.a, 4.0 * self.c_o * torch.cat([wi, -wr])
        q, v = self.q / self.a, 2.0 * self.c_o / self.a * w[:3 * no].reshape(3, no).T.contiguous()
        lam = w[3 * no + r:]
        s = 2.0 * (x @ lam[:3])
        if fault_x is not None and lam.numel() > 3:
            s = s + 2.0 * lam[3] * fault_x
        g = (2.0 * lam[:3]).expand(x.shape[0], 3).clone() if gradient else None
        tile = 1024
        rows = max(1, chunk // tile)
        for x0 in range(0, x.shape[0], rows):
            X = x[x0:x0 + rows] / self.a
            e = slice(x0, x0 + rows)
            for j in range(0, src.shape[0], tile):
                p, pw = src[j:j + tile], sw[j:j + tile]
                h = [X[:, None, d] - p[None, :, d] for d in range(3)]
                t = h[0] * h[0]
                t.addcmul_(h[1], h[1]).addcmul_(h[2], h[2])
                rho = t.sqrt()
                k = (t * 0.75).sub_(3.5).mul_(t).add_(8.75).mul_(rho).sub_(7.0).mul_(t).add_(1.0)
                far = t >= 1.0 if self.a < 1700.0 else None
                if far is not None:
                    k.masked_fill_(far, 0.0)
                s[e] += k @ pw
                if gradient:
                    k = (t * 5.25).sub_(17.5).mul_(t).add_(26.25).mul_(rho).sub_(14.0)
                    if far is not None:
                        k.masked_fill_(far, 0.0)
                    for d in range(3):
                        g[e, d] += ((k * h[d]) @ pw) / self.a
            for j in range(0, no, tile):
                p, pv = q[j:j + tile], v[j:j + tile]
                h = [X[:, None, d] - p[None, :, d] for d in range(3)]
                t = h[0] * h[0]
                t.addcmul_(h[1], h[1]).addcmul_(h[2], h[2])
                rho = t.sqrt()
                k = (t * 5.25).sub_(17.5).mul_(t).add_(26.25).mul_(rho).sub_(14.0)
                far = t >= 1.0 if self.a < 1700.0 else None
                if far is not None:
                    k.masked_fill_(far, 0.0)
                for d in range(3):
                    s[e] -= (k * h[d]) @ pv[:, d]
                if gradient:
                    k2 = (1.0 - t).square_().mul_(26.25).div_(rho.clamp_(min=1e-140))
                    if far is not None:
                        k2.masked_fill_(far, 0.0)
                    dot = sum(h[u] * pv[None, :, u] for u in range(3))
                    k2.mul_(dot)
                    for d in range(3):
                        g[e, d] -= ((k @ pv[:, d]) + (k2 * h[d]).sum(1)) / self.a
        return s, g

    def thresholds(self, w, fault_ref=None):
        return self.field(self.ref, w, fault_x=fault_ref)[0]


def _ids(s, thr):
    up = len(thr) >= 2 and float(thr[0]) < float(thr[-1])
    i = torch.ones_like(s, dtype=torch.int32)
    for k in thr:
        i += (s > k) if up else (s < k)
    return i


def _exact_faulted(case, seed):
    m = prepare(case, seed)["model"]
    x = torch.tensor(m.grid.values(), dtype=torch.float64, device="cuda")
    kopts, rows, thr, fid = m.options.kernel_options, [], [], None
    for st in m.stacks:
        fs = fx = fr = None
        if st.faults:
            e, w, t = fid
            fs = _ids(e.field(torch.tensor(st.sp_xyz, device="cuda"), w)[0], t).double()
            fx, fr = _ids(rows[0], t).double(), fs[torch.as_tensor(_split(st.counts)[0], device="cuda")]
        e = _Exact(st, kopts, fault_sp=fs)
        w = e.solve()
        t = e.thresholds(w, fr)
        rows.append(e.field(x, w, fault_x=fx)[0])
        thr.append(t)
        if fid is None:
            fid = (e, w, t)
    return {"lith": None, "scalar": torch.stack(rows), "thresholds": torch.cat(thr).cpu().numpy(), "fault": None,
            "octree": None}


def exact(case, seed):
    kind = case["kind"]
    if kind == "mesh":
        return {"n_vertices": None, "n_faces": None, "vertices": _exact_vertices(case, seed), "faces": None}
    if kind == "faulted":
        return _exact_faulted(case, seed)
    m = _fold(case, seed)
    if kind == "adjoint":
        st = m.stacks[0]
        sp = torch.tensor(st.sp_xyz, dtype=torch.float64, device="cuda", requires_grad=True)
        g = torch.tensor(st.ori_grad, dtype=torch.float64, device="cuda", requires_grad=True)
        obs = torch.tensor(_points(case["n"], seed), device="cuda")
        s = _obs_field(_Exact(st, _kernel(case), sp=sp, grad=g), obs)
        loss = ((s - _target(obs)) ** 2).mean()
        loss.backward()
        return {"field": s.detach(), "loss": loss.detach(), "d_points": sp.grad, "d_gradients": g.grad}
    e = _Exact(m.stacks[0], _kernel(case))
    if kind == "solve":
        w = e.solve()
        s = e.field(torch.tensor(m.stacks[0].sp_xyz, device="cuda"), w)[0]
        return {"thresholds": e.thresholds(w).cpu().numpy(), "scalar": s}
    if kind == "model":
        w = e.solve()
        x = torch.tensor(_grid(case).values(), device="cuda")
        s, g = e.field(x, w, case["gradient"])
        return {"lith": None, "scalar": s[None], "thresholds": e.thresholds(w).cpu().numpy(), "gradient": g}
    w = _weights(case, seed).cuda()
    if kind == "operator":
        no, r = e.q.shape[0], e.rest.shape[0]
        s = e.field(torch.cat([e.rest, e.ref]), w)[0]
        _, g = e.field(e.q, w, True)
        y1 = (g / 2.0 + e.qn[:, None] * w[:3 * no].reshape(3, no).T).T.reshape(-1)
        y2 = s[:r] - s[r:][e.surf] + e.nug * w[3 * no:3 * no + r]
        y3 = w[:3 * no].reshape(3, no).sum(1) + (2.0 * (e.rest - e.ref[e.surf])).T.contiguous() @ w[3 * no:3 * no + r]
        return {"y": torch.cat([y1, y2, y3])}
    x = torch.tensor(_points(case["n"], seed) if kind == "points" else _grid(case).values(), device="cuda")
    s, g = e.field(x, w, case["gradient"])
    return {"scalar": s, "gradient": g, "ids": None}


def _obs_field(e, x):
    """The field at the observation points, differentiable."""
    w = e.solve()
    no, r = e.q.shape[0], e.rest.shape[0]
    wi = w[3 * no:3 * no + r]
    wr = torch.zeros(e.ref.shape[0], dtype=w.dtype, device=w.device).index_add(0, e.surf, wi)
    h = _diff(x, e.q, e.a)
    s = -(2.0 * e.c_o / e.a) * ((_d1(_sq(h))[..., None] * h) * w[:3 * no].reshape(3, no).T[None]).sum((1, 2))
    s = s + 4.0 * e.c_o * (_c(_sq(_diff(x, e.rest, e.a))) @ wi - _c(_sq(_diff(x, e.ref, e.a))) @ wr)
    return s + 2.0 * (x @ w[3 * no + r:])


def _exact_vertices(case, seed):
    """Crossings of the lattice edges of the meshed cubes, by point then axis."""
    f, m = _mesh_input(case, seed)
    g, n = _grid(case), _res(case)
    f = f.reshape(n)
    cube = torch.ones([k - 1 for k in n], dtype=torch.bool, device=f.device) if m is None else \
        m.reshape(n)[1:, 1:, 1:].bool()
    up = f > 0.0
    pos, key = [], []
    for d in range(3):
        cut = lambda lo, hi: tuple(slice(lo, n[k] + hi) if k == d else slice(0, n[k]) for k in range(3))   # noqa: E731
        v0, v1 = f[cut(0, -1)], f[cut(1, 0)]
        cross = up[cut(0, -1)] ^ up[cut(1, 0)]
        touch = torch.zeros_like(cross)                # edges of a meshed cube
        o = [k for k in range(3) if k != d]
        for i in (0, 1):
            for j in (0, 1):
                at = [slice(0, n[d] - 1)] * 3
                at[o[0]], at[o[1]] = slice(i, n[o[0]] - 1 + i), slice(j, n[o[1]] - 1 + j)
                touch[tuple(at)] |= cube
        idx = (cross & touch).nonzero()
        a0, a1 = v0[tuple(idx.T)], v1[tuple(idx.T)]
        p = idx.double()
        p[:, d] += (0.0 - a0) / (a1 - a0)
        pos.append(p)
        key.append(3 * ((idx[:, 0] * n[1] + idx[:, 1]) * n[2] + idx[:, 2]) + d)
    p = torch.cat(pos)[torch.cat(key).argsort()]
    out = torch.zeros((_most_vertices(case), 3), dtype=torch.float64, device=p.device)
    out[:p.shape[0]] = torch.tensor(g.origin, device=p.device) + p * torch.tensor(g.spacing, device=p.device)
    return out

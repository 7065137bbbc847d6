"""Workloads of the framework as its users run them, for timing and for
checking results: each is one call (or one short sequence of calls) of the C
ABI through p4pdes_amd.capi on a solver that is already set up.

Kinds of case:

  ksp      p4g_ksp_solve_device: A x = b, CG + geometric multigrid, b and x on
           the GPU (fish's linear solve with the set-up kept)
  cells    the same with a cell-centred variable coefficient
  op       p4g_mat_mult_device and p4g_pc_apply_device: one operator and one
           preconditioner application, what a caller's own Krylov loop uses
  vi       p4g_vi_solve: the obstacle problem, grid-sequenced, host arrays
  ms       p4g_ms_solve: the minimal-surface equation, grid-sequenced, host arrays
  serve    a burst of mixed-size requests through the solve server, host arrays

Grids are (g - 1) 2^r + 1 points per side, as -da_grid_x g -da_refine r makes
them, so all sizes are odd and rarely a multiple of a tile.
"""
import collections
import ctypes
import math

import numpy as np
import torch

from p4pdes_amd import capi

CHEB_JACOBI = "-pc_type mg -mg_levels_ksp_type chebyshev -mg_levels_pc_type jacobi -mg_coarse_pc_type cholesky"


# ------------------------------------------------------------------ cases

def listed():
    return [
        # the 129^2 grid of the reference's smallest multigrid studies: launch latency only
        {"name": "fish 2d 129", "kind": "ksp", "dim": 2, "gx": 3, "gy": 3, "gz": 1, "refine": 6,
         "smooth": "jacobi", "steps": 1, "cycle": "v", "mixed": False, "norm": "preconditioned", "rtol": 1e-10},
        # a small 3D problem, as a parameter study solves many of
        {"name": "fish 3d 33", "kind": "ksp", "dim": 3, "gx": 3, "gy": 3, "gz": 3, "refine": 4,
         "smooth": "jacobi", "steps": 1, "cycle": "v", "mixed": False, "norm": "preconditioned", "rtol": 1e-10},
        # the benchmark's 257^3 FP64 solve, the size of the reference's cluster run
        {"name": "fish 3d 257", "kind": "ksp", "dim": 3, "gx": 3, "gy": 3, "gz": 3, "refine": 7,
         "smooth": "jacobi", "steps": 1, "cycle": "v", "mixed": False, "norm": "preconditioned", "rtol": 1e-10},
        # the benchmark's headline: 135 million unknowns, noisy right-hand side, V(2,2), in FP64
        {"name": "fish 3d 513", "kind": "ksp", "dim": 3, "gx": 3, "gy": 3, "gz": 3, "refine": 8,
         "smooth": "jacobi", "steps": 2, "cycle": "v", "mixed": False, "norm": "unpreconditioned", "rtol": 1e-10},
        # the headline with the FP32 V-cycle inside FP64 refinement
        {"name": "fish 3d 513 mixed", "kind": "ksp", "dim": 3, "gx": 3, "gy": 3, "gz": 3, "refine": 8,
         "smooth": "jacobi", "steps": 2, "cycle": "v", "mixed": True, "norm": "unpreconditioned", "rtol": 1e-10},
        # the benchmark's heterogeneous medium, 256^3 cells
        {"name": "cells 257", "kind": "cells", "dim": 3, "gx": 3, "gy": 3, "gz": 3, "refine": 7,
         "smooth": "jacobi", "steps": 1, "cycle": "v", "mixed": False, "norm": "unpreconditioned", "rtol": 1e-10},
        # c/README.md's "-da_refine 9 -pc_type mg": 1025^2 with PETSc's default Chebyshev/SOR smoother
        {"name": "fish 2d 1025 sor", "kind": "ksp", "dim": 2, "gx": 3, "gy": 3, "gz": 1, "refine": 9,
         "smooth": "sor", "steps": 2, "cycle": "v", "mixed": False, "norm": "preconditioned", "rtol": 1e-5},
        # c/ch8/cluster.sh's fish command: 257^3, Chebyshev/SOR, rtol 1e-5, its coarsest grid 9^3
        {"name": "fish 3d 257 sor", "kind": "ksp", "dim": 3, "gx": 9, "gy": 9, "gz": 9, "refine": 5,
         "smooth": "sor", "steps": 2, "cycle": "v", "mixed": False, "norm": "preconditioned", "rtol": 1e-5},
        # a caller's own Krylov method on a box that is no cube: MatMult and PCApply, V(2,2)
        {"name": "op 193x161x129", "kind": "op", "dim": 3, "gx": 7, "gy": 6, "gz": 5, "refine": 5,
         "smooth": "jacobi", "steps": 2, "cycle": "v", "mixed": False, "norm": "preconditioned", "rtol": 1e-10},
        # the obstacle problem as c/ch8/cluster.sh sequences it (33^2 base), its first stages
        {"name": "obstacle 129", "kind": "vi", "gx": 33, "gy": 33, "stages": 3},
        # the minimal-surface equation as c/ch8/cluster.sh sequences it (33^2 base), to 513^2
        {"name": "minimal 513", "kind": "ms", "gx": 33, "gy": 33, "stages": 5},
        # a burst at the server, of the sizes the serving benchmark mixes
        {"name": "serve mix", "kind": "serve", "shapes": "3:33 3:33 3:65 3:129 2:257 2:257 2:1025"},
    ]


def _base(rng, lo, hi):
    """Base points per side of a box whose sides stay within a factor of two."""
    g = rng.randint(lo, hi)
    side = [g] + [max(3, min(hi, int(round((g - 1) * 2 ** rng.uniform(-0.5, 0.5))) + 1)) for _ in range(2)]
    rng.shuffle(side)
    return side


def draw(rng):
    kind = rng.choices(["ksp", "sor", "mixed", "cells", "op", "vi", "ms", "serve"],
                       [6, 3, 2, 2, 2, 1, 1, 1])[0]
    if kind == "vi" or kind == "ms":
        g = rng.randint(9, 33)
        return {"kind": kind, "gx": g, "gy": max(9, min(33, g + rng.randint(-4, 4))),
                "stages": rng.randint(2, 3 if kind == "vi" and g > 20 else 4)}
    if kind == "serve":
        sizes = {2: [65, 129, 257, 513, 1025], 3: [17, 33, 65, 129]}
        shapes = []
        for _ in range(rng.randint(2, 8)):
            dim = rng.choice([2, 3])
            shapes.append("%d:%d" % (dim, rng.choice(sizes[dim])))
        return {"kind": "serve", "shapes": " ".join(shapes)}
    dim = 3 if kind in ("cells", "op") else rng.choice([2, 3, 3])
    # sides of about 2^a points, spread over the logarithm of the size
    top = {("sor", 2): 10, ("sor", 3): 7.5}.get((kind, dim), 8.5 if dim == 3 else 11)
    a = rng.uniform(4 if dim == 3 else 6, top)
    gx, gy, gz = _base(rng, 3, 9)
    refine = max(1, int(round(a - math.log2(max(gx, gy) - 1))))
    if dim == 3:
        while max(gx - 1, gy - 1, gz - 1) * 2 ** refine > 2 ** top * 1.05:
            refine -= 1
    steps = rng.choice([1, 2])
    return {"kind": kind if kind in ("cells", "op") else "ksp", "dim": dim, "gx": gx, "gy": gy,
            "gz": gz if dim == 3 else 1, "refine": refine, "smooth": "sor" if kind == "sor" else "jacobi",
            "steps": steps, "cycle": rng.choice(["v", "v", "v", "w"]) if dim == 2 else "v",
            "mixed": kind == "mixed", "norm": rng.choice(["preconditioned", "unpreconditioned"]),
            "rtol": rng.choice([1e-5, 1e-8]) if kind == "sor" else rng.choice([1e-8, 1e-10])}


def _sides(case):
    m = [(case["g" + c] - 1) * 2 ** case["refine"] + 1 for c in "xyz"]
    return m[:case["dim"]]     # x first


def _options(case):
    o = "-da_grid_x %d -da_grid_y %d -da_grid_z %d -da_refine %d" % (
        case["gx"], case["gy"], max(case["gz"], 3), case["refine"])
    o += " -pc_type mg" if case["smooth"] == "sor" else " " + CHEB_JACOBI
    o += " -mg_levels_ksp_max_it %d -pc_mg_cycle_type %s -ksp_rtol %g" % (case["steps"], case["cycle"], case["rtol"])
    if case["mixed"]:
        return o + " -p4g_precision mixed"
    return o + " -ksp_norm_type %s" % case["norm"]


# ------------------------------------------------------- solvers, kept set up

class Plan:
    """The solver handles one case needs; a program keeps them over many right-hand sides."""

    def __init__(self, case):
        self.case = dict(case)
        self.lib = capi.lib()
        self.lib.p4g_vi_solve.argtypes = [ctypes.c_void_p] * 6
        self.lib.p4g_ms_solve.argtypes = [ctypes.c_void_p, ctypes.c_double] + [ctypes.c_void_p] * 5
        self.keep, self.sessions, self.das, self.solvers, self.server = [], [], [], [], None
        kind = case["kind"]
        if kind in ("ksp", "op"):
            s = capi.Session("-fsh_dim %d -fsh_problem zero %s" % (case["dim"], _options(case)))
            self.sessions.append(s)
            self.solver = s.solver
        elif kind == "cells":
            mx, my, mz = _sides(case)
            self.kcell = _medium(mx - 1, my - 1, mz - 1)
            da = self._da(3, 3, 3, 3, _options(case))
            host = self.kcell.cpu().numpy().ravel()
            capi.check(self.lib.p4g_da_set_cell_coefficient(da, host.ctypes.data))
            self.solver = self._solver(da, _options(case))
            capi.check(self.lib.p4g_solver_setup(self.solver))
        elif kind == "vi":
            self.force = [None] * case["stages"]
            for k in range(case["stages"]):
                opts = "-da_grid_x %d -da_grid_y %d -da_refine %d -pc_type mg" % (case["gx"], case["gy"], k)
                da = self._da(2, 3, 3, 1, opts)
                self._poisson2d(da, case, k)
                self._solver(da, opts)
        elif kind == "ms":
            for k in range(case["stages"]):
                opts = "-da_grid_x %d -da_grid_y %d -da_refine %d -pc_type mg -snes_fd_color" % (
                    case["gx"], case["gy"], k)
                da = self._da(2, 3, 3, 1, opts)
                self._jacobian2d(da)
                self._solver(da, opts)
        elif kind == "serve":
            self.by_shape = {}
            for shape in case["shapes"].split():
                if shape not in self.by_shape:
                    dim, m = (int(v) for v in shape.split(":"))
                    r = (m - 1).bit_length() - 2
                    s = capi.Session("-fsh_dim %d -fsh_problem zero -da_refine %d -pc_mg_levels %d %s "
                                     "-mg_levels_ksp_max_it 1 -p4g_precision mixed -ksp_rtol 1e-8"
                                     % (dim, r, r, CHEB_JACOBI))
                    self.sessions.append(s)
                    self.by_shape[shape] = s.solver
            self.server = capi.Server(16 << 30, "-p4g_serve_staging_mb 256")

    def _da(self, dim, mx, my, mz, opts):
        da = ctypes.c_void_p()
        capi.check(self.lib.p4g_da_create(dim, mx, my, mz, 1.0, 1.0, 1.0, ctypes.byref(da)))
        self.das.append(da)
        capi.check(self.lib.p4g_da_set_from_options(da, opts.encode()))
        return da

    def _solver(self, da, opts):
        s = ctypes.c_void_p()
        capi.check(self.lib.p4g_solver_create(da, opts.encode(), ctypes.byref(s)))
        self.solvers.append(s)
        return s

    def _poisson2d(self, da, case, stage):
        """Residual (-Laplace u - f, u = 0 on the boundary; f from self.force) and Jacobian callbacks."""
        mx, my = (case["gx"] - 1) * 2 ** stage + 1, (case["gy"] - 1) * 2 ** stage + 1
        sx, sy = (mx - 1.0) / (my - 1.0), (my - 1.0) / (mx - 1.0)

        def grid(rows):
            p = ctypes.cast(rows, ctypes.POINTER(ctypes.POINTER(ctypes.c_double)))[0]
            return np.ctypeslib.as_array(p, shape=(my, mx))

        def residual(info, au, aF, ctx):
            u, F = grid(au), grid(aF)
            v = np.zeros((my, mx))
            v[1:-1, 1:-1] = u[1:-1, 1:-1]
            F[:] = 2.0 * (sx + sy) * u
            F[1:-1, 1:-1] -= (sx * (v[1:-1, :-2] + v[1:-1, 2:]) + sy * (v[:-2, 1:-1] + v[2:, 1:-1])
                              + self.force[stage][1:-1, 1:-1] / ((mx - 1) * (my - 1)))
            return 0

        vp = ctypes.c_void_p
        fn = ctypes.CFUNCTYPE(ctypes.c_int, vp, vp, vp, vp)(residual)
        self.keep.append(fn)
        self.lib.p4g_da_set_function_local.argtypes = [vp, vp, vp]
        capi.check(self.lib.p4g_da_set_function_local(da, ctypes.cast(fn, vp), None))
        self._jacobian2d(da)

    def _jacobian2d(self, da):
        """The library's own Poisson Jacobian callback (what obstacle.c and minimal.c register)."""
        vp = ctypes.c_void_p
        ctx = (ctypes.c_double * 9)(1, 1, 1, 1, 1, 1, 0, 0, 0)      # PoissonCtx: unit lengths and coefficients
        self.keep.append(ctx)
        self.lib.p4g_da_set_jacobian_local.argtypes = [vp, vp, vp]
        capi.check(self.lib.p4g_da_set_jacobian_local(
            da, ctypes.cast(capi.fishlib().Poisson2DJacobianLocal, vp), ctypes.cast(ctx, vp)))

    def __del__(self):
        try:
            if self.server is not None:
                self.server.close()
            for s in self.solvers:
                self.lib.p4g_solver_destroy(ctypes.byref(s))
            for da in self.das:
                self.lib.p4g_da_destroy(ctypes.byref(da))
            for s in self.sessions:
                s.close()
        except Exception:      # noqa: BLE001 - interpreter shutting down
            pass


_plans = collections.OrderedDict()


def _plan(case):
    """The case's solver, the last one kept: set-up is paid once for all its right-hand sides."""
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    if key not in _plans:
        _plans.clear()
        _plans[key] = Plan(case)
    return _plans[key]


# ------------------------------------------------------------------ inputs

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _axes(sides):
    return [torch.linspace(0, 1, m, dtype=torch.float64, device=_device()) for m in sides]


def _outer(vs):
    """x-fastest product of per-axis vectors (x first in vs)."""
    out = vs[0]
    for v in vs[1:]:
        out = v.reshape([-1] + [1] * out.dim()) * out
    return out


def _modes(sides, rng, count=8, noise=0.0, seed=0):
    """Sum of random sine modes with N(0,1) amplitudes, plus noise; zero on the boundary."""
    f = None
    xs = _axes(sides)
    for _ in range(count):
        a = float(rng.standard_normal())
        ks = rng.integers(1, 9, size=len(sides))
        t = _outer([torch.sin(math.pi * float(k) * x) for k, x in zip(ks, xs)]) * a
        f = t if f is None else f.add_(t)
    if noise:
        g = torch.Generator(device=_device())
        g.manual_seed(seed)
        f.add_(torch.randn(f.shape, dtype=f.dtype, device=f.device, generator=g), alpha=noise)
    return _clear_boundary(f)


def _clear_boundary(f):
    for ax in range(f.dim()):
        f.select(ax, 0).zero_()
        f.select(ax, f.shape[ax] - 1).zero_()
    return f


def _rhs(case, seed):
    sides = _sides(case)
    rng = np.random.default_rng(seed)
    vol = 1.0 / np.prod([m - 1.0 for m in sides])
    return _modes(sides, rng, noise=1e-3, seed=seed).mul_(vol)


def _medium(nx, ny, nz):
    """exp of a smooth Gaussian random field on the cells (a fixed medium: it belongs to the operator)."""
    rng = np.random.default_rng(11)
    c = [(torch.arange(n, dtype=torch.float64, device=_device()) + 0.5) / n for n in (nx, ny, nz)]
    G = torch.zeros((nz, ny, nx), dtype=torch.float64, device=_device())
    for _ in range(48):
        w = rng.standard_normal(3) / 0.1
        ph = rng.uniform(0, 2 * math.pi)
        arg = (w[2] * c[2]).reshape(-1, 1, 1) + (w[1] * c[1]).reshape(-1, 1) + (w[0] * c[0] + ph)
        G.add_(torch.cos(arg), alpha=math.sqrt(2.0 / 48))
    return torch.exp(G)


def _cells_apply(k, u):
    """-div(k grad u) with the library's row scaling, u zero on the boundary."""
    nz, ny, nx = k.shape
    vol = 1.0 / (nx * ny * nz)
    ax, ay, az = vol * nx * nx, vol * ny * ny, vol * nz * nz
    I = slice(1, -1)
    kx = 0.25 * ax * (k[:-1, :-1] + k[1:, :-1] + k[:-1, 1:] + k[1:, 1:])           # (nz-1, ny-1, nx)
    ky = 0.25 * ay * (k[:-1, :, :-1] + k[1:, :, :-1] + k[:-1, :, 1:] + k[1:, :, 1:])
    kz = 0.25 * az * (k[:, :-1, :-1] + k[:, 1:, :-1] + k[:, :-1, 1:] + k[:, 1:, 1:])
    out = torch.zeros_like(u)
    gx = kx * (u[I, I, 1:] - u[I, I, :-1])
    gy = ky * (u[I, 1:, I] - u[I, :-1, I])
    gz = kz * (u[1:, I, I] - u[:-1, I, I])
    out[I, I, I] = (gx[:, :, :-1] - gx[:, :, 1:] + gy[:, :-1] - gy[:, 1:] + gz[:-1] - gz[1:])
    return out


def _obstacle(case, seed, stage):
    """(psi, f) at the nodes: a dome, as the reference's, that stays below zero at the boundary, and a load."""
    rng = np.random.default_rng(seed)
    my, mx = (case["gy"] - 1) * 2 ** stage + 1, (case["gx"] - 1) * 2 ** stage + 1
    x, y = np.linspace(0, 1, mx)[None, :], np.linspace(0, 1, my)[:, None]
    cx, cy = rng.uniform(0.42, 0.58, 2)
    ax, ay = rng.uniform(2.0, 5.0, 2)
    psi = rng.uniform(0.12, 0.25) - ax * (x - cx) ** 2 - ay * (y - cy) ** 2
    f = np.zeros((my, mx))
    for _ in range(3):
        i, j = rng.integers(1, 4, 2)
        f += rng.standard_normal() * np.sin(i * math.pi * x) * np.sin(j * math.pi * y)
    return psi, f


def _wire(case, seed, stage):
    """Boundary values of a minimal surface: a catenoid's, c random, with a ripple along the frame."""
    rng = np.random.default_rng(seed)
    my, mx = (case["gy"] - 1) * 2 ** stage + 1, (case["gx"] - 1) * 2 ** stage + 1
    x, y = np.linspace(0, 1, mx)[None, :], np.linspace(0, 1, my)[:, None]
    c = rng.uniform(1.15, 1.6)
    g = np.sqrt(np.maximum((c * np.cosh(x / c)) ** 2 - y ** 2, 0.0))
    return np.ascontiguousarray(g + rng.uniform(0.01, 0.04) * np.sin(2 * math.pi * (x + rng.uniform()))
                                * np.cos(2 * math.pi * (y + rng.uniform())))


def _spanned(g):
    """The frame's boundary values carried inward (transfinite interpolation): a first guess of the surface."""
    my, mx = g.shape
    x, y = np.linspace(0, 1, mx)[None, :], np.linspace(0, 1, my)[:, None]
    u = ((1 - x) * g[:, :1] + x * g[:, -1:] + (1 - y) * g[:1] + y * g[-1:]
         - (1 - x) * (1 - y) * g[0, 0] - x * (1 - y) * g[0, -1] - (1 - x) * y * g[-1, 0] - x * y * g[-1, -1])
    return np.ascontiguousarray(u)


def _finer(u):
    """Q1 interpolation of nodal values to the once-refined grid."""
    my, mx = u.shape
    v = np.empty((2 * my - 1, 2 * mx - 1))
    v[::2, ::2] = u
    v[::2, 1::2] = 0.5 * (u[:, 1:] + u[:, :-1])
    v[1::2] = 0.5 * (v[2::2] + v[:-1:2])
    return v


def prepare(case, seed):
    plan = _plan(case)
    kind = case["kind"]
    st = {"case": case, "plan": plan}
    if kind in ("ksp", "op"):
        st["b"] = _rhs(case, seed)
        st["x"] = torch.empty_like(st["b"])
        if kind == "op":
            st["p"] = _rhs(case, seed + 7919) * 1e3
            st["w"] = torch.empty_like(st["b"])
    elif kind == "cells":
        u = _solution(case, seed)
        st["b"] = _cells_apply(plan.kcell, u)
        st["x"] = torch.empty_like(u)
    elif kind == "vi":
        st["grids"] = [_obstacle(case, seed, k) for k in range(case["stages"])]
    elif kind == "ms":
        st["grids"] = [_wire(case, seed, k) for k in range(case["stages"])]
    elif kind == "serve":
        st["reqs"] = []
        for q, shape in enumerate(case["shapes"].split()):
            dim, m = (int(v) for v in shape.split(":"))
            b = _modes([m] * dim, np.random.default_rng([seed, q])).mul_((m - 1.0) ** -dim).cpu().numpy().ravel()
            st["reqs"].append((plan.by_shape[shape], b))
    if torch.cuda.is_available():
        torch.cuda.synchronize()
    return st


def _solution(case, seed):
    return _modes(_sides(case), np.random.default_rng(seed), count=12)


# --------------------------------------------------------------------- run

def run(st):
    kind, plan = st["case"]["kind"], st["plan"]
    L = plan.lib
    if kind in ("ksp", "cells"):
        rep = capi.Report()
        capi.check(L.p4g_ksp_solve_device(plan.solver, st["b"].data_ptr(), st["x"].data_ptr(), ctypes.byref(rep)))
        if rep.reason <= 0:
            raise RuntimeError("the solve did not converge: %s" % capi.REASONS.get(rep.reason, rep.reason))
        return st["x"]
    if kind == "op":
        capi.check(L.p4g_mat_mult_device(plan.solver, st["p"].data_ptr(), st["w"].data_ptr()))
        capi.check(L.p4g_pc_apply_device(plan.solver, st["b"].data_ptr(), st["x"].data_ptr()))
        return [st["w"], st["x"]]
    if kind == "vi":
        u = F = None
        for k, (psi, f) in enumerate(st["grids"]):
            plan.force[k] = f
            u = np.zeros_like(psi) if k == 0 else _finer(u)
            F = np.empty_like(u)
            rep = capi.VIReport()
            capi.check(L.p4g_vi_solve(plan.solvers[k], psi.ctypes.data, None, u.ctypes.data, F.ctypes.data,
                                      ctypes.addressof(rep)))
            if rep.reason <= 0:
                raise RuntimeError("obstacle stage %d did not converge (%d)" % (k, rep.reason))
        return [u, F]
    if kind == "ms":
        u = None
        for k, g in enumerate(st["grids"]):
            u = _spanned(g) if k == 0 else _finer(u)
            rep = (ctypes.c_char * 256)()
            capi.check(L.p4g_ms_solve(plan.solvers[k], -0.5, g.ctypes.data, u.ctypes.data, None, None,
                                      ctypes.addressof(rep)))
            if ctypes.c_int.from_buffer(rep, 4).value <= 0:
                raise RuntimeError("minimal-surface stage %d did not converge" % k)
        return u
    ids = [plan.server.submit(solver, b) for solver, b in st["reqs"]]
    return [plan.server.wait(i)[0] for i in ids]


# -------------------------------------------------------------------- work

def _solve_bytes(n, dim, word, its, steps, coef=0.0):
    """CG iterations of 9 vector moves (p = z + b p; w = A p; r -= a w; x += a p), each with a V-cycle of
    2 + 2 + 3 moves (smooth, residual and restriction, prolongation and smoothing; sweeps of one smoothing in
    one pass) over the levels, and `coef` coefficient vectors read by each of the four operator passes."""
    levels = 8.0 / 7.0 if dim == 3 else 4.0 / 3.0
    return its * n * word * (9 + coef + levels * (7 + 3 * coef))


def work(case):
    kind = case["kind"]
    if kind in ("ksp", "cells", "op"):
        n, dim = float(np.prod(_sides(case))), case["dim"]
        if kind == "op":
            return {"bytes": 8 * n * (2 + 8.0 / 7.0 * 7), "flops": n * (13 + 8.0 / 7.0 * (17 * 2 * case["steps"] + 30))}
        digits = -math.log10(case["rtol"])
        per = 0.9 if case["smooth"] == "sor" else 2.0 if kind == "cells" else 1.2
        its = max(2.0, round(per * digits))
        flops = its * n * (25 + 8.0 / 7.0 * (17 * 2 * case["steps"] * (2 if case["smooth"] == "sor" else 1) + 30))
        return {"bytes": _solve_bytes(n, dim, 4 if case["mixed"] else 8, its, case["steps"],
                                      1.0 if kind == "cells" else 0.0) + 16 * n, "flops": flops}
    if kind in ("vi", "ms"):
        n = sum(((case["gx"] - 1) * 2.0 ** k + 1) * ((case["gy"] - 1) * 2.0 ** k + 1) for k in range(case["stages"]))
        its = 3 * 6.0            # Newton steps of a few Krylov iterations each, 9 operator planes
        return {"bytes": _solve_bytes(n, 2, 8, its, 2, 9.0) + 24 * n, "flops": its * n * 300}
    total = 0.0
    for shape in case["shapes"].split():
        dim, m = (int(v) for v in shape.split(":"))
        total += _solve_bytes(float(m) ** dim, dim, 4, 10, 1) + 16.0 * float(m) ** dim
    return {"bytes": total, "flops": total}


# --------------------------------------------------------------- tolerance

def tolerance(case):
    """Four times the error against exact() that was measured: the solves are stopped by their tolerance, so
    another implementation's iterate differs by up to that error; one application differs by rounding only."""
    kind = case["kind"]
    if kind in ("ksp", "cells"):
        return {"rel": 4.0 * case["rtol"] if case["rtol"] <= 1e-8 else case["rtol"]}
    return {"rel": {"op": 1e-12, "vi": 1e-9, "ms": 1e-8, "serve": 2e-9}[kind]}


# ------------------------------------------------------------------- exact

def _sine(m):
    """Orthonormal symmetric matrix of interior sine modes and the 1D eigenvalues times h^2."""
    k = torch.arange(1, m - 1, dtype=torch.float64, device=_device())
    S = torch.sin(math.pi / (m - 1) * torch.outer(k, k)) * math.sqrt(2.0 / (m - 1))
    return S, 4.0 * torch.sin(0.5 * math.pi / (m - 1) * k) ** 2


def _along(S, t, ax):
    """S applied along axis ax."""
    t = t.movedim(ax, -1).contiguous()
    return torch.mm(t.reshape(-1, t.shape[-1]), S).reshape(t.shape).movedim(-1, ax)


def _scales(sides):
    vol = 1.0 / np.prod([m - 1.0 for m in sides])
    return [vol * (m - 1.0) ** 2 for m in sides]


class Poisson:
    """The constant-coefficient operator's inverse in the sine basis (interior points)."""

    def __init__(self, sides):
        self.sides = sides
        self.S, lam = zip(*[_sine(m) for m in sides])
        sc = _scales(sides)
        self.lam = sum((s * l).reshape([-1] + [1] * q) for q, (s, l) in enumerate(zip(sc, lam)))

    def transform(self, t):
        d = len(self.sides)
        for q in range(d):
            t = _along(self.S[q], t, d - 1 - q)
        return t

    def solve(self, b):
        return self.transform(self.transform(b) / self.lam)

    def full(self, t):
        out = torch.zeros([m for m in reversed(self.sides)], dtype=t.dtype, device=t.device)
        out[(slice(1, -1),) * t.dim()] = t
        return out


def _inner(t):
    return t[(slice(1, -1),) * t.dim()]


def _laplace(sides, u):
    """The interior rows of the operator applied to u (zero on the boundary)."""
    sc = _scales(sides)
    d = len(sides)
    out = 0.0
    for q in range(d):
        ax = d - 1 - q
        mid = [slice(1, -1)] * d
        lo, hi = list(mid), list(mid)
        lo[ax], hi[ax] = slice(0, -2), slice(2, None)
        out = out + sc[q] * (2.0 * u[tuple(mid)] - u[tuple(lo)] - u[tuple(hi)])
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "cells":
        return _solution(case, seed)
    if kind == "ksp":
        P = Poisson(_sides(case))
        return P.full(P.solve(_inner(_rhs(case, seed))))
    if kind == "op":
        p = _rhs(case, seed + 7919) * 1e3
        w = torch.zeros_like(p)
        w[(slice(1, -1),) * 3] = _laplace(_sides(case), p)
        return [w, None]
    if kind == "serve":
        out = []
        for q, shape in enumerate(case["shapes"].split()):
            dim, m = (int(v) for v in shape.split(":"))
            P = Poisson([m] * dim)
            b = _modes([m] * dim, np.random.default_rng([seed, q])).mul_((m - 1.0) ** -dim)
            out.append(P.full(P.solve(_inner(b))).reshape(-1))
        return out
    if kind == "vi":
        return _exact_obstacle(case, seed)
    return _exact_minimal(case, seed)


def _exact_obstacle(case, seed):
    """The discrete variational inequality by active sets; each reduced system by CG with the sine-basis
    inverse restricted to the inactive vertices."""
    stage = case["stages"] - 1
    psi, f = (torch.from_numpy(a).to(_device()) for a in _obstacle(case, seed, stage))
    sides = [psi.shape[1], psi.shape[0]]
    P = Poisson(sides)
    psi = _inner(psi)
    rhs = _inner(f) / ((sides[0] - 1.0) * (sides[1] - 1.0))
    A = lambda v: _laplace(sides, P.full(v))       # noqa: E731
    c = float(P.lam.max())
    u = torch.maximum(P.solve(rhs), psi)
    act = torch.zeros_like(psi, dtype=torch.bool)
    for _ in range(200):
        new = (rhs - A(u)) + c * (u - psi) < 0
        new &= u <= psi + 1e-9 if act.any() else new
        if act.any() and bool((new == act).all()):
            break
        act = new
        free = (~act).to(psi.dtype)
        u = torch.where(act, psi, u)
        r = free * (rhs - A(u))
        z = free * P.solve(r)
        p, rz, r0 = z.clone(), float((r * z).sum()), float(r.norm())
        for _ in range(2000):
            if float(r.norm()) <= 1e-13 * max(r0, 1e-300):
                break
            w = free * A(p)
            al = rz / float((p * w).sum())
            u = u + al * p
            r = r - al * w
            z = free * P.solve(r)
            rz, old = float((r * z).sum()), rz
            p = z + (rz / old) * p
        u = torch.where(act, u, torch.maximum(u, psi))
    full = P.full(u)
    F = P.full(A(u) - rhs)
    return [full.cpu().numpy(), F.cpu().numpy()]


def _ms_residual(u, hx, hy):
    """c/ch7/minimal.c:230-301 at the interior nodes, q = -1/2."""
    C, E, W = u[1:-1, 1:-1], u[1:-1, 2:], u[1:-1, :-2]
    N, S = u[2:, 1:-1], u[:-2, 1:-1]
    NE, NW, SE, SW = u[2:, 2:], u[2:, :-2], u[:-2, 2:], u[:-2, :-2]
    D = lambda a, b: (1.0 + a * a + b * b) ** -0.5     # noqa: E731
    De = D((E - C) / hx, (N + NE - S - SE) / (4 * hy))
    Dw = D((C - W) / hx, (NW + N - SW - S) / (4 * hy))
    Dn = D((E + NE - W - NW) / (4 * hx), (N - C) / hy)
    Ds = D((E + SE - W - SW) / (4 * hx), (C - S) / hy)
    return -(hy / hx) * (De * (E - C) - Dw * (C - W)) - (hx / hy) * (Dn * (N - C) - Ds * (C - S))


def _exact_minimal(case, seed):
    """The discrete minimal surface by Anderson acceleration of u <- u - Laplace^-1 F(u) / D."""
    g = torch.from_numpy(_wire(case, seed, case["stages"] - 1)).to(_device())
    sides = [g.shape[1], g.shape[0]]
    hx, hy = 1.0 / (sides[0] - 1), 1.0 / (sides[1] - 1)
    P = Poisson(sides)
    u = g.clone()
    u[1:-1, 1:-1] = 0.0
    u[1:-1, 1:-1] = P.solve(-_laplace(sides, u))      # the harmonic surface on the same frame
    xs, gs = [], []
    x = u[1:-1, 1:-1].reshape(-1).clone()
    for it in range(400):
        u[1:-1, 1:-1] = x.reshape(sides[1] - 2, sides[0] - 2)
        d = -1.3 * P.solve(_ms_residual(u, hx, hy)).reshape(-1)
        if float(d.norm()) <= 1e-14 * float(x.norm()):
            break
        xs, gs = (xs + [x])[-13:], (gs + [d])[-13:]
        if len(xs) > 1:
            dG = torch.stack([gs[i + 1] - gs[i] for i in range(len(gs) - 1)], 1)
            dX = torch.stack([xs[i + 1] - xs[i] for i in range(len(xs) - 1)], 1)
            gam = torch.linalg.lstsq(dG.cpu(), d.cpu().reshape(-1, 1), driver="gelsd").solution.to(d.device)
            x = x + d - ((dX + dG) @ gam).reshape(-1)
        else:
            x = x + d
    u[1:-1, 1:-1] = x.reshape(sides[1] - 2, sides[0] - 2)
    return u.cpu().numpy()

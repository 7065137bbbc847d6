"""The block factorization of a coarsest Newton operator (k_blk_factor,
k_blk_inverse) at band widths on either side of each rule: blocks of 16 rows
(narrow bands), 4 MR rows of 16, 36 and 63, one block, and a last block that
is not full.  The obstacle is symmetric in x and y, so a grid and its
transpose (another band width; from 64 on another path) have one solution;
each is converged to rtol 1e-12 and the coarse solve is direct, so both agree
to 1e-9 of the norm and take the same Newton steps.  The minimal surface's
finite-difference Jacobian is not symmetric: there two Newton steps with
loosely solved systems, whose result depends on the preconditioner, are
compared with the oracle."""
import ctypes
import itertools

import numpy as np
import pytest

from oracle import oracle_py as O
from p4pdes_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cx,cy", [(3, 5), (3, 70), (15, 66), (16, 20), (35, 40), (36, 56), (28, 64), (62, 9)])
def test_coarse_blocks_transposed(cx, cy):
    sols = []
    for gx, gy in ((cx, cy), (cy, cx)):
        print("coarse blocks", gx, gy, flush=True)
        rc, text, res, u = capi.obstacle_run(
            "-da_grid_x %d -da_grid_y %d -da_refine 1 -pc_type mg -pc_mg_levels 2 -ksp_rtol 1e-12 -snes_rtol 1e-12"
            % (gx, gy), want_u=True)
        assert rc == 0 and res.reason > 0, text
        sols.append((res, u.reshape(2 * gy - 1, 2 * gx - 1)))
    (r0, u0), (r1, u1) = sols
    assert np.abs(u0).max() > 0
    assert r0.its == r1.its
    assert np.linalg.norm(u0 - u1.T) <= 1e-9 * np.linalg.norm(u0)


# blocks of 16 rows, 4 MR rows of 16, 36 and 63, and bands of 64 and more (band LU on the host)
@pytest.mark.parametrize("cx,cy", [(5, 11), (3, 60), (15, 16), (16, 20), (35, 20), (36, 20), (62, 9), (63, 9), (66, 15)])
def test_coarse_blocks_nonsymmetric(cx, cy):
    args = ("-da_grid_x %d -da_grid_y %d -da_refine 1 -ms_problem tent -ms_tent_H 3 -snes_fd_color -pc_type mg "
            "-pc_mg_levels 2 -snes_max_it 2 -ksp_rtol 1e-2" % (cx, cy))
    print("coarse blocks, nonsymmetric", cx, cy, flush=True)
    rc, text, res, u = capi.minimal_run(args, want_u=True)
    assert rc == 0, text
    rc, text, ores, ou = O.minimal_run(args, want_u=True)
    assert rc == 0, text
    assert res.its == ores.its == 2
    assert res.ksp_its_total == ores.ksp_its_total
    # the finite differences turn a rounding of F into 1e-8 of a coefficient;
    # an inverse of the transposed operator, or with the couplings between two
    # blocks exchanged, moves u by 8e-6 to 3e-3 of its maximum (in the oracle)
    assert np.max(np.abs(u - ou)) <= 1e-7 * np.max(np.abs(ou))


def _vi_box(m, psi, f, opts, dim=3):
    """p4g_vi_solve of -Laplace u >= f, u >= psi on a box of m points (x first); psi, f indexed (z, y, x)."""
    L, vp = capi.lib(), ctypes.c_void_p
    r = 1
    base = [(v - 1) // 2 + 1 for v in m]
    o = ("-da_grid_x %d -da_grid_y %d -da_grid_z %d -da_refine %d -pc_type mg -pc_mg_levels 2 %s"
         % (*base, r, opts)).encode()
    da, solver, rep = vp(), vp(), capi.VIReport()
    ctx = (ctypes.c_double * 9)(1, 1, 1, 1, 1, 1, 0, 0, 0)      # PoissonCtx: unit lengths and coefficients
    load = np.ascontiguousarray(-f / np.prod([v - 1.0 for v in m[:dim]]))

    def residual(info, au, aF, c):                              # the solver asks for F(0) only
        p = ctypes.cast(aF, ctypes.POINTER(ctypes.c_double))
        for _ in range(dim - 1):
            p = ctypes.cast(p, ctypes.POINTER(ctypes.POINTER(ctypes.c_double)))[0]
        np.ctypeslib.as_array(p, shape=(load.size,))[:] = load.ravel()
        return 0

    cb = ctypes.CFUNCTYPE(ctypes.c_int, vp, vp, vp, vp)(residual)
    L.p4g_da_set_function_local.argtypes = [vp, vp, vp]
    L.p4g_da_set_jacobian_local.argtypes = [vp, vp, vp]
    capi.check(L.p4g_da_create(dim, 3, 3, 3, 1.0, 1.0, 1.0, ctypes.byref(da)))
    try:
        capi.check(L.p4g_da_set_from_options(da, o))
        capi.check(L.p4g_da_set_function_local(da, ctypes.cast(cb, vp), None))
        jac = getattr(capi.fishlib(), "Poisson%dDJacobianLocal" % dim)
        capi.check(L.p4g_da_set_jacobian_local(da, ctypes.cast(jac, vp), ctypes.cast(ctx, vp)))
        capi.check(L.p4g_solver_create(da, o, ctypes.byref(solver)))
        lo = np.ascontiguousarray(psi)
        u = np.zeros_like(lo)
        capi.check(L.p4g_vi_solve(solver, lo.ctypes.data, None, u.ctypes.data, None, ctypes.byref(rep)))
        return rep, u
    finally:
        L.p4g_solver_destroy(ctypes.byref(solver))
        L.p4g_da_destroy(ctypes.byref(da))


# coarsest boxes whose band is below 64 in every order of their sides, and one that is 73 or 65 (host) in some
@pytest.mark.parametrize("base", [(2, 3, 4), (3, 4, 5), (3, 5, 7), (3, 8, 8)])
def test_coarse_blocks_3d_in_every_order(base):
    # a box's sides in another order: another band and another set of
    # couplings, the same iterates up to rounding (Jacobi smoothing without
    # estimated bounds).  Two Newton steps of loosely solved systems, whose
    # result depends on the coarse inverse
    rng = np.random.default_rng(base)
    mx, my, mz = m = [2 * (b - 1) + 1 for b in base]
    z, y, x = np.meshgrid(*[np.linspace(0, 1, v) for v in (mz, my, mx)], indexing="ij")
    psi = 0.05 - 3 * (x - 0.45) ** 2 - 2 * (y - 0.55) ** 2 - 4 * (z - 0.5) ** 2
    f = rng.standard_normal(psi.shape)
    ref = None
    for order in itertools.permutations(range(3)):              # axis order[i] of (z, y, x) becomes axis i
        print("coarse blocks 3d", base, order, flush=True)
        p, g = psi.transpose(order), f.transpose(order)
        rep, u = _vi_box(p.shape[::-1], np.ascontiguousarray(p), np.ascontiguousarray(g),
                         "-mg_levels_ksp_type richardson -mg_levels_ksp_richardson_scale 0.7 "
                         "-mg_levels_pc_type jacobi -ksp_rtol 1e-2 -snes_max_it 2")
        u = u.transpose(np.argsort(order))
        if ref is None:
            ref = rep, u
            assert rep.ksp_its_total > 0 and np.abs(u).max() > 0
        assert (rep.its, rep.ksp_its_total, rep.active) == (ref[0].its, ref[0].ksp_its_total, ref[0].active)
        diff = np.abs(u - ref[1]).max() / np.abs(ref[1]).max()
        assert diff <= 1e-11


@pytest.mark.parametrize("cx", [3, 16, 17, 500])
def test_coarse_blocks_1d(cx):
    # one dimension: a tridiagonal coarsest operator; converged, against the
    # complementarity conditions themselves
    m = 2 * (cx - 1) + 1
    x = np.linspace(0, 1, m)
    psi = 0.1 - 2 * (x - 0.4) ** 2
    f = -1.0 - np.sin(5 * x)
    print("coarse blocks 1d", m, flush=True)
    rep, u = _vi_box((m, 3, 3), psi, f, "-mg_levels_pc_type jacobi -ksp_rtol 1e-13 -snes_rtol 1e-10 -snes_max_it 200", dim=1)
    assert rep.reason > 0
    h = 1.0 / (m - 1)
    F = np.zeros(m)
    v = np.concatenate([[0.0], u[1:-1], [0.0]])
    F[1:-1] = (2 * v[1:-1] - v[:-2] - v[2:]) / h - f[1:-1] * h
    assert (u >= psi - 1e-12).all()
    free = u[1:-1] > psi[1:-1] + 1e-7
    assert free.any() and np.abs(F[1:-1][free]).max() <= 1e-8 * np.abs(f * h).max()

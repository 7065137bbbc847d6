"""Pipelined SOR sweeps (k_sor2, k_sor7) against the hyperplane sweeps
(k_sor_plane): every point is updated from the same values in the same order,
so one preconditioner application agrees bit for bit, and with it a whole
Newton solve whose levels have 9-point operators.  One-level grids take
any size (the smoother is the preconditioner): the edges of a strip's 64 rows,
of the batches of steps and of the plane groups, 35 strips (on two XCDs), 258
(two launches), single interior points, 3D strips whose steps just fill 64 or
128 or go one past, and boxes longer in each direction."""
import ctypes
import threading
import time

import numpy as np
import pytest

from p4pdes_amd import capi

pytestmark = pytest.mark.gpu

GRIDS_2D = [(19, 2200), (5, 16500), (3, 3), (4, 3), (3, 70), (35, 5), (66, 66), (67, 65), (34, 131), (130, 67), (260, 130), (97, 200)]
GRIDS_3D = [(3, 3, 3), (4, 5, 6), (66, 5, 3), (5, 66, 7), (6, 67, 8), (7, 4, 70), (33, 34, 35), (67, 130, 9), (65, 65, 65),
            (33, 33, 9), (34, 33, 9), (3, 63, 5), (3, 64, 5), (3, 66, 5), (3, 67, 5), (98, 32, 11)]


def _apply(args, b):
    with capi.Session(args) as s:
        assert s.n == b.size
        A = capi.Solver(s)
        return A.pc_apply(b), A.pc_apply(b)


def _pair(args, n, seed):
    b = np.random.default_rng(seed).standard_normal(n)
    print("sor pair", args, flush=True)
    z0, _ = _apply(args + " -p4g_sor_pipeline 0", b)
    z1, z2 = _apply(args, b)
    assert np.isfinite(z0).all()
    assert np.array_equal(z0, z1), np.max(np.abs(z1 - z0))
    assert np.array_equal(z1, z2)          # the tags of the next sweeps


@pytest.mark.parametrize("grid", GRIDS_2D, ids=lambda g: "x".join(map(str, g)))
def test_sor2_matches_hyperplanes(grid):
    mx, my = grid
    _pair("-fsh_dim 2 -fsh_problem zero -fsh_cx 1.7 -da_grid_x %d -da_grid_y %d -pc_type mg -pc_mg_levels 1 "
          "-mg_levels_ksp_max_it 2" % (mx, my), mx * my, mx + my)


@pytest.mark.parametrize("grid", GRIDS_3D, ids=lambda g: "x".join(map(str, g)))
def test_sor7_matches_hyperplanes(grid):
    mx, my, mz = grid
    _pair("-fsh_dim 3 -fsh_problem zero -fsh_cx 1.7 -fsh_cz 0.6 -da_grid_x %d -da_grid_y %d -da_grid_z %d "
          "-pc_type mg -pc_mg_levels 1 -mg_levels_ksp_max_it 3" % (mx, my, mz), mx * my * mz, mx + my + mz)


def test_sor2_multigrid_matches_hyperplanes():
    _pair("-fsh_dim 2 -fsh_problem zero -da_refine 8 -pc_type mg -pc_mg_cycle_type w", 513 * 513, 5)


# 9-point levels: one strip and less, edges of strips and of batches of steps, 35 strips (on two XCDs), 258 (two launches)
GRIDS_9PT = [(3, 3), (5, 4), (35, 5), (67, 65), (130, 67), (97, 200), (19, 2200), (5, 16500)]


def _newton_pair(run, args, mg):
    print("sor9 pair", args, mg, flush=True)
    out = []
    for extra in (" -p4g_sor_pipeline 0", ""):
        rc, text, res, u = run(args + " -pc_type mg -pc_mg_levels %d" % mg + extra, want_u=True)
        assert rc == 0, text
        out.append((res.its, res.ksp_its_total, res.reason, res.fnorm, u))
    assert out[0][1] > 0                   # the preconditioner was applied
    assert np.isfinite(out[0][4]).all()
    assert out[0][:4] == out[1][:4]
    assert np.array_equal(out[0][4], out[1][4])


@pytest.mark.parametrize("grid", GRIDS_9PT, ids=lambda g: "x".join(map(str, g)))
def test_sor9_matches_hyperplanes(grid):
    # one level (the smoother is the preconditioner): the obstacle problem's
    # reduced operator, two Newton steps of loosely solved systems
    _newton_pair(capi.obstacle_run, "-da_grid_x %d -da_grid_y %d -ksp_rtol 0.3 -snes_max_it 2" % grid, 1)


@pytest.mark.parametrize("grid", [(5, 4), (35, 5), (67, 65), (66, 130)], ids=lambda g: "x".join(map(str, g)))
def test_sor9_nonsymmetric_matches_hyperplanes(grid):
    # the minimal surface's finite-difference Jacobian
    _newton_pair(capi.minimal_run, "-da_grid_x %d -da_grid_y %d -snes_fd_color -ksp_rtol 0.3 -snes_max_it 2" % grid, 1)


def test_sor9_multigrid_matches_hyperplanes():
    _newton_pair(capi.obstacle_run, "-da_grid_x 10 -da_grid_y 12 -da_refine 4", 5)
    _newton_pair(capi.minimal_run, "-da_grid_x 9 -da_grid_y 10 -da_refine 3 -snes_fd_color", 4)


def test_sor2_stall_stops_the_solve():
    # a 2D sweep of two strips whose waits cannot succeed: every kernel ends
    # and the solve reports it; a fresh solve then runs normally
    args = "-fsh_dim 2 -fsh_problem manupoly -da_refine 6 -pc_type mg -ksp_rtol 1e-8"
    rc, text, _, _ = capi.fish_run(args + " -p4g_sor_test_stall 1")
    assert rc == 76, text
    assert "pipelined SOR sweep stalled" in text
    rc, text, _, _ = capi.fish_run(args)
    assert rc == 0, text


# grids of several strips, and 3D plane groups; Richardson smoothing, so that set-up runs no sweeps
STALLS = {"2d": ("-fsh_dim 2 -fsh_problem zero -da_grid_x 40 -da_grid_y 200", 40 * 200),
          "3d": ("-fsh_dim 3 -fsh_problem zero -da_grid_x 6 -da_grid_y 67 -da_grid_z 18", 6 * 67 * 18)}
RICH = " -pc_type mg -pc_mg_levels 1 -mg_levels_ksp_type richardson -mg_levels_ksp_max_it 2"


def _call(s, entry, b):
    """(error code, result) of one entry point on device copies of b."""
    L = capi.lib()
    d = [L.p4g_device_malloc(b.nbytes) for _ in range(2)]
    try:
        capi.check(L.p4g_memcpy_htod(d[0], b.ctypes.data, b.nbytes))
        if entry == "ksp":
            rep = capi.Report()
            rc = L.p4g_ksp_solve_device(s.solver, d[0], d[1], ctypes.byref(rep))
        else:
            rc = getattr(L, "p4g_pc_apply_device" + entry)(s.solver, d[0], d[1])
        x = np.empty_like(b)
        capi.check(L.p4g_memcpy_dtoh(x.ctypes.data, d[1], b.nbytes))
        return rc, x
    finally:
        for p in d:
            L.p4g_device_free(p)


@pytest.mark.parametrize("entry", ["", "_noalloc", "ksp"])
@pytest.mark.parametrize("dim", sorted(STALLS))
def test_stalled_call_is_reported_and_the_next_is_right(dim, entry):
    # the first call's waits give up at once: it must say so, and leave nothing
    # behind that a later call on the handle could take for its own
    args, n = STALLS[dim]
    b = np.random.default_rng(n).standard_normal(n)
    print("sor stall", dim, entry, flush=True)
    with capi.Session(args + RICH + " -p4g_sor_pipeline 0") as s:
        capi.check(capi.lib().p4g_solver_setup(s.solver))
        rc, ref = _call(s, entry, b)
        assert rc == 0
    with capi.Session(args + RICH + " -p4g_sor_test_stall once") as s:
        capi.check(capi.lib().p4g_solver_setup(s.solver))
        rc, _ = _call(s, entry, b)
        assert rc == 76 and "pipelined SOR sweep stalled" in capi.last_error()
        for _ in range(2):
            rc, x = _call(s, entry, b)
            assert rc == 0
            assert np.array_equal(x, ref)


def test_stall_during_setup_is_reported():
    # the eigenvalue estimates run sweeps: bounds from a stalled one must not stay
    L, vp = capi.lib(), ctypes.c_void_p
    ctx = (ctypes.c_double * 9)(1, 1, 1, 1, 1, 1, 0, 0, 0)      # PoissonCtx: unit lengths and coefficients
    L.p4g_da_set_jacobian_local.argtypes = [vp, vp, vp]

    def bounds(extra, codes):
        opts = ("-da_grid_x 11 -da_grid_y 101 -da_refine 1 -pc_type mg" + extra).encode()
        da, solver, rep = vp(), vp(), capi.Report()
        capi.check(L.p4g_da_create(2, 3, 3, 1, 1.0, 1.0, 1.0, ctypes.byref(da)))
        try:
            capi.check(L.p4g_da_set_from_options(da, opts))
            capi.check(L.p4g_da_set_jacobian_local(da, ctypes.cast(capi.fishlib().Poisson2DJacobianLocal, vp),
                                                   ctypes.cast(ctx, vp)))
            capi.check(L.p4g_solver_create(da, opts, ctypes.byref(solver)))
            for code in codes:
                assert L.p4g_solver_setup(solver) == code
                if code:
                    assert "PCSetUp: a pipelined SOR sweep stalled" in capi.last_error()
            capi.check(L.p4g_solver_get_report(solver, ctypes.byref(rep)))
            return rep.emax_fine
        finally:
            L.p4g_solver_destroy(ctypes.byref(solver))
            L.p4g_da_destroy(ctypes.byref(da))

    assert bounds(" -p4g_sor_test_stall once", [76, 0]) == bounds(" -p4g_sor_pipeline 0", [0]) > 0


@pytest.mark.parametrize("polls", [1 << 12, 1 << 22])
def test_late_neighbour_is_awaited_to_the_limit(polls):
    # a strip that waits for the one before it polls through L2, 0.35 us each
    # (0.3 allowed for); the chain of steps, which waits in LDS, must not give
    # up for it first.  1.5 s at the larger limit, a quarter of the real one
    args, n = STALLS["2d"]
    print("sor late neighbour", polls, flush=True)
    with capi.Session(args + RICH + " -p4g_sor_test_stall %d" % polls) as s:
        b = np.ones(n)
        t = time.perf_counter()
        rc, _ = _call(s, "", b)
        t = time.perf_counter() - t
    assert rc == 76 and "pipelined SOR sweep stalled" in capi.last_error()
    assert t >= 0.3e-6 * polls


def test_sweeps_of_several_solvers_at_once():
    # solvers on threads of their own, each with its own stream and sweep
    # arrays: 35 strips on two XCDs, 16 on one, 3D plane groups; every result
    # is the one that the solver gives alone
    args = ["-fsh_dim 2 -fsh_problem zero -da_grid_x 19 -da_grid_y 2200 -pc_mg_levels 1",
            "-fsh_dim 2 -fsh_problem zero -da_refine 9", "-fsh_dim 2 -fsh_problem zero -da_refine 9",
            "-fsh_dim 3 -fsh_problem zero -da_refine 6", "-fsh_dim 3 -fsh_problem zero -da_grid_x 5 -da_refine 5"]
    sessions = [capi.Session(a + " -pc_type mg") for a in args]
    bad = []
    try:
        rhs = [np.random.default_rng(i).standard_normal(s.n) for i, s in enumerate(sessions)]
        alone = [capi.Solver(s).pc_apply(b) for s, b in zip(sessions, rhs)]

        def work(i):
            for _ in range(8):
                if not np.array_equal(capi.Solver(sessions[i]).pc_apply(rhs[i]), alone[i]):
                    bad.append(i)

        print("sweeps at once", flush=True)
        threads = [threading.Thread(target=work, args=(i,)) for i in range(len(sessions))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    finally:
        for s in sessions:
            s.close()
    assert not bad

"""The coarse end of a V-cycle in one launch (k_vtail) against the separate
passes it stands for, one preconditioner application: the same formulas, in
FP64 up to the rounding of a few sums over at most six levels (1e-13 of the
result's norm; 2e-16 per operation)."""
import numpy as np
import pytest

from p4pdes_amd import capi

pytestmark = pytest.mark.gpu

# the tail's top level: the smallest, odd boxes, the largest that fits in LDS (65^2, 17^3), one beyond
CASES = [
    ("-fsh_dim 2 -da_grid_x 3 -da_grid_y 3 -da_refine 2", 1),
    ("-fsh_dim 2 -da_grid_x 3 -da_grid_y 3 -da_refine 6", 1),
    ("-fsh_dim 2 -da_grid_x 3 -da_grid_y 3 -da_refine 7", 2),
    ("-fsh_dim 2 -da_grid_x 7 -da_grid_y 4 -da_refine 4 -fsh_cx 1.7", 3),
    ("-fsh_dim 2 -da_grid_x 4 -da_grid_y 19 -da_refine 3", 4),
    ("-fsh_dim 3 -da_grid_x 3 -da_grid_y 3 -da_grid_z 3 -da_refine 2", 1),
    ("-fsh_dim 3 -da_grid_x 3 -da_grid_y 3 -da_grid_z 3 -da_refine 4", 2),
    ("-fsh_dim 3 -da_grid_x 5 -da_grid_y 4 -da_grid_z 3 -da_refine 3 -fsh_cz 0.6", 1),
    ("-fsh_dim 3 -da_grid_x 3 -da_grid_y 5 -da_grid_z 6 -da_refine 3", 3),
]
SMOOTH = {"cheb": "-mg_levels_ksp_type chebyshev -mg_levels_pc_type jacobi",
          "rich": "-mg_levels_ksp_type richardson -mg_levels_ksp_richardson_scale 0.7 -mg_levels_pc_type jacobi"}


@pytest.mark.parametrize("smoother", sorted(SMOOTH))
@pytest.mark.parametrize("grid,nu", CASES)
def test_tail_matches_the_passes(grid, nu, smoother):
    args = "%s -fsh_problem zero -pc_type mg %s -mg_levels_ksp_max_it %d" % (grid, SMOOTH[smoother], nu)
    print("tail", args, flush=True)
    z = []
    for extra in (" -p4g_tail 0", ""):
        with capi.Session(args + extra) as s:
            b = np.random.default_rng(s.n).standard_normal(s.n)
            z.append(capi.Solver(s).pc_apply(b))
    assert np.isfinite(z[0]).all() and np.linalg.norm(z[0]) > 0
    assert np.linalg.norm(z[1] - z[0]) <= 1e-13 * np.linalg.norm(z[0])


def test_tail_mixed_precision_solve():
    # the FP32 cycle through the tail inside FP64 refinement: the same
    # iterations and a solution to the solve's own tolerance
    args = ("-fsh_dim 3 -fsh_problem manusin -da_refine 4 -pc_type mg %s -mg_levels_ksp_max_it 1 "
            "-p4g_precision mixed -ksp_rtol 1e-10" % SMOOTH["cheb"])
    rc0, t0, r0, u0 = capi.fish_run(args + " -p4g_tail 0", want_u=True)
    rc1, t1, r1, u1 = capi.fish_run(args, want_u=True)
    assert rc0 == 0 and rc1 == 0, (t0, t1)
    assert abs(r0.its - r1.its) <= 1 and r1.reason > 0
    assert np.linalg.norm(u1 - u0) <= 1e-9 * np.linalg.norm(u0)

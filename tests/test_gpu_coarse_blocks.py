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

"""The block factorization of a coarsest Newton operator (k_blk_factor,
k_blk_inverse) at band widths on either side of each rule: blocks of 16 rows
(narrow bands), 4 MR rows of 16, 36 and 63, one block, and a last block that
is not full.  The obstacle is symmetric in x and y, so a grid and its
transpose (another band width; from 64 on another path) have one solution;
each is converged to rtol 1e-12 and the coarse solve is direct, so both agree
to 1e-9 of the norm and take the same Newton steps."""
import numpy as np
import pytest

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

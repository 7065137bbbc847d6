"""The marching chunks of the 2D passes (one row a thread, two beyond 4.5
million points): the operator against numpy and a V(1,1)-preconditioned solve
against its own residual in numpy, on square, wide and tall grids on both
sides of the rule, with uneven last chunks."""
import numpy as np
import pytest

from p4pdes_amd import capi

pytestmark = pytest.mark.gpu


def _apply(u, c):
    """The library's rows of -c u_xx - u_yy on the unit square: boundary rows diagonal, their columns dropped."""
    my, mx = u.shape
    sx, sy = c * (mx - 1.0) / (my - 1.0), (my - 1.0) / (mx - 1.0)
    v = np.zeros_like(u)
    v[1:-1, 1:-1] = u[1:-1, 1:-1]
    out = 2.0 * (sx + sy) * u
    out[1:-1, 1:-1] -= sx * (v[1:-1, :-2] + v[1:-1, 2:]) + sy * (v[:-2, 1:-1] + v[2:, 1:-1])
    return out


# coarsest (gx, gy), refinements: 129x49, 4.46 and 4.33 million points, and 4.74, 4.94, 4.94 and 4.59 million
@pytest.mark.parametrize("gx,gy,r", [(9, 4, 4), (34, 34, 6), (133, 9, 6), (34, 36, 6), (300, 2, 7), (2, 300, 7),
                                     (9, 36, 7)])
def test_2d_chunks(gx, gy, r):
    mx, my = (gx - 1) * 2 ** r + 1, (gy - 1) * 2 ** r + 1
    c = ((my - 1.0) / (mx - 1.0)) ** 2           # couplings alike in x and y, so that point smoothing converges
    args = ("-fsh_dim 2 -fsh_problem zero -fsh_cx %r -da_grid_x %d -da_grid_y %d -da_refine %d -pc_type mg "
            "-mg_levels_ksp_type chebyshev -mg_levels_pc_type jacobi -mg_levels_ksp_max_it 1 "
            "-ksp_norm_type unpreconditioned -ksp_rtol 1e-6 -ksp_max_it 60" % (c, gx, gy, r))
    print("2d chunks", mx, my, flush=True)
    with capi.Session(args) as s:
        b = np.random.default_rng(s.n).standard_normal((my, mx))
        S = capi.Solver(s)
        Ab = S.mat_mult(b.ravel()).reshape(b.shape)
        x, rep = S.ksp_solve(b.ravel())
    ref = _apply(b, c)
    # a row is five products and four sums: nine roundings of partial sums up to twice the diagonal's term
    assert np.abs(Ab - ref).max() <= 20 * 2.0 ** -53 * np.abs(ref).max()
    assert rep.reason == 2
    # the recurrence's residual and the true one differ by its roundings only
    assert np.linalg.norm(_apply(x.reshape(b.shape), c) - b) <= 1.001e-6 * np.linalg.norm(b)

"""The cell-coefficient operator's marched cell layers and the V(1,1) cycle
that forms its zero-guess step on the fly, at sides where rows, chunks and
lanes end unevenly, against numpy: a two-level cycle is written out from the
formulas (a few sums of 7 products a point and level: 1e-13 of the norm)."""
import ctypes

import numpy as np
import pytest

from p4pdes_amd import capi

pytestmark = pytest.mark.gpu

OMEGA = 0.7


def _mat(k):
    """The operator as a dense matrix: rows scaled by the cell volume; boundary rows diagonal, their columns dropped."""
    nz, ny, nx = k.shape
    mz, my, mx = nz + 1, ny + 1, nx + 1
    vol = 1.0 / (nx * ny * nz)
    a = {0: vol * nz * nz, 1: vol * ny * ny, 2: vol * nx * nx}
    n = mx * my * mz
    idx = np.arange(n).reshape(mz, my, mx)
    A = np.zeros((n, n))
    top = (mz - 1, my - 1, mx - 1)
    for p in np.ndindex(mz, my, mx):
        q = idx[p]
        lo = [max(p[d] - 1, 0) for d in range(3)]
        hi = [min(p[d], top[d] - 1) for d in range(3)]
        if any(p[d] in (0, top[d]) for d in range(3)):
            c = k[lo[0]:hi[0] + 1, lo[1]:hi[1] + 1, lo[2]:hi[2] + 1]
            A[q, q] = 2.0 * sum(a.values()) * c.mean()
            continue
        for d in range(3):
            for s in (0, 1):
                sl = [slice(p[e] - 1, p[e] + 1) for e in range(3)]
                sl[d] = slice(p[d] - 1 + s, p[d] + s)
                w = a[d] * k[tuple(sl)].mean()
                A[q, q] += w
                r = list(p)
                r[d] += 2 * s - 1
                if 0 < r[d] < top[d]:
                    A[q, idx[tuple(r)]] = -w
    return A


def _prolong(m, M):
    P = np.zeros((m, M))
    for i in range(m):
        P[i, i // 2] += 0.5
        P[i, (i + 1) // 2] += 0.5
    return P


def _coarsen(k):
    return 0.125 * sum(k[a::2, b::2, c::2] for a in (0, 1) for b in (0, 1) for c in (0, 1))


class _Cells:
    def __init__(self, base, refine, k, nu=1):
        L = capi.lib()
        opts = ("-da_refine %d -pc_type mg -pc_mg_levels %d -mg_levels_ksp_type richardson "
                "-mg_levels_ksp_richardson_scale %g -mg_levels_pc_type jacobi -mg_levels_ksp_max_it %d"
                % (refine, refine + 1, OMEGA, nu)).encode()
        self.L, self.da, self.solver = L, ctypes.c_void_p(), ctypes.c_void_p()
        capi.check(L.p4g_da_create(3, *base, 1.0, 1.0, 1.0, ctypes.byref(self.da)))
        capi.check(L.p4g_da_set_from_options(self.da, opts))
        kk = np.ascontiguousarray(k)
        capi.check(L.p4g_da_set_cell_coefficient(self.da, kk.ctypes.data))
        capi.check(L.p4g_solver_create(self.da, opts, ctypes.byref(self.solver)))
        capi.check(L.p4g_solver_setup(self.solver))
        self.n = (k.shape[0] + 1) * (k.shape[1] + 1) * (k.shape[2] + 1)

    def close(self):
        self.L.p4g_solver_destroy(ctypes.byref(self.solver))
        self.L.p4g_da_destroy(ctypes.byref(self.da))


@pytest.mark.parametrize("base", [(3, 3, 3), (3, 5, 4), (6, 3, 5), (4, 7, 3), (7, 4, 6)])
@pytest.mark.parametrize("nu", [1, 2])     # the zero-guess step formed on the fly, or a pass for each step
def test_cells_cycle_matches_numpy(base, nu):
    mx, my, mz = (2 * (b - 1) + 1 for b in base)
    print("cells", mx, my, mz, nu, flush=True)
    rng = np.random.default_rng(mx * 100 + my * 10 + mz)
    k = np.exp(rng.standard_normal((mz - 1, my - 1, mx - 1)))
    c = _Cells(base, 1, k, nu)
    try:
        b = rng.standard_normal(c.n)
        S = capi.Solver(c)
        Au, z = S.mat_mult(b), S.pc_apply(b)
    finally:
        c.close()
    A, Ac = _mat(k), _mat(_coarsen(k))
    P = np.kron(_prolong(mz, base[2]), np.kron(_prolong(my, base[1]), _prolong(mx, base[0])))
    assert np.linalg.norm(Au - A @ b) <= 1e-13 * np.linalg.norm(Au)
    D = A.diagonal()
    x = np.zeros(b.size)
    for step in range(2 * nu):
        if step == nu:
            x = x + P @ np.linalg.solve(Ac, P.T @ (b - A @ x))
        x = x + OMEGA * (b - A @ x) / D
    assert np.linalg.norm(z - x) <= 1e-12 * np.linalg.norm(x)

"""Arrays that only make a solver faster (the SOR sweeps' own, the reciprocal
diagonal of a cell-coefficient level) give way where the device's memory is
short (-p4g_test_free_mb, an assumed amount): the solver then takes none of
them and computes the same."""
import ctypes

import numpy as np
import pytest
import torch

from p4pdes_amd import capi

pytestmark = pytest.mark.gpu


def _used(make):
    """(result, device bytes taken) of make(), which keeps its allocations until it returns them."""
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    keep = make()
    return keep, free0 - torch.cuda.mem_get_info()[0]


@pytest.mark.parametrize("args", ["-fsh_dim 3 -da_refine 6", "-fsh_dim 2 -da_refine 9"])
def test_sor_without_room_takes_the_hyperplanes(args):
    args += " -fsh_problem zero -pc_type mg"
    out = []
    for extra in ("", " -p4g_test_free_mb 0"):
        print("room", args + extra, flush=True)
        s, used = _used(lambda: capi.Session(args + extra))
        b = np.random.default_rng(s.n).standard_normal(s.n)
        out.append((used, capi.Solver(s).pc_apply(b)))
        n = s.n
        s.close()
    (full, z0), (short, z1) = out
    # the sweeps of the finest level alone hold a vector in their own order
    assert full - short >= 8 * n
    assert np.array_equal(z0, z1)


def test_cells_without_room_form_the_zero_guess_apart():
    L, m, r = capi.lib(), 129, 6
    k = np.exp(np.random.default_rng(3).standard_normal((m - 1,) * 3))
    b = np.random.default_rng(4).standard_normal(m ** 3)
    out = []
    for extra in ("", " -p4g_test_free_mb 0"):
        print("room cells", extra, flush=True)
        opts = ("-da_refine %d -pc_type mg -mg_levels_ksp_type chebyshev -mg_levels_pc_type jacobi "
                "-mg_levels_ksp_max_it 1%s" % (r, extra)).encode()
        da, solver = ctypes.c_void_p(), ctypes.c_void_p()
        capi.check(L.p4g_da_create(3, 3, 3, 3, 1.0, 1.0, 1.0, ctypes.byref(da)))
        capi.check(L.p4g_da_set_from_options(da, opts))
        capi.check(L.p4g_da_set_cell_coefficient(da, k.ctypes.data))
        capi.check(L.p4g_solver_create(da, opts, ctypes.byref(solver)))
        _, used = _used(lambda: capi.check(L.p4g_solver_setup(solver)))
        z = np.empty_like(b)
        capi.check(L.p4g_pc_apply(solver, b.ctypes.data, z.ctypes.data))
        out.append((used, z))
        L.p4g_solver_destroy(ctypes.byref(solver))
        L.p4g_da_destroy(ctypes.byref(da))
    (full, z0), (short, z1) = out
    assert full - short >= 8 * m ** 3
    # the step formed on the fly or stored first: the same products, their sums rounded alike
    assert np.linalg.norm(z0 - z1) <= 1e-13 * np.linalg.norm(z0)

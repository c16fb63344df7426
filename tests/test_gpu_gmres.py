"""GMRES kept on the device (fe_gmres.hip): one to three rows' chunk of the dot
products, cycle lengths around the 64-vector variant of the projection
kernels and at the ends of the accepted range, both orthogonalizations,
against dense solves; the iteration budget and the repeated solve."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _system(N):
    from feng_amd.api import FN_CONST, TRI_P1, Fn, Mesh
    from feng_amd.problems import advection_diffusion_system
    one = Fn(FN_CONST, 1.0)
    S, num = advection_diffusion_system(Mesh.square(N, 0.2, N), TRI_P1, 2, [Fn(FN_CONST, 30.0), Fn(FN_CONST, -20.0)], one,
                                        Fn(FN_CONST, -1.0))
    S.assemble(3)
    ia, ja = S.get_csr()
    val, rhs = S.get_system()
    D = np.zeros((num.nInc, num.nInc))
    D[np.repeat(np.arange(num.nInc), np.diff(ia)), ja] = val
    return S, D, rhs


@pytest.mark.parametrize("N", [2, 3, 24, 41])
@pytest.mark.parametrize("restart", [2, 63, 64, 65, 120])
def test_gmres_matches_dense_solve(N, restart):
    from feng_amd.api import KSP_GMRES, PC_JACOBI
    print("gmres", N, restart, flush=True)
    S, D, rhs = _system(N)
    x = np.linalg.solve(D, rhs)
    # ||x - x*|| <= ||D^-1|| ||r||, ||r|| <= rtol ||b|| (and the rounding of the dense solve)
    rtol = 1e-10
    bound = np.linalg.norm(np.linalg.inv(D), 2) * 1.01 * rtol * np.linalg.norm(rhs)
    for orth in (1, 2):
        S.set_tuning("gmres_orth", orth)
        r, du = S.solve(ksp=KSP_GMRES, pc=PC_JACOBI, rtol=rtol, restart=restart, max_iter=20000, want_du=True)
        assert r.converged and r.reason == 2 and r.relres <= rtol
        assert np.linalg.norm(du - x) <= bound
        assert np.linalg.norm(rhs - D @ du) <= 1.01 * rtol * np.linalg.norm(rhs) + 1e-14 * np.linalg.norm(D) * np.linalg.norm(x)
        assert abs(r.norm_dx_inf - np.abs(du).max()) <= 1e-15 * np.abs(du).max()
        assert r.norm_rhs_inf == np.abs(rhs).max()
        again, du2 = S.solve(ksp=KSP_GMRES, pc=PC_JACOBI, rtol=rtol, restart=restart, max_iter=20000, want_du=True)
        assert again.iterations == r.iterations and np.array_equal(du, du2)  # bitwise repeatable
    S.close()


def test_gmres_iteration_budget_and_zero_rhs():
    from feng_amd.api import KSP_GMRES, PC_JACOBI
    S, D, rhs = _system(24)
    for restart, most in ((50, 7), (4, 4), (4, 6), (50, 0)):
        r, du = S.solve(ksp=KSP_GMRES, pc=PC_JACOBI, rtol=1e-12, restart=restart, max_iter=most, want_du=True)
        assert not r.converged and r.reason == -3 and r.iterations == most
        assert abs(r.relres - np.linalg.norm(rhs - D @ du) / np.linalg.norm(rhs)) <= 1e-10
    S.set_system(rhs=np.zeros_like(rhs))
    r, du = S.solve(ksp=KSP_GMRES, pc=PC_JACOBI, rtol=1e-12, want_du=True)
    assert r.converged and r.iterations == 0 and not du.any()
    S.close()


@pytest.mark.parametrize("kind, N", [(1, 2), (1, 9), (2, 20), (5, 7), (6, 6), (3, 6), (1, 129), (1, 130)])
def test_exact_ilu0_application(kind, N):
    """One GMRES step from x = 0 returns a multiple of U^-1 L^-1 b: the exact
    application of the factor against host triangular solves, one unknown to
    the largest vector of the one-launch schedule (16,384) and past it."""
    import scipy.sparse as sp
    import scipy.sparse.linalg as sl
    from feng_amd.api import FN_CONST, KSP_GMRES, PC_ILU0, Fn, Mesh
    from feng_amd.problems import advection_diffusion_system, navier_stokes_system
    print("ilu0 application", kind, N, flush=True)
    m = Mesh.square(N, 0.2, N)
    if kind == 3:  # Taylor-Hood: rows of two fields
        S, num = navier_stokes_system(m, 40.0, 5)
    else:
        S, num = advection_diffusion_system(m, kind, 4, [Fn(FN_CONST, 5.0), Fn(FN_CONST, -3.0)], Fn(FN_CONST, 1.0),
                                            Fn(FN_CONST, -1.0))
    S.assemble(3)
    b = np.random.default_rng(N).normal(size=num.nInc)
    S.set_system(rhs=b)
    r, du = S.solve(ksp=KSP_GMRES, pc=PC_ILU0, rtol=1e-14, restart=2, max_iter=1, want_du=True)
    ia, ja = S.get_csr()
    lu = sp.csr_matrix((S.get_factor(), ja, ia), shape=(num.nInc, num.nInc))
    y = sl.spsolve_triangular((sp.tril(lu, -1) + sp.identity(num.nInc)).tocsr(), b, lower=True)
    z = sl.spsolve_triangular(sp.triu(lu).tocsr(), y, lower=False)
    t = du @ z / (z @ z)
    # rounding of the solves only: (longest row + levels) units in the last place, amplified by the growth in z
    assert np.linalg.norm(du - t * z) <= 1e-10 * np.linalg.norm(du)
    S.close()


def _free_bytes():
    """Free device memory, from the HIP runtime the library has loaded."""
    path = next(ln.split()[-1] for ln in open("/proc/self/maps") if "libamdhip64.so" in ln)
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL(path).hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_a_large_workspace_is_given_back():
    """360,000 rows at restart 120: 367 MB during the solve, freed after it; the
    results of repeated solves do not depend on it."""
    from feng_amd.api import KSP_GMRES, PC_JACOBI, FN_CONST, Fn, Mesh
    from feng_amd.problems import diffusion_system
    S, _ = diffusion_system(Mesh.square(600), 1, 4, Fn(FN_CONST, 1.0), Fn(FN_CONST, -1.0))
    S.assemble(3)
    opts = dict(ksp=KSP_GMRES, pc=PC_JACOBI, restart=120, rtol=1e-12, max_iter=20, want_du=True)
    S.solve(**{**opts, "restart": 2, "max_iter": 2})
    free = _free_bytes()
    r0, x0 = S.solve(**opts)
    assert free - _free_bytes() <= 64 << 20
    r1, x1 = S.solve(**opts)
    assert r0.iterations == r1.iterations == 20 and np.array_equal(x0, x1)
    S.close()


def test_what_a_solve_without_iterations_reports():
    from feng_amd.api import KSP_GMRES, PC_JACOBI
    S, _, rhs = _system(12)
    bad = rhs.copy()
    bad[3] = np.nan
    # a zero right-hand side starts no cycle; no budget left is -3 whatever the residual, not a number -4
    for b, max_iter, want in ((0.0 * rhs, 50, (0, 0, True, 2)), (rhs, 0, (0, 0, False, -3)), (bad, 50, (0, 1, False, -4)),
                              (bad, 0, (0, 0, False, -3))):
        S.set_system(rhs=b)
        r = S.solve(ksp=KSP_GMRES, pc=PC_JACOBI, max_iter=max_iter)
        assert (r.iterations, r.outer_iterations, r.converged, r.reason) == want
    S.close()

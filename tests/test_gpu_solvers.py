"""GPU preconditioners and Krylov methods: device ILU(0)/IC(0) factor vs the
oracle, split IC(0)-pattern PCG, GMRES(m) + ILU(0) on Taylor-Hood systems,
Newton on the Kovasznay flow."""
import math

import numpy as np
import pytest

from tests.cases import relerr

pytestmark = pytest.mark.gpu


def _fn(k, c0=0.0, data=None):
    from feng_amd.api import Fn
    return Fn(k, c0, 0.0, data)


@pytest.mark.parametrize("case", ["p1_square", "ns_th"])
def test_device_ilu0_matches_oracle(oracle, case):
    from feng_amd.api import KSP_CG, KSP_GMRES, PC_IC0, PC_ILU0, Mesh
    from feng_amd.problems import diffusion_system, navier_stokes_system
    print("case", case, flush=True)
    if case == "p1_square":
        m = Mesh.square(40, 0.2, 1)
        S, num = diffusion_system(m, 1, 2, _fn(2, 4.0), _fn(0, -1.0))
        S.assemble(3)
        S.solve(ksp=KSP_CG, pc=PC_IC0, rtol=1e-8)
    else:
        m = Mesh.square(12, 0.2, 1)
        S, num = navier_stokes_system(m, 40.0, 5)
        S.assemble(3)
        S.solve(ksp=KSP_GMRES, pc=PC_ILU0, rtol=1e-8, restart=50)
    ia, ja = S.get_csr()
    val, rhs = S.get_system()
    lu = S.get_factor()
    lu0, rc = oracle.ilu0(ia, ja, val)
    assert rc == 0
    assert relerr(lu, lu0) <= 1e-12
    levels, shifts = S.pc_info()
    assert levels > 1 and shifts == 0
    S.close()


def test_split_ic0_pcg_beats_jacobi(oracle):
    from feng_amd.api import FN_ELEM, PC_IC0, PC_JACOBI, PREC_FP32_IR, Mesh
    from feng_amd.problems import diffusion_system
    m = Mesh.cube(16)
    k = m.coeff_grf(0.1, 1.5, 256, 2)
    S, num = diffusion_system(m, 4, 1, _fn(FN_ELEM, data=k), _fn(0, -1.0))
    S.assemble(3, PREC_FP32_IR)
    rj = S.solve(pc=PC_JACOBI, rtol=1e-8)
    ri, du = S.solve(pc=PC_IC0, rtol=1e-8, want_du=True)
    ri32 = S.solve(pc=PC_IC0, precision=PREC_FP32_IR, rtol=1e-8, inner_rtol=1e-2)
    assert rj.converged and ri.converged and ri32.converged
    assert ri.iterations < 0.7 * rj.iterations
    # by launches: FP32 inner solves, tiled (pipe_kernel 1) and not, and the FP64 forms
    S.set_tuning("resident", 0)
    for pipe in (2, 1, 0):
        S.set_tuning("pipe_kernel", pipe)
        r64 = S.solve(pc=PC_IC0, rtol=1e-8)
        r32 = S.solve(pc=PC_IC0, precision=PREC_FP32_IR, rtol=1e-8, inner_rtol=1e-2)
        assert r64.converged and r32.converged and r32.outer_iterations >= 2 and r64.iterations < 0.7 * rj.iterations
    ia, ja = S.get_csr()
    val, rhs = S.get_system()
    res = rhs - oracle.spmv(ia, ja, val, du)
    assert np.linalg.norm(res) <= 1.01e-8 * np.linalg.norm(rhs)
    S.close()


def test_gmres_ilu0_kovasznay_newton(oracle):
    """Newton + GMRES(50)/ILU(0) on the Kovasznay flow (Re = 40): converges
    quadratically and the discrete solution approaches the exact field."""
    from feng_amd.api import KSP_GMRES, PC_ILU0, Mesh
    from feng_amd.problems import NLSolverOptions, kovasznay, navier_stokes_system, solve_newton
    m = Mesh.square(24, 0.2, 0)
    S, num = navier_stokes_system(m, 40.0, 5)
    rep = solve_newton(S, NLSolverOptions(tolResidual=1e-9, tolCorrection=1e-12, maxIter=12),
                       ksp=KSP_GMRES, pc=PC_ILU0, rtol=1e-10, restart=50, max_iter=20000)
    assert rep.converged and rep.iterations <= 8
    u = S.get_solution()
    lam, ufn, pfn = kovasznay(40.0)
    xyz = num.dof_xyz.reshape(-1, 3)
    uf = num.dof_field == 0
    ue = ufn(xyz[uf, 0], xyz[uf, 1], xyz[uf, 2], num.dof_comp[uf])
    assert np.abs(u[uf] - ue).max() < 5e-3
    S.close()


def test_fieldsplit_gmres_matches_oracle_gmres_ilu0(oracle):
    """GMRES(50) with the block Schur preconditioner (FE_PC_FIELDSPLIT) on one
    Newton system of the jittered 24^2 Kovasznay problem: the solution of the
    same (values, RHS) as the oracle's GMRES(50) + ILU(0) (or_gmres_ilu0, the
    reference's PETSc combination restated), both to tight tolerances; with
    classical Gram-Schmidt (the default, PETSc's) and with CGS2."""
    from feng_amd.api import KSP_GMRES, PC_FIELDSPLIT, Mesh
    from feng_amd.problems import navier_stokes_system
    print("fieldsplit vs oracle gmres-ilu0", flush=True)
    m = Mesh.square(24, 0.2, 0)
    S, num = navier_stokes_system(m, 40.0, 5)
    S.setToZero()
    S.assemble(3)
    ia, ja = S.get_csr()
    val, rhs = S.get_system()
    r, du = S.solve(ksp=KSP_GMRES, pc=PC_FIELDSPLIT, rtol=1e-11, restart=50, max_iter=5000, want_du=True)
    assert r.converged and r.relres <= 1e-11
    lu, rc = oracle.ilu0(ia, ja, val)
    assert rc == 0
    x0, it0, rr0 = oracle.gmres_ilu0(ia, ja, val, lu, rhs, 50, 1e-12, 20000)
    assert rr0 <= 1e-12
    err = np.abs(du - x0).max() / np.abs(x0).max()
    print(f"fieldsplit GMRES {r.iterations} its, oracle GMRES-ILU(0) {it0} its, max rel diff {err:.2e}", flush=True)
    assert err <= 1e-7
    res = rhs - oracle.spmv(ia, ja, val, du)
    assert np.linalg.norm(res) <= 1.01e-11 * np.linalg.norm(rhs)
    # the Arnoldi steps with one reorthogonalization (CGS2, gmres_orth 2)
    # instead of classical Gram-Schmidt: the same solution
    S.set_tuning("gmres_orth", 2)
    r2, du2 = S.solve(ksp=KSP_GMRES, pc=PC_FIELDSPLIT, rtol=1e-11, restart=50, max_iter=5000, want_du=True)
    S.set_tuning("gmres_orth", 1)
    assert r2.converged and r2.relres <= 1e-11
    assert abs(r2.iterations - r.iterations) <= max(2, r.iterations // 20), (r.iterations, r2.iterations)
    assert np.abs(du2 - x0).max() / np.abs(x0).max() <= 1e-7
    S.close()


def test_fieldsplit_gmres_newton_converges_at_128():
    """Kovasznay flow (Re = 40) on the jittered 128^2 Taylor-Hood mesh,
    n = 146,179: every Newton step's GMRES(50) reaches rel-res 1e-8 within
    3000 iterations with the block Schur preconditioner.  At this size
    ILU(0) applied by two Jacobi sweeps per factor does not (its first Newton
    step stops at 7.8e-7 after 3000 iterations), and exact ILU(0) needs
    about 2000 iterations per step."""
    from feng_amd.api import KSP_GMRES, PC_FIELDSPLIT, Mesh
    from feng_amd.problems import NLSolverOptions, kovasznay, navier_stokes_system, solve_newton
    print("fieldsplit newton 128", flush=True)
    m = Mesh.square(128, 0.2, 0)
    S, num = navier_stokes_system(m, 40.0, 5)
    steps = []
    rep = solve_newton(S, NLSolverOptions(tolResidual=1e-9, tolCorrection=1e-12, maxIter=8),
                       progress=lambda it, r: steps.append(r), ksp=KSP_GMRES, pc=PC_FIELDSPLIT, rtol=1e-8,
                       restart=50, max_iter=3000)
    print("GMRES iterations per Newton step:", [r.iterations for r in steps], flush=True)
    assert rep.converged and rep.iterations <= 6
    assert all(r.converged and r.relres <= 1e-8 and r.iterations < 3000 for r in steps)
    u = S.get_solution()
    _, ufn, _ = kovasznay(40.0)
    xyz = num.dof_xyz.reshape(-1, 3)
    uf = num.dof_field == 0
    ue = ufn(xyz[uf, 0], xyz[uf, 1], xyz[uf, 2], num.dof_comp[uf])
    err = np.abs(u[uf] - ue).max()
    print(f"max velocity error vs the exact flow: {err:.2e}", flush=True)
    assert err < 1e-4
    S.close()


def test_parallel_ic0_converges_to_the_exact_factor(oracle):
    """Parallel IC(0) sweeps (Chow & Patel): the fixed point is the exact
    IC(0) factor (oracle ILU(0) of the symmetric matrix), and three sweeps
    already precondition as well as the exact factor."""
    from feng_amd.api import FN_ELEM, PC_IC0, Mesh
    from feng_amd.problems import diffusion_system
    m = Mesh.cube(10)
    k = m.coeff_grf(0.1, 1.5, 64, 3)
    S, num = diffusion_system(m, 4, 1, _fn(FN_ELEM, data=k), _fn(0, -1.0))
    S.assemble(3)
    ia, ja = S.get_csr()
    val, _ = S.get_system()
    lu_o, rc = oracle.ilu0(ia, ja, val)
    r_exact = S.solve(pc=PC_IC0, rtol=1e-8)
    S.set_tuning("ic0_sweeps", 40)
    S.solve(pc=PC_IC0, rtol=1e-8)
    assert relerr(S.get_factor(), lu_o) < 1e-10
    S.set_tuning("ic0_sweeps", 3)
    r3 = S.solve(pc=PC_IC0, rtol=1e-8)
    assert r3.converged and abs(r3.iterations - r_exact.iterations) <= 3
    S.close()

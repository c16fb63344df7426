"""GPU parity of the diffusion path (libfe_hip.so through the C ABI) against
the reference fixtures and the CPU oracle."""
import math

import numpy as np
import pytest

from tests.cases import DIFF_CASES, coeffs_of, kind_of, load, product_mesh, relerr

pytestmark = pytest.mark.gpu


def _fn(t):
    from feng_amd.api import Fn
    return Fn(t[0], t[1], t[2], t[3])


@pytest.mark.parametrize("asm_kernel", [0, 1])
@pytest.mark.parametrize("name", DIFF_CASES)
def test_device_csr_and_assembly_match_reference(name, asm_kernel):
    """Both element paths (0: scalar loop in the reference's order, 1: MFMA
    GEMM form) against the reference's CSR, matrix and RHS."""
    from feng_amd.problems import diffusion_system
    print("case", name, asm_kernel, flush=True)
    g = load(name)
    m = product_mesh(g)
    k, s = coeffs_of(g)
    S, num = diffusion_system(m, kind_of(g), g["deg"], _fn(k), _fn(s))
    S.set_tuning("asm_kernel", asm_kernel)
    ia, ja = S.get_csr()
    assert np.array_equal(ia, g["ia"]) and np.array_equal(ja, g["ja"])
    S.assemble(3)
    val, rhs = S.get_system()
    assert relerr(val, g["val"]) <= 1e-12
    assert relerr(rhs, g["rhs"]) <= 1e-12
    S.close()


def _oracle_system(oracle, m, num, kind, deg, k, s):
    ia, ja = oracle.csr(num.nInc, [(num.adr[0], num.adr[0].size // m.E, num.adr[0], num.adr[0].size // m.E)])
    val, rhs = oracle.assemble_diffusion(kind, m.xyz, m.conn, num.adr[0], num.nInc, ia, ja, deg, k, s,
                                         np.zeros(num.nDofs))
    return ia, ja, val, rhs


@pytest.mark.parametrize("cfg", ["c1_p1_64", "p2_blocks_48", "tet_grf_12"])
def test_end_to_end_vs_oracle(oracle, cfg):
    """Device CSR bit-exact vs the oracle, values <= 1e-12, CG reaches the
    FP64 true-residual target (checked on the host with the oracle SpMV)."""
    from feng_amd.api import FN_ELEM, Fn, Mesh
    from feng_amd.problems import diffusion_system
    print("case", cfg, flush=True)
    if cfg == "c1_p1_64":
        m, kind, deg = Mesh.square(64), 1, 2
        k, s = (0, 1.0, 0.0, None), (1, -2 * math.pi ** 2, 0.0, None)
        rtol = 1e-10
    elif cfg == "p2_blocks_48":
        m, kind, deg = Mesh.square(48), 2, 2
        kk = m.coeff_blocks(16, 1e-2, 1e2, 9)
        k, s = (4, 0.0, 0.0, kk), (0, -1.0, 0.0, None)
        rtol = 1e-10
    else:
        m, kind, deg = Mesh.cube(12), 4, 1
        kk = m.coeff_grf(0.1, 1.5, 256, 4)
        k, s = (4, 0.0, 0.0, kk), (0, -1.0, 0.0, None)
        rtol = 1e-8
    S, num = diffusion_system(m, kind, deg, _fn(k), _fn(s))
    ia0, ja0, val0, rhs0 = _oracle_system(oracle, m, num, kind, deg, k, s)
    ia, ja = S.get_csr()
    assert np.array_equal(ia, ia0) and np.array_equal(ja, ja0)
    S.assemble(3)
    val, rhs = S.get_system()
    assert relerr(val, val0) <= 1e-12 and relerr(rhs, rhs0) <= 1e-12
    r, du = S.solve(rtol=rtol, want_du=True)
    assert r.converged and r.relres <= rtol
    res = rhs0 - oracle.spmv(ia0, ja0, val0, du)
    assert np.linalg.norm(res) <= 1.01 * rtol * np.linalg.norm(rhs0)
    x0, it0, rr0 = oracle.cg_jacobi(ia0, ja0, val0, rhs0, rtol * 0.1, 20000)
    assert np.abs(du - x0).max() <= 1e-5 * np.abs(x0).max()
    S.close()


def test_fp32_refinement_reaches_fp64_tolerance(oracle):
    from feng_amd.api import PREC_FP32_IR, Mesh
    from feng_amd.problems import diffusion_system
    m = Mesh.square(64, 0.2, 0)
    S, num = diffusion_system(m, 2, 2, _fn((0, 1.0, 0.0, None)), _fn((1, -2 * math.pi ** 2, 0.0, None)))
    S.assemble(3, PREC_FP32_IR)
    r = S.solve(precision=PREC_FP32_IR, rtol=1e-10)
    assert r.converged and r.relres <= 1e-10 and S.get_tuning("resident_ran") == 1  # FP64, in one launch
    S.set_tuning("resident", 0)
    for pipe in (2, 1, 0):  # FP32 inner solves: Chronopoulos-Gear, tiled, Chronopoulos-Gear
        S.set_tuning("pipe_kernel", pipe)
        r = S.solve(precision=PREC_FP32_IR, rtol=1e-10)
        assert r.converged and r.relres <= 1e-10 and r.outer_iterations >= 2
    # FP32 values that are no longer the matrix's: the first correction is rejected, FP64 inner solves finish
    val, rhs = S.get_system()
    S.set_system(val=3.0 * val, rhs=rhs)
    for pipe in (2, 1, 0):
        S.set_tuning("pipe_kernel", pipe)
        r, x = S.solve(precision=PREC_FP32_IR, rtol=1e-10, want_du=True)
        assert r.converged and r.relres <= 1e-10 and r.outer_iterations >= 2
        ia, ja = S.get_csr()
        res = rhs - oracle.spmv(ia, ja, 3.0 * val, x)
        assert np.linalg.norm(res) <= 1.01e-10 * np.linalg.norm(rhs)
    S.set_system(val=val, rhs=rhs)
    r64 = S.solve(rtol=1e-10)
    assert r64.converged
    S.close()


def test_assembly_is_deterministic():
    from feng_amd.api import Mesh
    from feng_amd.problems import diffusion_system
    m = Mesh.square(40, 0.2, 2)
    S, num = diffusion_system(m, 2, 5, _fn((2, 4.0, 0.0, None)), _fn((0, -1.0, 0.0, None)))
    S.assemble(3)
    v1, r1 = S.get_system()
    S.setToZero()
    S.assemble(3)
    v2, r2 = S.get_system()
    assert np.array_equal(v1, v2) and np.array_equal(r1, r2)
    S.close()


# scalarFE_diffusion.output (tests/withLinearSolver/ of the reference): L2
# error of P1 and P2 Lagrange diffusion on mmsMeshes/square1-4, degree-8
# quadrature, u = sin(pi x) sin(pi y), printed with 6 significant digits.
REF_TABLE = {
    1: ["7.907546e-02", "2.113277e-02", "5.377435e-03", "1.350436e-03"],
    2: ["4.327628e-03", "5.480619e-04", "6.873916e-05", "8.600535e-06"],
}


@pytest.mark.parametrize("order", [1, 2])
def test_reference_convergence_table(oracle, order):
    from feng_amd.api import Mesh
    from feng_amd.problems import NLSolverOptions, diffusion_system, solve_newton
    from tests.conftest import GOLDEN
    out = []
    for lvl in range(1, 5):
        m = Mesh.read_msh(GOLDEN / "meshes" / f"square{lvl}.msh")
        bc = lambda x, y, z, c: np.sin(np.pi * x) * np.sin(np.pi * y)
        S, num = diffusion_system(m, order, 8, _fn((0, 1.0, 0.0, None)), _fn((1, -2 * math.pi ** 2, 0.0, None)),
                                  u_bc=bc)
        rep = solve_newton(S, NLSolverOptions(), rtol=1e-13)
        assert rep.converged
        u = S.get_solution()
        err = oracle.l2_error_sinsin(order, m.xyz, m.conn, num.adr[0], u, 8)
        out.append(f"{err:.6e}")
        S.close()
    assert out == REF_TABLE[order]


@pytest.mark.parametrize("kind,deg", [(1, 2), (2, 2), (2, 5), (4, 1), (4, 2)])
def test_fp32_mfma_element_matrices(kind, deg):
    """FP32 element matrices on the matrix cores vs the FP64 assembly:
    single-precision accuracy, same pattern."""
    from feng_amd.api import FN_ELEM, PREC_FP32_IR, Mesh
    from feng_amd.problems import diffusion_system
    m = Mesh.cube(6) if kind == 4 else Mesh.square(24, 0.2, 4)
    k = np.exp(np.random.default_rng(kind).standard_normal(m.E))
    S, num = diffusion_system(m, kind, deg, _fn((FN_ELEM, 0.0, 0.0, k)), _fn((0, -1.0, 0.0, None)))
    S.set_tuning("fp32_values", 1)
    S.assemble(3, PREC_FP32_IR)
    v64, r64 = S.get_system()
    r = S.solve(precision=PREC_FP32_IR, rtol=1e-10)
    assert r.converged and r.relres <= 1e-10
    S.set_tuning("resident", 0)  # FP32 inner solves from here on
    r = S.solve(precision=PREC_FP32_IR, rtol=1e-10)
    assert r.converged and r.relres <= 1e-10 and r.outer_iterations >= 2
    # the FP32 values themselves: solve with them must reach the FP64 target
    S.set_tuning("fp32_values", 0)
    S.setToZero()
    S.assemble(3, PREC_FP32_IR)
    r0 = S.solve(precision=PREC_FP32_IR, rtol=1e-10)
    assert r0.converged and r0.outer_iterations >= 2
    S.close()


# convergenceLaplace.output (tests/withLinearSolver/ of the reference): L2
# error of u = x^6 + y^6, k = 1, on data/square1-4.msh with the degree-12
# triangle rule (33 points), P1 and P2 rows.
LAPLACE_TABLE = {
    1: [5.939644e-02, 1.536748e-02, 3.879072e-03, 9.723478e-04],
    2: [3.209814e-03, 4.066278e-04, 5.111231e-05, 6.408018e-06],
    3: [1.524938e-04, 9.733075e-06, 6.093175e-07, 3.800562e-08],
    4: [4.353604e-06, 1.366429e-07, 4.289450e-09, 1.344400e-10],
}


@pytest.mark.parametrize("order", [1, 2, 3, 4])
def test_reference_convergence_laplace_table(order):
    """convergenceLaplace.output, P1 to P4 (P3 / P4: cubic and quartic
    triangles, AMG-PCG; errors below 1e-9 to 5e-15 absolute, the rounding of
    the solve in their 7th digit)."""
    from feng_amd.api import FN_CONST, FN_QP, KSP_CG, NORM_L2_ERROR, PC_AMG, Mesh
    from feng_amd.problems import NLSolverOptions, diffusion_system, solve_newton
    from tests.conftest import GOLDEN
    from tests.test_oracle_time import _qp_table
    print("laplace", order, flush=True)
    err = []
    for lvl in range(1, 5):
        m = Mesh.read_msh(GOLDEN / "meshes" / "data" / f"square{lvl}.msh")
        src = _qp_table(m, 12, lambda x, y: 30.0 * (x ** 4 + y ** 4))
        kind = {1: 1, 2: 2, 3: 5, 4: 6}[order]
        S, num = diffusion_system(m, kind, 12, _fn((FN_CONST, 1.0, 0.0, None)), _fn((FN_QP, 0.0, 0.0, src)),
                                  u_bc=lambda x, y, z, c: x ** 6 + y ** 6)
        if order <= 2:
            rep = solve_newton(S, NLSolverOptions(), rtol=1e-13)
        else:
            rep = solve_newton(S, NLSolverOptions(1e-12, 1e-12, 1e4, 20), ksp=KSP_CG, pc=PC_AMG, rtol=1e-13,
                               max_iter=5000)
        assert rep.converged
        err.append(S.norm(NORM_L2_ERROR, 0, 12, [_fn((FN_QP, 0.0, 0.0, _qp_table(m, 12, lambda x, y: x ** 6 + y ** 6)))]))
        S.close()
    assert all(abs(e - r) <= max(1e-6 * r, 5e-15) for e, r in zip(err, LAPLACE_TABLE[order])), err


@pytest.mark.parametrize("dim", [2, 3])
def test_upload_refuses_negative_jacobian(dim):
    """fe_hip_upload_mesh returns FE_STATUS_ERROR on a reversed element, as
    feCncGeo::computeJacobians does (feCncGeo.cpp:346-353, :388-395, :410-412);
    nothing is uploaded or launched."""
    from feng_amd.api import FeError, LinearSystemHIP, Mesh
    print("negative jacobian upload", dim, flush=True)
    good = Mesh.square(4) if dim == 2 else Mesh.cube(2)
    conn = good.conn.reshape(good.E, good.nvpe).copy()
    conn[3, [1, 2]] = conn[3, [2, 1]]
    m = Mesh.from_arrays(dim, good.xyz.reshape(-1, 3), conn)
    S = LinearSystemHIP(0)
    with pytest.raises(FeError, match="Negative or zero jacobian"):
        S.upload_mesh(m)
    S.close()

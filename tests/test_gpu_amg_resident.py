"""Multigrid-PCG with all iterations in one launch (fe_amg_resident.hip)
against the launch-per-level kernels on the same systems: hierarchies with one
to three distributed levels, one workgroup and many, the three row lengths,
rows too long for it, budgets, a zero right-hand side, the heat stack."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _system(kind, N, contrast=1.0):
    from feng_amd.api import FN_CONST, FN_ELEM, TET_P1, Fn, Mesh
    from feng_amd.problems import diffusion_system
    m = Mesh.cube(N) if kind == TET_P1 else Mesh.square(N, 0.2, N)
    k = np.exp(np.random.default_rng(N).normal(0.0, contrast, m.E))
    deg = 1 if kind == TET_P1 else 4
    S, num = diffusion_system(m, kind, deg, Fn(FN_ELEM, data=k), Fn(FN_CONST, -1.0))
    S.assemble(3)
    return S, num


# kind 1 (P1 triangles, 8 entries a row), 4 (P1 tets, 16), 2 (P2, 24), 5 (P3: rows too long)
@pytest.mark.parametrize("kind, N", [(1, 10), (1, 24), (1, 33), (1, 100), (1, 300), (1, 500), (1, 512), (1, 520), (4, 6), (4, 10),
                                     (4, 21), (4, 37), (4, 50), (4, 64), (2, 8), (2, 60), (2, 150), (5, 10)])
def test_resident_amg_equals_launch_per_level(kind, N):
    from feng_amd.api import PC_AMG
    print("resident amg", kind, N, flush=True)
    S, num = _system(kind, N)
    out = {}
    for resident in (0, 1):
        S.set_tuning("resident", resident)
        out[resident] = S.solve(pc=PC_AMG, rtol=1e-9, max_iter=5000, want_du=True)
        # workgroups are cut at whole aggregates: two rows a thread of the device are not quite reached
        fits = S.n <= 262144 and kind != 5 and (kind, N) != (1, 512)
        assert S.get_tuning("resident_ran") == (resident and fits) and S.get_tuning("resident_gave_up") == 0
    (r0, x0), (r1, x1) = out[0], out[1]
    assert r0.converged and r1.converged and r1.relres <= 1e-9
    # the same method, sums in another order and the smoother's level-0 values in FP64 instead of their FP32
    # rounding (2^-24 relative in the preconditioner): the stop moves by an iteration or two
    assert abs(r1.iterations - r0.iterations) <= 2 + r0.iterations // 20
    assert np.linalg.norm(x1 - x0) <= 1e-7 * np.linalg.norm(x0)
    ia, ja = S.get_csr()
    val, rhs = S.get_system()
    res = rhs - np.add.reduceat(val * x1[ja], ia[:-1])
    assert np.linalg.norm(res) <= 1.02e-9 * np.linalg.norm(rhs)
    # an entry of b - A x summed in two orders: at most (row length + 1) eps sum |a_ij x_j| apart
    terms = np.add.reduceat(np.abs(val * x1[ja]), ia[:-1]) + np.abs(rhs)
    assert abs(r1.norm_axb_inf - np.abs(res).max()) <= 25 * 2.3e-16 * terms.max()
    assert r1.norm_rhs_inf == np.abs(rhs).max() and r1.norm_dx_inf == np.abs(x1).max()
    again, x2 = S.solve(pc=PC_AMG, rtol=1e-9, max_iter=5000, want_du=True)
    assert again.iterations == r1.iterations and np.array_equal(x1, x2)  # bitwise repeatable
    if r1.iterations > 5:
        rb, xb = S.solve(pc=PC_AMG, rtol=1e-9, max_iter=4, want_du=True)
        assert not rb.converged and rb.reason == -3 and rb.iterations == 4
        rr = np.linalg.norm(rhs - np.add.reduceat(val * xb[ja], ia[:-1])) / np.linalg.norm(rhs)
        assert abs(rb.relres - rr) <= 1e-9 * rr
    # new values on the same pattern, then a zero right-hand side
    S.set_system(val=2.0 * val, rhs=rhs)
    rn, xn = S.solve(pc=PC_AMG, rtol=1e-9, want_du=True)
    assert rn.converged and np.linalg.norm(2.0 * xn - x1) <= 1e-7 * np.linalg.norm(x1)
    S.set_system(rhs=np.zeros_like(rhs))
    rz, xz = S.solve(pc=PC_AMG, want_du=True)
    assert rz.converged and rz.iterations == 0 and not xz.any()
    S.close()


def test_resident_amg_high_contrast_and_floor():
    """A 1e4-contrast coefficient, and a target at the FP64 floor, where the
    solve restarts from the true residual inside the launch."""
    from feng_amd.api import PC_AMG
    S, _ = _system(2, 40, 2.0)
    for rtol in (1e-8, 1e-11, 1e-15):
        S.set_tuning("resident", 0)
        r0, x0 = S.solve(pc=PC_AMG, rtol=rtol, max_iter=3000, want_du=True)
        S.set_tuning("resident", 1)
        r1, x1 = S.solve(pc=PC_AMG, rtol=rtol, max_iter=3000, want_du=True)
        print(rtol, r0, r1, flush=True)
        if r0.converged:
            assert r1.converged and r1.relres <= rtol
        assert np.linalg.norm(x1 - x0) <= 1e-6 * np.linalg.norm(x0)
    S.close()


@pytest.mark.parametrize("kernel,resident", [(2, 1), (2, 0), (1, 1)])
def test_fp32_multigrid_runs_the_fp64_iteration(kernel, resident):
    """Up to 700,000 rows FP32_IR multigrid-PCG is the FP64 iteration: the same
    iterates bit for bit, from an FP32 assembly as from an FP64 one."""
    from feng_amd.api import PC_AMG, PREC_FP32_IR, PREC_FP64
    S, num = _system(4, 9)
    S.set_tuning("amg_kernel", kernel)
    S.set_tuning("resident", resident)
    out = {}
    for prec in (PREC_FP64, PREC_FP32_IR):
        S.setToZero()
        S.assemble(3, prec)
        out[prec] = S.solve(pc=PC_AMG, precision=prec, rtol=1e-8, inner_rtol=1e-3, want_du=True)
    (r0, d0), (r1, d1) = out[PREC_FP64], out[PREC_FP32_IR]
    assert r0.converged and r1.iterations == r0.iterations and r1.outer_iterations == r0.outer_iterations
    assert np.array_equal(d0, d1)
    S.close()


@pytest.mark.parametrize("resident", [0, 1])
def test_set_up_time_is_reported(resident):
    """ms_setup: the hierarchy of the first solve (some milliseconds of host
    work); next to nothing on later ones."""
    from feng_amd.api import PC_AMG
    S, _ = _system(4, 24)
    S.set_tuning("resident", resident)
    first, second = S.solve(pc=PC_AMG), S.solve(pc=PC_AMG)
    assert S.get_tuning("resident_ran") == resident
    assert first.ms_setup > 0.3 and first.ms_setup > 5 * second.ms_setup and first.ms_setup < first.ms_solve
    S.close()


def test_a_zero_right_hand_side_builds_no_hierarchy():
    from feng_amd.api import PC_AMG
    S, _ = _system(4, 24)
    _, rhs = S.get_system()
    S.set_system(rhs=np.zeros_like(rhs))
    r, x = S.solve(pc=PC_AMG, want_du=True)
    assert r.converged and r.iterations == r.outer_iterations == 0 and r.relres == 0.0 and not x.any()
    assert r.ms_setup < 0.1 and S.get_tuning("resident_ran") == 0
    S.set_system(rhs=rhs)
    r = S.solve(pc=PC_AMG)
    assert r.converged and r.ms_setup > 0.3 and S.get_tuning("resident_ran") == 1
    S.close()

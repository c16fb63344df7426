"""Jacobi-PCG with all iterations in one launch (fe_resident.hip) against the
launch-per-iteration kernels on the same systems: one unknown, one workgroup
and the first of the next, rows a workgroup that no longer divide it, the
three row lengths, rows too long for it, the iteration budget, two threads."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _system(kind, N, seed=0):
    from feng_amd.api import FN_CONST, FN_ELEM, TET_P1, Fn, Mesh
    from feng_amd.problems import diffusion_system
    m = Mesh.cube(N) if kind == TET_P1 else Mesh.square(N, 0.2, N)
    k = np.exp(np.random.default_rng(seed + N).normal(0.0, 1.0, m.E))
    deg = 1 if kind == TET_P1 else 4
    S, num = diffusion_system(m, kind, deg, Fn(FN_ELEM, data=k), Fn(FN_CONST, -1.0))
    S.assemble(3)
    return S, num


# kind 1 (P1 triangles, 8 entries a row), 4 (P1 tets, 16), 2 (P2, 24), 5 (P3: rows too long)
@pytest.mark.parametrize("kind, N", [(1, 2), (1, 3), (1, 17), (1, 18), (1, 63), (1, 300), (1, 512), (1, 514), (4, 2),
                                     (4, 7), (4, 21), (4, 40), (2, 4), (2, 40), (2, 150), (5, 6)])
def test_resident_equals_launch_per_iteration(kind, N):
    print("resident", kind, N, flush=True)
    S, num = _system(kind, N)
    out = {}
    for resident in (0, 1):
        S.set_tuning("resident", resident)
        out[resident] = S.solve(rtol=1e-9, max_iter=20000, want_du=True)
        # more than one row a thread of the device, or rows of more than 24 entries, do not fit
        fits = S.n <= 262144 and kind != 5
        assert S.get_tuning("resident_ran") == (resident and fits) and S.get_tuning("resident_gave_up") == 0
    (r0, x0), (r1, x1) = out[0], out[1]
    assert r0.converged and r1.converged and r1.relres <= 1e-9
    # the same recurrences with sums in another order: the stop moves by a few
    # iterations; where the drift of the recurrences forces a restart from the
    # true residual, when it happens moves too and the counts are not compared
    if r0.outer_iterations == r1.outer_iterations == 1:
        assert abs(r1.iterations - r0.iterations) <= 2 + r0.iterations // 20
    # both within rtol of A x = b: ||x1 - x0|| <= 2 rtol cond(A) ||x||, cond ~ 1 / h^2 times the contrast, far
    # from attained for these smooth right-hand sides
    assert np.linalg.norm(x1 - x0) <= 1e-6 * np.linalg.norm(x0)
    ia, ja = S.get_csr()
    val, rhs = S.get_system()
    res = rhs - np.add.reduceat(val * x1[ja], ia[:-1])
    assert np.linalg.norm(res) <= 1.02e-9 * np.linalg.norm(rhs)
    again, x2 = S.solve(rtol=1e-9, max_iter=20000, want_du=True)
    assert again.iterations == r1.iterations and np.array_equal(x1, x2)  # bitwise repeatable
    # a budget below the need: the iterations asked for, a residual that is the true one
    if r1.iterations > 6:
        rb, xb = S.solve(rtol=1e-9, max_iter=5, want_du=True)
        assert not rb.converged and rb.reason == -3 and rb.iterations == 5
        rr = np.linalg.norm(rhs - np.add.reduceat(val * xb[ja], ia[:-1])) / np.linalg.norm(rhs)
        assert abs(rb.relres - rr) <= 1e-9 * rr
    S.close()


def test_resident_restarts_from_the_true_residual():
    """A target at the floor of the recurrences: the solve restarts inside."""
    S, _ = _system(1, 64)
    r, x = S.solve(rtol=1e-13, max_iter=5000, want_du=True)
    S.set_tuning("resident", 0)
    r0, x0 = S.solve(rtol=1e-13, max_iter=5000, want_du=True)
    assert r.converged == r0.converged and np.linalg.norm(x - x0) <= 1e-10 * np.linalg.norm(x0)
    S.close()


# sizes of which several fit the device together, and ones that need all of it
@pytest.mark.parametrize("sizes", [[(1, 90), (1, 90), (4, 24), (4, 24)],
                                   [(1, 20), (1, 40), (4, 12), (4, 30), (1, 500), (4, 60), (1, 64), (4, 16)]])
def test_resident_threads(sizes):
    systems = [_system(kind, N, s)[0] for s, (kind, N) in enumerate(sizes)]
    want = [S.solve(rtol=1e-9, want_du=True)[1] for S in systems]
    got = [None] * len(systems)

    def work(i):
        for _ in range(5):
            got[i] = systems[i].solve(rtol=1e-9, want_du=True)[1]
    ts = [threading.Thread(target=work, args=(i,)) for i in range(len(systems))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for g, w in zip(got, want):
        assert np.array_equal(g, w)
    for S in systems:
        assert S.get_tuning("resident_ran") == 1 and S.get_tuning("resident_gave_up") == 0
        S.close()


@pytest.mark.parametrize("pc", ["jacobi", "ic0", "amg"])
def test_a_wait_that_runs_out_leaves_the_solve_to_the_launches(pc):
    """No waiting at all: the first value of another workgroup that has not
    arrived ends the launch.  The solve is the launch-per-iteration one bit for
    bit, later solves stay there, and setting `resident` again tries anew."""
    from feng_amd.api import PC_AMG, PC_IC0, PC_JACOBI
    pcn = {"jacobi": PC_JACOBI, "ic0": PC_IC0, "amg": PC_AMG}[pc]
    S, _ = _system(4, 21)

    def solve():
        return S.solve(pc=pcn, rtol=1e-9, want_du=True)
    S.set_tuning("resident", 0)
    r0, x0 = solve()
    S.set_tuning("resident", 1)
    S.set_tuning("resident_wait_us", 0)
    for _ in range(2):
        r1, x1 = solve()
        assert S.get_tuning("resident_ran") == 0 and S.get_tuning("resident_gave_up") == 1
        assert r1.converged and r1.iterations == r0.iterations and np.array_equal(x1, x0)
    S.set_tuning("resident_wait_us", 50000)
    S.set_tuning("resident", 1)
    r2, x2 = solve()
    assert S.get_tuning("resident_ran") == 1 and S.get_tuning("resident_gave_up") == 0
    assert r2.converged and np.linalg.norm(x2 - x0) <= 1e-6 * np.linalg.norm(x0)
    S.close()


# rows of 8, 16 and 24 entries; one workgroup, its edge, many; 1024 threads (4, 52); rows too long (5, 6)
@pytest.mark.parametrize("pc", ["ic0", "learned"])
@pytest.mark.parametrize("kind, N", [(1, 2), (1, 3), (1, 24), (1, 150), (4, 3), (4, 9), (4, 30), (4, 52), (2, 12), (2, 90),
                                     (5, 6)])
def test_resident_split_equals_launch_per_iteration(kind, N, pc):
    from feng_amd.api import PC_IC0, PC_LEARNED
    print("resident split", kind, N, pc, flush=True)
    S, num = _system(kind, N)
    if pc == "learned":
        from feng_amd.learned import load_weights
        load_weights(S)
    pcn = PC_IC0 if pc == "ic0" else PC_LEARNED
    out = {}
    for resident in (0, 1):
        S.set_tuning("resident", resident)
        out[resident] = S.solve(pc=pcn, rtol=1e-9, max_iter=20000, want_du=True)
        assert S.get_tuning("resident_ran") == (resident and kind != 5) and S.get_tuning("resident_gave_up") == 0
    (r0, x0), (r1, x1) = out[0], out[1]
    if not r0.converged:  # a learned factor outside its training range: no iteration is possible in either form
        assert r0.iterations == r1.iterations == 0 and r1.reason == r0.reason
        S.close()
        return
    assert r1.converged and r1.relres <= 1e-9
    # as above: the same recurrences with sums in another order
    if r0.outer_iterations == r1.outer_iterations == 1:
        assert abs(r1.iterations - r0.iterations) <= 2 + r0.iterations // 20
    assert np.linalg.norm(x1 - x0) <= 1e-6 * np.linalg.norm(x0)
    ia, ja = S.get_csr()
    val, rhs = S.get_system()
    res = rhs - np.add.reduceat(val * x1[ja], ia[:-1])
    assert np.linalg.norm(res) <= 1.02e-9 * np.linalg.norm(rhs)
    assert r1.norm_rhs_inf == np.abs(rhs).max() and r1.norm_dx_inf == np.abs(x1).max()
    again, x2 = S.solve(pc=pcn, rtol=1e-9, max_iter=20000, want_du=True)
    assert again.iterations == r1.iterations and np.array_equal(x1, x2)  # bitwise repeatable
    if r1.iterations > 6:
        rb, xb = S.solve(pc=pcn, rtol=1e-9, max_iter=5, want_du=True)
        assert not rb.converged and rb.reason == -3 and rb.iterations == 5
        rr = np.linalg.norm(rhs - np.add.reduceat(val * xb[ja], ia[:-1])) / np.linalg.norm(rhs)
        assert abs(rb.relres - rr) <= 1e-9 * rr
    S.set_system(rhs=np.zeros_like(rhs))
    rz, xz = S.solve(pc=pcn, want_du=True)
    assert rz.converged and rz.iterations == 0 and not xz.any()
    S.close()


@pytest.mark.parametrize("pc", ["jacobi", "ic0", "amg"])
@pytest.mark.parametrize("prec", [0, 1])
def test_a_target_above_the_right_hand_side_takes_no_iteration(pc, prec):
    """atol above ||b||: the zero correction is the answer of the multigrid, the
    split and the refined solves (FP64 Jacobi-PCG aims at half the target and
    iterates), and no budget is none; both as by launches."""
    from feng_amd.api import PC_AMG, PC_IC0, PC_JACOBI, PREC_FP32_IR
    pcn = {"jacobi": PC_JACOBI, "ic0": PC_IC0, "amg": PC_AMG}[pc]
    S, _ = _system(4, 12)
    S.setToZero()
    S.assemble(3, PREC_FP32_IR)
    bn = np.linalg.norm(S.get_system()[1])
    for opts in (dict(atol=1.5 * bn), dict(atol=20.0 * bn), dict(max_iter=0)):
        out = []
        for resident in (0, 1):
            S.set_tuning("resident", resident)
            r, x = S.solve(pc=pcn, precision=prec, want_du=True, **opts)
            assert S.get_tuning("resident_ran") == resident
            out.append((r.iterations, r.outer_iterations, r.converged, r.reason, r.norm_rhs_inf))
            if (pc, prec) != ("jacobi", 0):
                assert out[-1][:4] == ((0, 0, False, -3) if "max_iter" in opts else (0, 0, True, 2))
                assert r.relres == 1.0 and not x.any() and r.norm_axb_inf == r.norm_rhs_inf
        assert out[0] == out[1], (opts, out)
    S.close()


@pytest.mark.parametrize("pc", ["jacobi", "ic0", "amg"])
def test_a_right_hand_side_that_is_not_a_number_is_reported(pc):
    from feng_amd.api import PC_AMG, PC_IC0, PC_JACOBI
    pcn = {"jacobi": PC_JACOBI, "ic0": PC_IC0, "amg": PC_AMG}[pc]
    S, _ = _system(4, 12)
    rhs = S.get_system()[1]
    rhs[3] = np.nan
    S.set_system(rhs=rhs)
    for resident in (0, 1):
        S.set_tuning("resident", resident)
        r = S.solve(pc=pcn, max_iter=50)
        assert S.get_tuning("resident_ran") == resident
        assert not r.converged and r.reason == -9 and np.isnan(r.relres)
    S.close()


@pytest.mark.parametrize("pc", ["jacobi", "ic0", "amg"])
@pytest.mark.parametrize("prec", [0, 1])
def test_a_target_below_the_floor_ends_after_the_same_restarts(pc, prec):
    """60 solves from a true residual at most, and then no reason code, as by
    launches; FP64 Jacobi-PCG has no such bound and ends with the budget or
    after 20 breakdowns of the recurrences."""
    from feng_amd.api import PC_AMG, PC_IC0, PC_JACOBI, PREC_FP32_IR
    pcn = {"jacobi": PC_JACOBI, "ic0": PC_IC0, "amg": PC_AMG}[pc]
    S, _ = _system(4, 12)
    S.setToZero()
    S.assemble(3, PREC_FP32_IR)
    out = []
    for resident in (0, 1):
        S.set_tuning("resident", resident)
        r, x = S.solve(pc=pcn, precision=prec, rtol=1e-17, max_iter=3000, want_du=True)
        assert S.get_tuning("resident_ran") == resident
        out.append(r)
        assert not r.converged and r.relres < 1e-14
        if (pc, prec) == ("jacobi", 0):
            assert r.reason == -3
        else:
            assert r.reason == 0 and r.outer_iterations == 60 and r.iterations < 3000
    S.close()


@pytest.mark.parametrize("pc", ["jacobi", "ic0", "amg"])
def test_a_launch_has_a_bounded_length(pc):
    """A solve that needs more iterations than one launch may take is the
    launch-per-iteration one; a budget within the limit is not affected."""
    from feng_amd.api import PC_AMG, PC_IC0, PC_JACOBI
    pcn = {"jacobi": PC_JACOBI, "ic0": PC_IC0, "amg": PC_AMG}[pc]
    S, _ = _system(4, 12)
    S.set_tuning("resident", 0)
    r0, x0 = S.solve(pc=pcn, rtol=1e-9, want_du=True)
    S.set_tuning("resident", 1)
    S.set_tuning("resident_max_iter", r0.iterations // 2)
    r1, x1 = S.solve(pc=pcn, rtol=1e-9, want_du=True)
    assert S.get_tuning("resident_ran") == 0 and S.get_tuning("resident_gave_up") == 0
    assert r1.converged and r1.iterations == r0.iterations and np.array_equal(x1, x0)
    r2 = S.solve(pc=pcn, rtol=1e-9, max_iter=r0.iterations // 2)
    assert S.get_tuning("resident_ran") == 1 and r2.reason == -3 and r2.iterations == r0.iterations // 2
    S.set_tuning("resident_max_iter", r0.iterations + 10)
    r3 = S.solve(pc=pcn, rtol=1e-9)
    assert S.get_tuning("resident_ran") == 1 and r3.converged
    S.close()


@pytest.mark.parametrize("pc", ["jacobi", "ic0"])
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("pipe", [0, 1, 2])
def test_pipe_kernel_picks_the_kernel(pc, prec, pipe):
    """One launch stands in for the tiled FP64 kernels and for the default choice
    at FE_PREC_FP32_IR; the kernels that pipe_kernel names otherwise run."""
    from feng_amd.api import PC_IC0, PC_JACOBI, PREC_FP32_IR
    pcn = {"jacobi": PC_JACOBI, "ic0": PC_IC0}[pc]
    S, _ = _system(4, 12)
    S.setToZero()
    S.assemble(3, PREC_FP32_IR)
    S.set_tuning("pipe_kernel", pipe)
    out = []
    for resident in (0, 1):
        S.set_tuning("resident", resident)
        out.append(S.solve(pc=pcn, precision=prec, rtol=1e-9, want_du=True))
    one = pipe == 2 or (pipe == 1 and prec == 0)
    assert S.get_tuning("resident_ran") == one
    assert out[0][0].converged and out[1][0].converged
    assert np.array_equal(out[0][1], out[1][1]) == (not one)
    S.close()

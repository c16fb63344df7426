"""Aggregation multigrid on the GPU (fe_amg.hip) against the CPU oracle
(oracle/fe_oracle_amg.py, pinned in tests/test_oracle_amg.py).

The hierarchy (rows and stored entries per level) is integer data and must
match exactly.  One V-cycle with FP64 level values matches the oracle to
1e-11 relative (the device sums the Galerkin entries, the l1 norms and the
row products in other orders, and inverts the coarsest level by Gauss-Jordan
instead of LAPACK); with FP32 level values (the default) to 1e-5, the FP32
rounding of the values carried through the cycle.  With FP32 level values the
nested PCG solves the coarse levels R .. D with the single-workgroup W-cycle
kernel (the levels it holds rounded to binary16 / bfloat16 as the oracle's
wcycle models them); its cycle matches oracle.wcycle to 1e-5.
"""
import numpy as np
import pytest
import scipy.sparse as sp

from oracle import fe_oracle_amg as amg

pytestmark = pytest.mark.gpu


def nrel(a, b):
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) / max(np.linalg.norm(b), 1e-300))


def _system(case):
    from feng_amd.api import FN_CONST, FN_ELEM, Fn, Mesh
    from feng_amd.problems import diffusion_system
    if case == "tet_grf_12":
        m = Mesh.cube(12)
        k, kind, deg = Fn(FN_ELEM, data=m.coeff_grf(0.1, 1.5, 64, 5)), 4, 1
    elif case == "p2_blocks_40":
        m = Mesh.square(40)
        k, kind, deg = Fn(FN_ELEM, data=m.coeff_blocks(16, 1e-2, 1e2, 9)), 2, 2
    else:  # p1_square_9: 64 unknowns, one level
        m = Mesh.square(9)
        k, kind, deg = Fn(FN_CONST, 1.0), 1, 2
    S, num = diffusion_system(m, kind, deg, k, Fn(FN_CONST, -1.0))
    S.assemble(3)
    return m, S, num


def _oracle_levels(S):
    ia, ja = S.get_csr()
    val, rhs = S.get_system()
    n = len(ia) - 1
    A = sp.csr_matrix((val, ja, ia), shape=(n, n))
    return A, rhs, amg.hierarchy(A)


@pytest.mark.parametrize("case", ["tet_grf_12", "p2_blocks_40", "p1_square_9"])
@pytest.mark.parametrize("variant", ["nested", "per_level", "header_tiles_big_block"])
def test_vcycle_matches_oracle(case, variant):
    """nested: the nested-ordered kernels (fe_amg_pcg.hip, the default);
    per_level: the per-level kernels over the original numbering."""
    print("case", case, variant, flush=True)
    m, S, num = _system(case)
    if variant != "nested":
        S.set_tuning("amg_kernel", 1)
    if variant == "header_tiles_big_block":
        # restriction through tile headers (the kernel for aggregates above
        # 256 rows) and larger levels in the single-workgroup kernel, whose
        # matrices it then reads from global memory
        S.set_tuning("amg_pad_tiles", 0)
        S.set_tuning("amg_block_rows", 8192)
    A, rhs, lv = _oracle_levels(S)
    r = np.random.default_rng(3).normal(size=A.shape[0])
    S.set_tuning("pc_values32", 0)
    z = S.amg_apply(r)
    rows, nnz = S.amg_levels()
    assert rows == [L.A.shape[0] for L in lv]
    assert nnz == [L.A.nnz for L in lv]
    zo = amg.vcycle(lv, r)
    assert nrel(z, zo) <= 1e-11, nrel(z, zo)
    if len(lv) == 1:
        assert nrel(A @ z, r) <= 1e-11
    S.set_tuning("pc_values32", 1)
    z32 = S.amg_apply(r)
    assert nrel(z32, zo) <= 1e-5, nrel(z32, zo)
    if variant == "nested":
        S.set_tuning("amg_wcycle", 1)
        z32w = S.amg_apply(r)
        R, D = S.get_tuning("amg_wcycle_level"), S.get_tuning("amg_wcycle_dense")
        if len(lv) > 2:
            assert R >= 1 and D > R, (R, D)
            zw = amg.wcycle(lv, r, R, D)
            assert nrel(z32w, zw) <= 1e-5, nrel(z32w, zw)
    S.close()


@pytest.mark.parametrize("N, R, D, kernel", [(40, 2, 4, "K64 + K32"), (64, 2, 4, "K160 + K32")])
def test_wcycle_kernel_matches_oracle_on_cubes(N, R, D, kernel):
    """The W-cycle kernel with two register levels (levels 2 and 3 of the P1
    tet GRF cubes 40^3 and 64^3, dense level 4) against oracle.wcycle;
    switched off (amg_wcycle 0, the default) the nested path is the V-cycle,
    with levels 1 .. coarsest in one launch (amg_fuse 1) bitwise equal to one
    launch per level (amg_fuse 0) and to the oracle's V-cycle to 1e-5."""
    from feng_amd.api import FN_CONST, FN_ELEM, Fn, Mesh
    from feng_amd.problems import diffusion_system
    print("W-cycle kernel", N, kernel, flush=True)
    m = Mesh.cube(N)
    S, num = diffusion_system(m, 4, 1, Fn(FN_ELEM, data=m.coeff_grf(0.1, 1.5, 512, 1)), Fn(FN_CONST, -1.0))
    S.assemble(3)
    A, rhs, lv = _oracle_levels(S)
    r = np.random.default_rng(11).normal(size=A.shape[0])
    S.set_tuning("amg_wcycle", 1)
    z = S.amg_apply(r)
    assert (S.get_tuning("amg_wcycle_level"), S.get_tuning("amg_wcycle_dense")) == (R, D)
    zo = amg.wcycle(lv, r, R, D)
    err = nrel(z, zo)
    print("W-cycle vs oracle", N, err, flush=True)
    assert err <= 1e-5, err
    S.set_tuning("amg_wcycle", 0)
    assert S.get_tuning("amg_wcycle_level") == 0
    S.set_tuning("amg_fuse", 1)
    zv = S.amg_apply(r)
    assert S.get_tuning("amg_fuse_grid") >= 2
    assert nrel(zv, amg.vcycle(lv, r)) <= 1e-5
    S.set_tuning("amg_fuse", 0)
    assert S.get_tuning("amg_fuse_grid") == 0
    assert np.array_equal(S.amg_apply(r), zv)
    S.close()


def test_numeric_setup_follows_new_values():
    m, S, num = _system("tet_grf_12")
    S.set_tuning("pc_values32", 0)
    r = np.random.default_rng(4).normal(size=num.nInc)
    S.amg_apply(r)
    S.update_coeff(0, 0, m.coeff_grf(0.1, 1.5, 64, 11))
    S.setToZero()
    S.assemble(3)
    A, rhs, lv = _oracle_levels(S)
    assert nrel(S.amg_apply(r), amg.vcycle(lv, r)) <= 1e-11
    S.close()


# amg_fp32_rows 0: FP32 iterations at FE_PREC_FP32_IR, as for systems of more than 700,000 rows
@pytest.mark.parametrize("fp32_rows", [700000, 0])
@pytest.mark.parametrize("case", ["tet_grf_16", "p2_blocks_64"])
def test_amg_pcg_converges(oracle, case, fp32_rows):
    from feng_amd.api import FN_CONST, FN_ELEM, PC_AMG, PC_JACOBI, PREC_FP32_IR, Fn, Mesh
    from feng_amd.problems import diffusion_system
    print("case", case, flush=True)
    if case == "tet_grf_16":
        m = Mesh.cube(16)
        k, kind, deg = Fn(FN_ELEM, data=m.coeff_grf(0.1, 1.5, 256, 2)), 4, 1
    else:
        m = Mesh.square(64)
        k, kind, deg = Fn(FN_ELEM, data=m.coeff_blocks(16, 1e-2, 1e2, 9)), 2, 2
    S, num = diffusion_system(m, kind, deg, k, Fn(FN_CONST, -1.0))
    S.assemble(3, PREC_FP32_IR)
    S.set_tuning("amg_fp32_rows", fp32_rows)
    rj = S.solve(pc=PC_JACOBI, rtol=1e-8, max_iter=20000)
    ra, du = S.solve(pc=PC_AMG, rtol=1e-8, want_du=True)
    ra32 = S.solve(pc=PC_AMG, precision=PREC_FP32_IR, rtol=1e-8, inner_rtol=1e-2)
    assert rj.converged and ra.converged and ra32.converged
    assert S.get_tuning("resident_ran") == (fp32_rows > 0) and (fp32_rows > 0 or ra32.outer_iterations >= 2)
    assert ra.iterations * 3 < rj.iterations, (ra.iterations, rj.iterations)
    ia, ja = S.get_csr()
    val, rhs = S.get_system()
    res = rhs - oracle.spmv(ia, ja, val, du)
    assert np.linalg.norm(res) <= 1.01e-8 * np.linalg.norm(rhs)
    S.close()


@pytest.mark.parametrize("resident", [1, 0])
@pytest.mark.parametrize("pcname", ["amg", "ic0"])
def test_graph_replay_matches_direct_launches(pcname, resident):
    """Iteration batches replayed from a captured HIP graph give the same
    iterates as direct launches, bit for bit, on every replayed solve (eager
    solves and host synchronisations in between).  Graphs hold the pipelined
    split and per-level multigrid iterations: a solve in one launch (resident)
    replays none and does not change either."""
    from feng_amd.api import PC_AMG, PC_IC0, PREC_FP32_IR
    pc = {"amg": PC_AMG, "ic0": PC_IC0}[pcname]
    m, S, num = _system("tet_grf_12")
    S.assemble(3, PREC_FP32_IR)
    if not resident:
        for key, v in (("resident", 0), ("amg_kernel", 1), ("amg_fp32_rows", 0), ("pipe_kernel", 1)):
            S.set_tuning(key, v)
    for prec in (0, PREC_FP32_IR):
        S.set_tuning("graph_iters", 0)
        r0, d0 = S.solve(pc=pc, precision=prec, rtol=1e-8, want_du=True)
        assert r0.converged
        for rep in range(3):
            S.set_tuning("graph_iters", 8)
            r1, d1 = S.solve(pc=pc, precision=prec, rtol=1e-8, want_du=True)
            assert r1.iterations == r0.iterations and r1.outer_iterations == r0.outer_iterations, (prec, rep)
            assert np.array_equal(d1, d0), (prec, rep)
            S.set_tuning("graph_iters", 0)
            r2, d2 = S.solve(pc=pc, precision=prec, rtol=1e-8, want_du=True)
            assert np.array_equal(d2, d0), (prec, rep)
    assert S.get_tuning("graphs") == (0 if resident else 2)  # one a precision, captured once
    S.close()


def test_vcycle_on_a_block_diagonal_batch_matches_oracle():
    """120 disjoint small problems in one system: every level keeps at least
    one row per problem, so coarsening stalls above the dense limit and the
    coarsest level is swept; hierarchy and V-cycle as the oracle's."""
    from feng_amd.batched import build_batch
    probs = [(6 + (p % 5), 1, 100 + p) for p in range(120)]
    b = build_batch([(N_, 1, s) for N_, _, s in probs], 1)
    S = b.S
    S.setToZero()
    S.assemble(3)
    A, rhs, lv = _oracle_levels(S)
    assert hasattr(lv[-1], "sweeps")
    r = np.random.default_rng(5).normal(size=A.shape[0])
    S.set_tuning("pc_values32", 0)
    z = S.amg_apply(r)
    rows, nnz = S.amg_levels()
    assert rows == [L.A.shape[0] for L in lv] and nnz == [L.A.nnz for L in lv]
    assert nrel(z, amg.vcycle(lv, r)) <= 1e-11
    S.close()


@pytest.mark.parametrize("fp32_rows", [700000, 0])
@pytest.mark.parametrize("case", ["tet_grf_16", "p2_blocks_64"])
def test_nested_pcg_matches_per_level_pcg(oracle, case, fp32_rows):
    """The nested-ordered PCG (standard CG, reductions folded into the next
    kernel) and the per-level pipelined PCG: both reach the FP64 target, in
    FP64 and with FP32 inner solves under FP64 refinement (amg_fp32_rows 0),
    the nested V-cycle in FP64 in one launch and by launches; with the V-cycle
    (amg_wcycle 0) their iteration counts are within 20% of each other, and
    the W-cycle kernel takes no more iterations than the V-cycle."""
    from feng_amd.api import FN_CONST, FN_ELEM, PC_AMG, PREC_FP32_IR, Fn, Mesh
    from feng_amd.problems import diffusion_system
    print("nested vs per-level", case, flush=True)
    if case == "tet_grf_16":
        m = Mesh.cube(16)
        k, kind, deg = Fn(FN_ELEM, data=m.coeff_grf(0.1, 1.5, 256, 2)), 4, 1
    else:
        m = Mesh.square(64)
        k, kind, deg = Fn(FN_ELEM, data=m.coeff_blocks(16, 1e-2, 1e2, 9)), 2, 2
    S, num = diffusion_system(m, kind, deg, k, Fn(FN_CONST, -1.0))
    S.assemble(3, PREC_FP32_IR)
    ia, ja = S.get_csr()
    val, rhs = S.get_system()
    out = {}
    S.set_tuning("amg_fp32_rows", fp32_rows)
    for kern in (2, 1, 3, 4):  # 3: nested with the V-cycle, 4: the same by launches
        S.set_tuning("amg_kernel", 2 if kern >= 3 else kern)
        S.set_tuning("amg_wcycle", 0 if kern >= 3 else 1)
        S.set_tuning("resident", int(kern != 4))
        for prec in (0, PREC_FP32_IR):
            r, du = S.solve(pc=PC_AMG, precision=prec, rtol=1e-8, inner_rtol=1e-4, want_du=True)
            assert r.converged and r.relres <= 1e-8, (kern, prec, r)
            res = rhs - oracle.spmv(ia, ja, val, du)
            assert np.linalg.norm(res) <= 1.01e-8 * np.linalg.norm(rhs), (kern, prec)
            one = kern == 3 and (prec == 0 or fp32_rows > 0)
            assert S.get_tuning("resident_ran") == one
            assert prec == 0 or fp32_rows > 0 or r.outer_iterations >= 2, (kern, r)
            out[(kern, prec)] = (r.iterations, du)
    for prec in (0, PREC_FP32_IR):
        itW, it1, itV = out[(2, prec)][0], out[(1, prec)][0], out[(3, prec)][0]
        print(case, "precision", prec, "iterations nested W / per-level / nested V:", itW, it1, itV, flush=True)
        assert abs(itV - it1) <= max(2, 0.2 * it1), (prec, itV, it1)
        assert itW <= itV + 1, (prec, itW, itV)
        assert abs(out[(4, prec)][0] - itV) <= 2, (prec, itV)
        for kern in (2, 3, 4):
            d2, d1 = out[(kern, prec)][1], out[(1, prec)][1]
            assert np.abs(d2 - d1).max() <= 1e-5 * np.abs(d1).max()
    S.close()

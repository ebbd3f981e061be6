"""Batched kernels that gather from tiles in LDS (divergence, fields, outer
residual): sample counts at and off the edges of the 16-sample chunks, with
and without each field term, against the single-sample path."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S, dmi, ku, field", [(64, False, True, False), (64, True, False, True), (63, True, True, False),
                                               (33, False, False, False), (18, True, True, True), (17, False, True, True)])
def test_tiles_match_single_sample(gpu_available, S, dmi, ku, field):
    """17,424 nodes: 545 tiles or more, more units than the kernels have
    blocks.  Both sides solve to 1e-13, so the fields agree to a few thousand
    times that (the systems' condition), 1e-9; the torque likewise."""
    from tetmag_amd import _native as N
    from tetmag_amd import problem as P
    from tetmag_amd.batch import BatchContext, from_batch, to_batch
    from tetmag_amd.context import FieldContext
    mat = P.Material(Ku=4e4 if ku else 0.0, ku_axis=(0.6, 0.0, 0.8), D=1e-3 if dmi else 0.0, B_ext=(0.01, 0.02, -0.03))
    prob = P.cuboid_problem("tiles", 32, 32, 15, 3.0, 0.1, 3, mat)
    assert prob.n * ((S + 15) // 16) >= 1024 * 32
    ctx = FieldContext(prob, tol=1e-13)
    try:
        if field:
            ctx.set_hext(prob.hext, 1e4 * np.random.default_rng(1).standard_normal(3 * prob.n))
        bc = BatchContext(ctx, S, N.TM_PREC_FP64)
        ms = P.smooth_random_fields(prob.mesh, S, seed=S)
        for rep in range(2):  # warm solves too
            dm, H, st = bc.eval_rhs_host(to_batch(ms))
            for s in (0, S // 2, S - 1):
                d1, h1, st1 = ctx.eval_rhs_host(ms[s])
                eh, ed = rel_l2(from_batch(H, s), h1), rel_l2(from_batch(dm, s), d1)
                print("S", S, "rep", rep, "sample", s, "Heff", eh, "dm/dt", ed, flush=True)
                assert eh < 1e-9 and ed < 1e-9
                assert abs(st["max_torque"][s] - st1["max_torque"]) <= 1e-9 * st1["max_torque"]
            ms = [m + 1e-3 * np.roll(m, 1) for m in ms]
        bc.close()
    finally:
        ctx.close()


@pytest.mark.parametrize("ny", [16, 15])
def test_inner_solve_tiles_match_fp64(gpu_available, ny):
    """64 FP32-preconditioned samples at and just under the size from which the
    inner solve's level-0 products come from tiles: 8,192 rows and 7,680.
    Both precisions solve to 1e-12; the demag potentials then agree to the
    systems' condition times that, 1e-8 (the bound of the solver's other tests)."""
    from tetmag_amd import _native as N
    from tetmag_amd import problem as P
    from tetmag_amd.batch import BatchContext, to_batch
    from tetmag_amd.context import FieldContext
    prob = P.cuboid_problem("inner tiles", 31, ny - 1, 15, 3.0, 0.1, 3, P.Material())
    assert (4 * prob.n >= 1024 * 32) == (ny == 16)
    ctx = FieldContext(prob, tol=1e-12)
    try:
        ms = to_batch(P.smooth_random_fields(prob.mesh, 64, seed=4))
        ms2 = ms + 1e-3 * np.roll(ms, 1, axis=1)
        u = {}
        for prec in (N.TM_PREC_FP64, N.TM_PREC_MIXED):
            bc = BatchContext(ctx, 64, prec)
            u[prec] = []
            for m in (ms, ms2):  # a cold and a warm solve
                bc.eval_rhs_host(m)
                u[prec] += list(bc.potentials())
            bc.close()
        for k, (a, b) in enumerate(zip(u[N.TM_PREC_MIXED], u[N.TM_PREC_FP64])):
            worst = max(rel_l2(a[:, s], b[:, s]) for s in range(64))
            print("ny", ny, "potential", k, worst, flush=True)
            assert worst < 1e-8
    finally:
        ctx.close()


@pytest.mark.parametrize("prec", ["FP64", "MIXED"])
@pytest.mark.parametrize("S, nx, ny, nz", [(1, 13, 11, 5), (16, 20, 20, 4), (17, 20, 20, 4), (63, 13, 11, 5), (40, 40, 30, 9), (33, 40, 30, 9)])
def test_coarsest_level_product(gpu_available, S, nx, ny, nz, prec):
    """Sample counts at and off the 16 of a block, coarsest levels reached from
    the first and from the second level.  Solves to 1e-13 on both sides: fields
    within a few thousand times that in FP64, 1e-9; 1e-8 for the mixed form
    (the bound of its other tests)."""
    from tetmag_amd import _native as N
    from tetmag_amd import problem as P
    from tetmag_amd.batch import BatchContext, from_batch, to_batch
    from tetmag_amd.context import FieldContext
    prob = P.cuboid_problem("coarse", nx, ny, nz, 3.0, 0.1, 3, P.Material())
    ctx = FieldContext(prob, tol=1e-13)
    try:
        print("n", prob.n, "levels", ctx.amg_levels(0), ctx.amg_levels(1), flush=True)
        bc = BatchContext(ctx, S, getattr(N, "TM_PREC_" + prec))
        ms = P.smooth_random_fields(prob.mesh, S, seed=S)
        dm, H, st = bc.eval_rhs_host(to_batch(ms))
        for s in sorted({0, S // 2, S - 1}):
            d1, h1, _ = ctx.eval_rhs_host(ms[s])
            eh, ed = rel_l2(from_batch(H, s), h1), rel_l2(from_batch(dm, s), d1)
            print("S", S, prec, "sample", s, eh, ed, flush=True)
            assert max(eh, ed) < (1e-9 if prec == "FP64" else 1e-8)
        bc.close()
    finally:
        ctx.close()


@pytest.mark.parametrize("S, nz, prec, names", [
    (18, 15, "FP64", {"k_b_div", "k_b_eval_t<DMI>", "k_b_resid_t<double>", "k_b_cg_spmv_t", "k_b_up_t (level 0)"}),
    (64, 15, "MIXED", {"k_b_div", "k_b_eval_t<DMI>", "k_b_resid_t<float>", "k_b_cg_spmv_t", "k_b_up_t (level 0)"}),
    (18, 3, "FP64", {"k_b_div_l2", "k_b_eval<DMI>", "k_b_resid<double>", "k_b_cg_spmv", "k_b_up (level 0)"}),
    (64, 3, "MIXED", {"k_b_div_l2", "k_b_eval_w<DMI>", "k_b_resid<float>", "k_b_cg_spmv_w", "k_b_up_w (level 0)"})])
def test_kernel_times_name_what_runs(gpu_available, S, nz, prec, names):
    """17,424 and 4,356 nodes: with tiles and gathering from L2."""
    from tetmag_amd import _native as N
    from tetmag_amd import problem as P
    from tetmag_amd.batch import BatchContext
    from tetmag_amd.context import FieldContext
    prob = P.cuboid_problem("names", 32, 32, nz, 3.0, 0.1, 3, P.Material(D=1e-3))
    ctx = FieldContext(prob, tol=1e-12)
    try:
        bc = BatchContext(ctx, S, getattr(N, "TM_PREC_" + prec))
        got = [k["kernel"] for k in bc.time_kernels(1)]
        print(S, prob.n, prec, got, flush=True)
        assert names <= set(got)
        bc.close()
    finally:
        ctx.close()

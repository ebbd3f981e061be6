"""The captured RK4 step that a batch keeps between calls of tm_batch_run_rk4:
what it reads belongs to the batch, or is part of what decides whether it can
be replayed."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


def _problem():
    from tetmag_amd import problem as P
    prob = P.small_problem(nx=18, ny=14, nz=5, h=3.0, jitter=0.1, seed=41, Ku=5e4, B_ext=(0.01, 0.0, -0.02))
    return prob, 20e-3 * prob.time_scale()


def _set_solvers(ctx, precond):
    from tetmag_amd import _native as N
    rpN, colN, valN = ctx.prob.neumann_matrix()
    rpD, colD, valD = ctx.prob.dirichlet_matrix()
    a = [N.i32(rpN), N.i32(colN), N.f64(valN), N.i32(rpD), N.i32(colD), N.f64(valD)]
    N.check(N.lib().tm_ctx_set_demag_solvers(ctx.h, *[N.ptr(x) for x in a], precond), "tm_ctx_set_demag_solvers")


@pytest.mark.parametrize("prec", ["FP64", "MIXED"])
@pytest.mark.parametrize("precond", ["AMG", "JACOBI"])
def test_survives_new_solvers_of_the_context(gpu_available, prec, precond):
    """tm_ctx_set_demag_solvers frees the hierarchy that the batch was made from
    and makes another (or none).  The batch goes on with the one it has, replayed
    and host-polled, as a batch on an untouched context does; memory freed
    since is filled with NaN in between.  (64 FP64 samples apply the coarsest
    level's inverse and the last restriction as one matrix, 64 mixed ones apart.)"""
    import torch
    from tetmag_amd import _native as N
    from tetmag_amd import problem as P
    from tetmag_amd.batch import BatchContext, to_batch
    from tetmag_amd.context import FieldContext
    prob, dtau = _problem()
    m = to_batch(P.smooth_random_fields(prob.mesh, 64, seed=31, lam_min=10.0, lam_max=60.0))
    ca, cb = FieldContext(prob, tol=1e-12), FieldContext(prob, tol=1e-12)
    a, b = BatchContext(ca, 64, getattr(N, "TM_PREC_" + prec)), BatchContext(cb, 64, getattr(N, "TM_PREC_" + prec))
    try:
        for bc in (a, b):
            bc.set_mag(m)
        for rep in range(3):
            _, ra = a.run_rk4(dtau, 3, use_graph=True)
            b.run_rk4(dtau, 3)
            d = rel_l2(a.get_mag(), b.get_mag())
            print(prec, precond, rep, ra["graph_steps"], ra["captures"], d, flush=True)
            # the bounds of the captured step's other test
            assert d < (1e-11 if prec == "FP64" else 1e-9)
            _set_solvers(ca, getattr(N, "TM_PRECOND_" + precond))
            fill = [torch.full((k,), float("nan"), dtype=torch.float64, device="cuda") for k in (1 << 14, 1 << 17, 1 << 20)]
            torch.cuda.synchronize()
            del fill
        Ha, Hb = a.eval_rhs_host(m)[1], b.eval_rhs_host(m)[1]
        assert rel_l2(Ha, Hb) < 1e-8
    finally:
        a.close()
        b.close()
        ca.close()
        cb.close()

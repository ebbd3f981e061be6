"""A batch with one sample whose magnetisation is not finite: the call says so
(TM_ERR_NONFINITE, as the single-sample path), the other samples come out as in
a batch without it, and the sample is right again as soon as its input is."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def base(gpu_available):
    from tetmag_amd import problem as P
    from tetmag_amd.context import FieldContext
    prob = P.small_problem(nx=18, ny=14, nz=5, h=3.0, jitter=0.1, seed=41, Ku=5e4, B_ext=(0.01, 0.0, -0.02))
    ctx = FieldContext(prob, tol=1e-12)
    yield prob, ctx
    ctx.close()


def _fails(N, call):
    with pytest.raises(N.TetmagError) as e:
        call()
    assert e.value.status == N.TM_ERR_NONFINITE


@pytest.mark.parametrize("prec", ["FP64", "MIXED", "MIXED_BEMI8"])
@pytest.mark.parametrize("first", [False, True])
def test_evaluation(base, prec, first):
    """first: the very first solve of the batch already meets the NaN.  Both
    batches solve to 1e-12; their samples agree to the systems' condition
    times that, 1e-8 (the bound of the batch tests; int8 products: 1e-6)."""
    from tetmag_amd import _native as N
    from tetmag_amd import problem as P
    from tetmag_amd.batch import BatchContext, to_batch
    prob, ctx = base
    S, k = 5, 2
    tol = 1e-6 if prec == "MIXED_BEMI8" else 1e-8
    ok = to_batch(P.smooth_random_fields(prob.mesh, S, seed=6))
    bad = ok.copy()
    bad[1, prob.n // 2, k] = np.nan
    a, b = BatchContext(ctx, S, getattr(N, "TM_PREC_" + prec)), BatchContext(ctx, S, getattr(N, "TM_PREC_" + prec))
    others = [s for s in range(S) if s != k]
    if not first:
        a.eval_rhs_host(ok)
        b.eval_rhs_host(ok)
    ref = b.eval_rhs_host(ok)[1]
    for _ in range(2):
        a.set_mag(bad)
        _fails(N, lambda: a.eval_rhs(None, want_heff=True))
        ctx.synchronize()
        H = a.heff.cpu().numpy()
        print(prec, first, [rel_l2(H[:, :, s], ref[:, :, s]) for s in others], flush=True)
        assert all(rel_l2(H[:, :, s], ref[:, :, s]) < tol for s in others)
        assert np.isnan(H[:, :, k]).any()
    for rep in range(3):  # finite again, from the first call on
        m = ok + 1e-3 * rep * np.roll(ok, 1, axis=1)
        Ha, Hb = a.eval_rhs_host(m)[1], b.eval_rhs_host(m)[1]
        assert np.isfinite(Ha).all()
        assert all(rel_l2(Ha[:, :, s], Hb[:, :, s]) < tol for s in range(S))
    a.close()
    b.close()


@pytest.mark.parametrize("graph", [False, True])
def test_steps(base, graph):
    """RK4 steps of 64 samples, host-polled and captured: every step is taken,
    a captured one is not redone for the sake of the sample that cannot converge."""
    from tetmag_amd import _native as N
    from tetmag_amd import problem as P
    from tetmag_amd.batch import BatchContext, to_batch
    import ctypes as C
    prob, ctx = base
    S, k, steps = 64, 41, 4
    dtau = 20e-3 * prob.time_scale()
    ok = to_batch(P.smooth_random_fields(prob.mesh, S, seed=6))
    bad = ok.copy()
    bad[0, 7, k] = np.nan
    a, b = BatchContext(ctx, S, N.TM_PREC_MIXED), BatchContext(ctx, S, N.TM_PREC_MIXED)
    b.set_mag(ok)
    b.run_rk4(dtau, steps)
    a.set_mag(bad)
    rk = N.RK4Stats()
    st = N.lib().tm_batch_run_rk4(a.h, dtau, steps, prob.alpha, N.TM_LLG_CLASSIC, int(graph), None, C.byref(rk))
    print("graph", graph, rk.as_dict(), flush=True)
    assert st == N.TM_ERR_NONFINITE
    assert rk.sync_steps + rk.graph_steps == steps and rk.redone_steps == 0
    if graph:
        assert rk.graph_steps >= steps - 1
    ma, mb = a.get_mag(), b.get_mag()
    assert np.isnan(ma[:, :, k]).any()
    for s in range(S):
        if s != k:
            assert rel_l2(ma[:, :, s], mb[:, :, s]) < 1e-8
    a.close()
    b.close()

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


@pytest.mark.parametrize("prec", ["FP64", "MIXED_BEMI8"])
def test_replayed_only_for_what_it_was_captured_for(gpu_available, prec):
    """One batch runs captured, another the same calls host-polled, while what
    the step depends on changes from call to call: the time step, the damping,
    the LLG form, the samples' fields, the per-node field (set, changed,
    cleared) and the buffer that holds m (an odd number of fused Euler steps
    swaps it).  Each is returned to its first value, so that the kept step of
    another call would fit in all but one of them."""
    from tetmag_amd import _native as N
    from tetmag_amd import problem as P
    from tetmag_amd.batch import BatchContext, to_batch
    from tetmag_amd.context import FieldContext
    prob, dt = _problem()
    S, n = 64, prob.n
    m = to_batch(P.smooth_random_fields(prob.mesh, S, seed=31, lam_min=10.0, lam_max=60.0))
    ctx = FieldContext(prob, tol=1e-12)
    a, b = BatchContext(ctx, S, getattr(N, "TM_PREC_" + prec)), BatchContext(ctx, S, getattr(N, "TM_PREC_" + prec))
    g = np.random.default_rng(2)
    field = 2e5 * g.standard_normal(3 * n)
    H0 = np.stack([np.linspace(-3e4, 3e4, S), np.zeros(S), np.full(S, 1e4)])
    tol = 1e-11 if prec == "FP64" else 1e-9
    calls = [("first", {}), ("again", {}), ("dt", {"dtau": 0.4 * dt}), ("dt back", {}), ("alpha", {"alpha": 0.02}),
             ("alpha back", {}), ("form", {"variant": N.TM_LLG_NOPREC}), ("form back", {}),
             ("samples' fields", {"H": -40 * H0}), ("samples' fields back", {}), ("node field", {"field": field}),
             ("other node field", {"field": -field}), ("cleared", {}), ("node field again", {"field": field}),
             ("m swapped", {"euler": 1}), ("m swapped back", {"euler": 1})]
    replayed = 0
    try:
        for bc in (a, b):
            bc.set_mag(m)
        for name, c in calls:
            before = a.get_mag()
            ctx.set_hext(prob.hext, c.get("field"))
            for bc in (a, b):
                bc.set_zeeman(c.get("H", H0))
                for _ in range(c.get("euler", 0)):
                    bc.eval_euler(dt, stats=False)
            kw = {"alpha": c.get("alpha", prob.alpha), "variant": c.get("variant", N.TM_LLG_CLASSIC)}
            _, ra = a.run_rk4(c.get("dtau", dt), 2, use_graph=True, **kw)
            b.run_rk4(c.get("dtau", dt), 2, **kw)
            ctx.synchronize()
            ma, mb = a.get_mag(), b.get_mag()
            d, moved = rel_l2(ma, mb), rel_l2(ma, before)
            print(f"{prec} {name}: replayed {ra['graph_steps']}, captured {ra['captures']}, apart {d:.1e}, "
                  f"moved {moved:.1e}", flush=True)
            replayed += ra["graph_steps"]
            # the two drift apart from call to call: each call's own bound adds up
            assert d < tol * (1 + [x for x, _ in calls].index(name)) and moved > 1e-4
        assert replayed >= len(calls)
    finally:
        a.close()
        b.close()
        ctx.close()


@pytest.mark.parametrize("prec", ["FP64", "MIXED"])
@pytest.mark.parametrize("how", ["set_mag", "eval_rhs"])
def test_first_step_of_a_given_state_is_host_polled(gpu_available, prec, how):
    """The budgets and kept solutions of one state say nothing about another: a
    replay would miss the tolerance, be redone host-polled and be captured
    anew.  Replays go on as soon as the state is the batch's own again."""
    from tetmag_amd import _native as N
    from tetmag_amd import problem as P
    from tetmag_amd.batch import BatchContext, to_batch
    from tetmag_amd.context import FieldContext
    prob, dt = _problem()
    fields = [to_batch(P.smooth_random_fields(prob.mesh, 64, seed=k, lam_min=10.0, lam_max=60.0)) for k in range(4)]
    ctx = FieldContext(prob, tol=1e-12)
    a, b = BatchContext(ctx, 64, getattr(N, "TM_PREC_" + prec)), BatchContext(ctx, 64, getattr(N, "TM_PREC_" + prec))
    try:
        for k, m in enumerate(fields):
            for bc in (a, b):
                if how == "set_mag":
                    bc.set_mag(m)
                else:
                    bc.eval_rhs_host(m)
            _, ra = a.run_rk4(dt, 1, use_graph=True)
            b.run_rk4(dt, 1)
            print(prec, how, k, {x: ra[x] for x in ("sync_steps", "graph_steps", "redone_steps", "captures")}, flush=True)
            assert (ra["sync_steps"], ra["graph_steps"], ra["redone_steps"], ra["captures"]) == (1, 0, 0, 0)
            replayed = sum(a.run_rk4(dt, 2, use_graph=True)[1]["graph_steps"] for _ in range(3))
            b.run_rk4(dt, 6)
            assert replayed >= 4
            assert rel_l2(a.get_mag(), b.get_mag()) < (1e-11 if prec == "FP64" else 1e-9)
    finally:
        a.close()
        b.close()
        ctx.close()


@pytest.mark.parametrize("prec", ["FP64", "MIXED_BEMI8"])
def test_live_gemm_events_leave_captured_steps_out(gpu_available, prec):
    """tm_batch_gemm_live while a step is captured and replayed: the host-polled
    step's four products are recorded, the replays' are not, and nothing that
    follows fails."""
    from tetmag_amd import _native as N
    from tetmag_amd import problem as P
    from tetmag_amd.batch import BatchContext, to_batch
    from tetmag_amd.context import FieldContext
    prob, dt = _problem()
    ctx = FieldContext(prob, tol=1e-12)
    bc = BatchContext(ctx, 64, getattr(N, "TM_PREC_" + prec))
    try:
        bc.set_mag(to_batch(P.smooth_random_fields(prob.mesh, 64, seed=31, lam_min=10.0, lam_max=60.0)))
        for _ in range(2):
            bc.gemm_live(True)
            _, rk = bc.run_rk4(dt, 4, use_graph=True)
            ms, count = bc.gemm_live(False)
            print(prec, rk, ms, count, flush=True)
            assert rk["graph_steps"] >= 3 and count == 4 * rk["sync_steps"] and (ms > 0) == (count > 0)
        bc.gemm_live(True)
        bc.eval_euler(dt, stats=False)
        assert bc.gemm_live(False)[1] == 1
    finally:
        bc.close()
        ctx.close()

"""Forms of the single-sample solver and of the boundary product that are
chosen by size: no AMG level (dense), one level with and without the dense
coarse product, several levels, and the one-lane-per-row form of large
systems; few and many column splits of the boundary product."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("which", ["neumann", "dirichlet"])
@pytest.mark.parametrize("cells", [(4, 4, 3), (9, 8, 5), (20, 20, 4), (24, 22, 9), (39, 37, 21), (53, 51, 51)])
def test_solver_forms(gpu_available, cells, which):
    """||b - A x|| <= tol ||b|| plus the drift of the recursive residual, at
    most eps ||A|| ||x|| per iteration; from zero, from the solver's own
    earlier solutions (three smoothly changing right-hand sides) and b = 0."""
    import scipy.sparse as sp
    from tetmag_amd import _native as N
    from tetmag_amd import problem as P
    prob = P.cuboid_problem("forms", *cells, 3.0, 0.1, 5)
    n = prob.n
    rp, col, val = prob.neumann_matrix() if which == "neumann" else prob.dirichlet_matrix()
    A = sp.csr_matrix((val, col, rp), shape=(n, n))
    norm = abs(A).sum(axis=1).max()
    h = C.c_void_p()
    L = N.lib()
    N.check(L.tm_solver_create(n, N.ptr(rp), N.ptr(col), N.ptr(val), N.TM_PRECOND_AMG, C.byref(h)), "create")
    try:
        rng = np.random.default_rng(8)
        b0, b1 = rng.standard_normal((2, n))
        x = np.zeros(n)
        it, tol = C.c_int(), 1e-10
        for k, warm in enumerate((0, 2, 2, 2, 0)):
            b = b0 + 1e-2 * k * b1
            N.check(L.tm_solver_solve(h, N.ptr(b), N.TM_HOST, N.ptr(x), N.TM_HOST, tol, 1000, warm, C.byref(it), None),
                    "solve")
            bound = tol * np.linalg.norm(b) + (it.value + 1) * 2.3e-16 * norm * np.linalg.norm(x)
            r = np.linalg.norm(b - A @ x)
            print(cells, which, n, "warm", warm, "iterations", it.value, "residual", r / np.linalg.norm(b), flush=True)
            assert r <= bound
        zero = np.zeros(n)
        for warm in (2, 0):
            N.check(L.tm_solver_solve(h, N.ptr(zero), N.TM_HOST, N.ptr(x), N.TM_HOST, tol, 1000, warm, None, None), "zero")
            assert not x.any()
    finally:
        L.tm_solver_destroy(h)


@pytest.mark.parametrize("b", [1, 2, 17, 255, 1122, 2049, 4111])
def test_boundary_product_splits(gpu_available, b):
    """y = B x against torch: both sum b products, so they differ by at most
    2 b eps |B| |x| (and far less on average)."""
    import torch
    from tetmag_amd import _native as N
    f = N.lib().tm_bem_apply_noalloc
    f.argtypes = [C.c_int, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p]
    ld = (b + 1) // 2 * 2
    g = torch.Generator(device="cuda").manual_seed(b)
    B = torch.randn((b, ld), generator=g, dtype=torch.float64, device="cuda")  # column j at B[j]
    x = torch.randn(b, generator=g, dtype=torch.float64, device="cuda")
    y = torch.full((b,), float("nan"), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    assert f(b, ld, B.data_ptr(), x.data_ptr(), y.data_ptr(), None) == N.TM_OK
    torch.cuda.synchronize()
    M = B[:, :b].T.contiguous()
    assert bool(((y - M @ x).abs() <= 2 * b * 2.3e-16 * (M.abs() @ x.abs())).all())

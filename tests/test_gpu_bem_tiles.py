"""The batched boundary products at the edges of their tiles.  From int8
digits: 16-row tiles, 8 or 4 per block; 64-column chunks.  FP64 (16 to 64 columns):
64 to 256 rows per block; 8- to 32-column chunks.  Both take three chunks per
pass of the loop and split the columns over several ranges."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec, S, tol", [("MIXED_BEMI8", 64, 2e-7), ("MIXED_BEMI8", 5, 2e-7), ("FP64", 64, 1e-13), ("FP64", 1, 1e-13),
                                          ("FP64", 16, 1e-13), ("FP64", 17, 1e-13), ("FP64", 48, 1e-13), ("FP64", 49, 1e-13)])
@pytest.mark.parametrize("nx, ny, nz", [(2, 2, 1), (5, 3, 2), (7, 3, 2), (6, 5, 4), (13, 8, 1), (12, 12, 3), (23, 11, 4)])
def test_product_at_tile_edges(gpu_available, nx, ny, nz, prec, S, tol):
    """Against the dense FP64 product on the host.  Five digits of B and six of
    U with the products p + q <= 5 kept err by about 2^-35 of the row
    maximum per entry; 2e-7 relative bounds the sum.  FP64 sums of 18 to 780
    terms: 1e-13.  (The bounds of the products' other test.)"""
    from tetmag_amd import _native as N
    from tetmag_amd import problem as P
    from tetmag_amd.batch import BatchContext
    from tetmag_amd.context import FieldContext
    prob = P.cuboid_problem("edges", nx, ny, nz, 3.0, 0.1, 3, P.Material())
    ctx = FieldContext(prob, tol=1e-12)
    try:
        bc = BatchContext(ctx, S, getattr(N, "TM_PREC_" + prec))
        B = ctx.bem_matrix()
        b = B.shape[0]
        X = np.random.default_rng(b).standard_normal((b, S))
        for x in (X, X[::-1].copy()):
            e = rel_l2(bc.bem_apply(x), B @ x)
            print("b", b, "tiles", -(-b // 16), "chunks", -(-b // 64), bc.gemm_info(), "err", e, flush=True)
            assert e < tol
        bc.close()
    finally:
        ctx.close()

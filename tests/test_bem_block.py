"""tm_bem_apply_noalloc on a block of a larger matrix (leading dimension well
above the block's size): the column splits' partial products are kept at a
stride of ld, so a large ld leaves room for fewer splits."""
import ctypes as C

import numpy as np
import pytest


def _noalloc():
    from tetmag_amd import _native as N
    f = N.lib().tm_bem_apply_noalloc
    f.argtypes = [C.c_int, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p]
    f.restype = C.c_int
    return N, f


# the largest even ld whose partials fit at 256 columns per split: 32 MiB hold
# 4,194,304 doubles, b rows in tiles of 2,048 take min(b / 256, 1,024 / tiles) splits
LIMITS = [(64, 4194304), (511, 4194304), (512, 2097152), (1122, 1048576), (4111, 262144), (8192, 131072), (92000, 93206)]


@pytest.mark.parametrize("b, ld", LIMITS)
def test_accepted_sizes(native, b, ld):
    """Accepted up to the limit, refused above it, decided before any device
    work (without a device the accepted call then fails there)."""
    N, f = _noalloc()
    count = C.c_int()
    if N.lib().tm_device_count(C.byref(count)) == N.TM_OK and count.value > 0:
        pytest.skip("the size check alone: needs a machine without a GPU")
    buf = np.zeros(4)
    p = buf.ctypes.data + (-buf.ctypes.data) % 16
    assert f(b, ld, p, p, p, None) not in (N.TM_OK, N.TM_ERR_BAD_ARG)
    assert f(b, ld + 2, p, p, p, None) == N.TM_ERR_BAD_ARG


@pytest.mark.gpu
@pytest.mark.parametrize("b, ld", [(64, 1 << 20), (1122, 59920), (4111, 16386), (4111, 65536)])
def test_product_of_a_block(gpu_available, b, ld):
    """Against torch, as the other split tests: at most 2 b eps |B| |x| apart."""
    import torch
    N, f = _noalloc()
    g = torch.Generator(device="cuda").manual_seed(b)
    B = torch.zeros((b, ld), dtype=torch.float64, device="cuda")  # column j at B[j]
    B[:, :b] = torch.randn((b, b), generator=g, dtype=torch.float64, device="cuda")
    x = torch.randn(b, generator=g, dtype=torch.float64, device="cuda")
    y = torch.full((b,), float("nan"), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    print("b", b, "ld", ld, flush=True)
    assert f(b, ld, B.data_ptr(), x.data_ptr(), y.data_ptr(), None) == N.TM_OK
    torch.cuda.synchronize()
    M = B[:, :b].T.contiguous()
    assert bool(((y - M @ x).abs() <= 2 * b * 2.3e-16 * (M.abs() @ x.abs())).all())


@pytest.mark.gpu
@pytest.mark.parametrize("b, ld, i0", [(64, 1000, 936), (1121, 5000, 3878), (2050, 6000, 3950), (4110, 4200, 90)])
def test_block_at_the_end_of_its_matrix(gpu_available, b, ld, i0):
    """The last rows and columns of a matrix, whose memory ends with the block's
    last column: only rows of the block are read (an odd b shares its last pair
    with the row after it), and what surrounds it (NaN here) has no part in the sums."""
    import torch
    N, f = _noalloc()
    assert i0 % 2 == 0 and b <= ld - i0 <= b + 1
    g = torch.Generator(device="cuda").manual_seed(b)
    A = torch.full((b, ld), float("nan"), dtype=torch.float64, device="cuda")  # column j at A[j]
    A[:, i0:i0 + b] = torch.randn((b, b), generator=g, dtype=torch.float64, device="cuda")
    x = torch.randn(b, generator=g, dtype=torch.float64, device="cuda")
    y = torch.full((b,), float("nan"), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    print("b", b, "ld", ld, "first row", i0, flush=True)
    assert f(b, ld, A.data_ptr() + 8 * i0, x.data_ptr(), y.data_ptr(), None) == N.TM_OK
    torch.cuda.synchronize()
    M = A[:, i0:i0 + b].T.contiguous()
    assert bool(((y - M @ x).abs() <= 2 * b * 2.3e-16 * (M.abs() @ x.abs())).all())

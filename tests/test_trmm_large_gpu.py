"""Triangles so large that the launch sizes of TRMM's own passes matter.

Bar: exact (integer entries).  The triangle is 2 on the diagonal and 1 in its
first row or column, so every entry of the product is known without forming it.
"""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side,uplo", [("L", "U"), ("R", "L")])
def test_strmm_65536_unknowns(torch_cuda, side, uplo):
    """One workgroup per 256 rows of every column would be 2^32 threads."""
    torch = torch_cuda
    from zynum_amd import _lib

    lib = _lib.load()
    na, other = 65536, 3
    if torch.cuda.mem_get_info()[0] < 45 << 30:
        pytest.skip("needs 35 GiB of device memory")
    i = lambda v: C.byref(C.c_int32(v))  # noqa: E731
    a = torch.zeros((na, na), device="cuda")  # a[j, i]: column j, row i
    a.diagonal().fill_(2.0)
    if uplo == "U":
        a[1:, 0] = 1.0  # first row
    else:
        a[0, 1:] = 1.0  # first column
    m, n = (na, other) if side == "L" else (other, na)
    b = torch.arange(m * n, device="cuda").remainder_(5).reshape(n, m).float()
    B = b.T.double()
    want = 2.0 * B
    if side == "L":  # row 0 of op(A) is (2, 1, 1, ...)
        want[0] += B[1:].sum(0)
    else:  # column 0 of A is (2, 1, 1, ...)
        want[:, 0] += B[:, 1:].sum(1)
    lib.strmm_(side.encode(), uplo.encode(), b"N", b"N", i(m), i(n), C.byref(C.c_float(1.0)), a.data_ptr(), i(na),
               b.data_ptr(), i(m))
    status = lib.zynum_gpu_last_status()
    torch.cuda.synchronize()
    lib.zynum_blas_shutdown()  # gives the 17 GB workspace back
    assert status == _lib.OK
    assert torch.equal(b.T.double(), want)

"""The error of FP32 products on the bf16 matrix cores where it is largest:
operands whose dropped part products are largest, sums of a single term, and
the routines that run on the same products.
"""
import ctypes as C

import pytest

from test_gemm_f32_split_gpu import FP32_TILE, call, draw
from test_gemm_f32_split_range_gpu import U, product

pytestmark = pytest.mark.gpu
# significand whose square loses most: 2^-24.01 of it
WORST = 1.0038986206054688


@pytest.mark.parametrize("shape", [(4096, 4096, 320), (2048, 2048, 2049), (4096, 4096, 8192)])
@pytest.mark.parametrize("signs", ["same", "mixed"])
def test_largest_dropped_products(torch_cuda, shape, signs):
    """Every product loses 2^-24 of itself, all with one sign or with both; the
    sum is rounded six times in 16 terms, by a unit in the last place at most."""
    torch = torch_cuda
    m, n, k = shape
    A, B = torch.full((k, m), WORST, device="cuda"), torch.full((n, k), WORST, device="cuda")
    if signs == "mixed":
        A, B = (x * torch.where(draw(torch, "uniform", x.shape, 5 + i) < 0, -1.0, 1.0) for i, x in enumerate((A, B)))
    ref = B.double() @ A.double()
    got = product(torch, m, n, k, "N", "N", A, B, 0)
    mag = k * WORST**2
    bound = (U * (1 + 2.0**-9) + 6 * ((k + 15) // 16) * 2 * U) * mag
    assert bool(((got.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("shape", [(4096, 4096, 333), (2048, 2048, 2049)])
def test_sums_of_one_term(torch_cuda, shape):
    """A scaled permutation: each sum is one product, short of 2^-24 of itself,
    the part products in it rounded to the last place (those before the last are
    2^-7 of it); times a power of two it is exact."""
    torch = torch_cuda
    m, n, k = shape
    A = torch.zeros((k, m), device="cuda")
    i = torch.arange(m, device="cuda")
    B = draw(torch, "normal", (n, k), 4)
    A[(i * 37 + 5) % k, i] = draw(torch, "positive", (m,), 3) + 0.5
    exact = B.double()[:, (i * 37 + 5) % k] * A[(i * 37 + 5) % k, i].double()
    got = product(torch, m, n, k, "N", "N", A, B, 0)
    bound = (U * (1 + 2.0**-9) + 2 * U * (1 + 5 * 2.0**-7)) * exact.abs()
    assert bool(((got.double() - exact).abs() <= bound).all())
    A[(i * 37 + 5) % k, i] = torch.exp2(torch.remainder(i, 9).float() - 4)
    exact = B[:, (i * 37 + 5) % k] * A[(i * 37 + 5) % k, i]
    assert torch.equal(product(torch, m, n, k, "N", "N", A, B, 0), exact)


def expanded(torch, A, uplo, kind):
    """The full matrix a routine reads (A rows x columns)."""
    tri = torch.tril(A) if uplo == "L" else torch.triu(A)
    return tri + tri.T - torch.diag(torch.diagonal(tri)) if kind == "symm" else tri


@pytest.mark.parametrize("routine", ["symm", "trmm"])
@pytest.mark.parametrize("side,uplo", [("L", "L"), ("R", "U"), ("L", "U"), ("R", "L")])
def test_symm_and_trmm_error_at_most_the_fp32_tile(torch_cuda, routine, side, uplo):
    """Against one product of the expanded matrix on the FP32 instruction."""
    torch = torch_cuda
    from zynum_amd import _lib

    lib = _lib.load()
    m, n = 3001, 2500
    na = m if side == "L" else n
    i = lambda v: C.byref(C.c_int32(v))  # noqa: E731
    one, zero = C.byref(C.c_float(1.0)), C.byref(C.c_float(0.0))
    A, B = draw(torch, "uniform", (na, na), 1), draw(torch, "uniform", (n, m), 2)  # column j is row j
    S = expanded(torch, A.T, uplo, routine)  # rows x columns
    ref = ((S.double() @ B.T.double()) if side == "L" else (B.T.double() @ S.double())).T
    fp32 = torch.empty((n, m), device="cuda")
    s_cols = S.T.contiguous()
    if side == "L":
        call(m, n, m, "N", "N", s_cols, m, B, m, fp32, m, tile=FP32_TILE)
    else:
        call(m, n, n, "N", "N", B, m, s_cols, n, fp32, m, tile=FP32_TILE)
    if routine == "symm":
        got = torch.empty((n, m), device="cuda")
        lib.ssymm_(side.encode(), uplo.encode(), i(m), i(n), one, A.data_ptr(), i(na), B.data_ptr(), i(m), zero, got.data_ptr(), i(m))
    else:
        got = B.clone()
        lib.strmm_(side.encode(), uplo.encode(), b"N", b"N", i(m), i(n), one, A.data_ptr(), i(na), got.data_ptr(), i(m))
    assert lib.zynum_gpu_last_status() == _lib.OK
    torch.cuda.synchronize()
    assert not torch.equal(got, fp32)
    assert (got.double() - ref).norm() <= (fp32.double() - ref).norm()


@pytest.mark.parametrize("side,uplo,trans", [("L", "L", "N"), ("L", "U", "T"), ("R", "U", "N"), ("R", "L", "T")])
def test_trsm_residual(torch_cuda, side, uplo, trans):
    """|op(A) X - B| <= 2 (K + 2) u |op(A)| |X| entrywise, the bound of a solve by
    substitution with products of that bound."""
    torch = torch_cuda
    from zynum_amd import _lib

    lib = _lib.load()
    m, n = (3001, 2600) if side == "L" else (2600, 3001)
    na = 3001
    i = lambda v: C.byref(C.c_int32(v))  # noqa: E731
    A = draw(torch, "uniform", (na, na), 1) / na**0.5
    A.diagonal().copy_(1 + draw(torch, "positive", (na,), 3))
    B = draw(torch, "uniform", (n, m), 2)
    X = B.clone()
    lib.strsm_(side.encode(), uplo.encode(), trans.encode(), b"N", i(m), i(n), C.byref(C.c_float(1.0)), A.data_ptr(), i(na), X.data_ptr(), i(m))
    assert lib.zynum_gpu_last_status() == _lib.OK
    torch.cuda.synchronize()
    T = expanded(torch, A.T, uplo, "tri").double()
    T = T.T if trans == "T" else T
    x, b = X.T.double(), B.T.double()
    resid, mag = ((T @ x - b), T.abs() @ x.abs()) if side == "L" else ((x @ T - b), x.abs() @ T.abs())
    assert bool((resid.abs() <= 2 * (na + 2) * U * mag).all())


@pytest.mark.parametrize("shape", [(4096, 4096, 333), (2048, 2048, 2049), (1024, 1024, 8192)])
@pytest.mark.parametrize("kind", ["4", "16", "64", "256", "constant", "signs", "positive"])
def test_structured_operands_error_at_most_the_fp32_tile(torch_cuda, shape, kind):
    """Few terms per sum (one entry of A in 4 .. 256 not zero), and operands whose
    roundings have one sign: the 2-norm error against 64 bits at most the FP32
    instruction's."""
    torch = torch_cuda
    m, n, k = shape
    A, B = draw(torch, "uniform", (k, m), 1), draw(torch, "uniform", (n, k), 2)
    if kind == "constant":
        A.fill_(WORST)
        B.fill_(WORST)
    elif kind == "signs":
        A, B = torch.sign(A) * WORST, torch.sign(B) * WORST
    elif kind == "positive":
        A, B = A.abs(), B.abs()
    else:
        A *= draw(torch, "positive", (k, m), 3) < 1 / int(kind)
    ref = B.double() @ A.double()
    err = [(product(torch, m, n, k, "N", "N", A, B, tile).double() - ref).norm() for tile in (0, FP32_TILE)]
    assert err[0] <= err[1], [x.item() for x in err]


@pytest.mark.parametrize("shape", [(4096, 4096, 333), (2048, 2048, 2049)])
def test_single_products_are_rounded_once(torch_cuda, shape):
    """The part products that are formed are the product but for 2^-34 of it; a0 b0
    is exact, the others (2^-7 of the product) are summed by themselves in seven
    steps of at most one unit, and one addition to nearest follows."""
    torch = torch_cuda
    m, n, k = shape
    A = torch.zeros((k, m), device="cuda")
    i = torch.arange(m, device="cuda")
    rows = (i * 37 + 5) % k
    B = draw(torch, "normal", (n, k), 4)
    A[rows, i] = draw(torch, "positive", (m,), 3) + 0.5
    exact = B.double()[:, rows] * A[rows, i].double()
    got = product(torch, m, n, k, "N", "N", A, B, 0)
    bound = U * (1 + 7 * 2.0**-6 + 2.0**-9) * exact.abs()
    assert bool(((got.double() - exact).abs() <= bound).all())

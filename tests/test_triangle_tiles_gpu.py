"""The triangular routines on every tile their sizes can select, at ragged
extents: integer operands, so every order of a sum is exact and the comparison
with float64 is for equality.
"""
import ctypes as C
import math

import pytest

pytestmark = pytest.mark.gpu


def i32(v):
    return C.byref(C.c_int32(v))


def trmm_tile(na, across):
    """The FP64 launch's choice among 128x128, 64x128 (along x across the
    triangle) and 64x64, by the same estimate (level3.hip, trmm_dma_us)."""

    def us(along, width, several, one):
        n_along, tiles = -(-na // along), -(-na // along) * -(-across // width)
        flop = 2.0 * along * width / 0.307e6
        mean = flop * ((n_along + 1) / 2 * along + 96.0)
        return max((tiles + 128) / 256 * mean / several, flop * (na + 96.0) / one)

    times = {"128x128": us(128, 128, 0.94, 0.80), "64x128": us(64, 128, 0.915, 0.75), "64x64": us(64, 64, 0.87, 0.71)}
    return min(times, key=times.get)


def integers(torch, rows, cols, ld, seed, hi=3):
    """(cols, ld) device tensor: column j is row j."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randint(-hi, hi + 1, (cols, ld), generator=g, device="cuda").double()


def stored_mask(torch, n, uplo):
    ones = torch.ones((n, n), dtype=torch.bool, device="cuda")
    return torch.tril(ones) if uplo == "L" else torch.triu(ones)


@pytest.mark.parametrize("tile,na,across", [("64x64", 2501, 2301), ("64x128", 3001, 5003), ("128x128", 8191, 8381)])
@pytest.mark.parametrize("side", "LR")
@pytest.mark.parametrize("uplo", "UL")
@pytest.mark.parametrize("trans", "NT")
@pytest.mark.parametrize("diag", "NU")
def test_dtrmm_on_each_tile(torch_cuda, tile, na, across, side, uplo, trans, diag):
    torch = torch_cuda
    from zynum_amd import _lib

    lib = _lib.load()
    assert trmm_tile(na, across) == tile
    m, n = (na, across) if side == "L" else (across, na)
    lda, ldb = na + 2, m + 3
    a, b = integers(torch, na, na, lda, 1), integers(torch, m, n, ldb, 2)
    A, B = a[:, :na].T, b[:, :m].T  # rows x columns
    T = torch.where(stored_mask(torch, na, uplo), A, 0.0)
    if diag == "U":
        T.diagonal().fill_(1.0)
    if trans == "T":
        T = T.T
    want = b.clone()
    want[:, :m] = -2.0 * (T @ B if side == "L" else B @ T).T
    a[:, :na].T[~stored_mask(torch, na, uplo)] = float("nan")  # never read
    lib.dtrmm_(side.encode(), uplo.encode(), trans.encode(), diag.encode(), i32(m), i32(n), C.byref(C.c_double(-2.0)),
               a.data_ptr(), i32(lda), b.data_ptr(), i32(ldb))
    assert lib.zynum_gpu_last_status() == _lib.OK
    torch.cuda.synchronize()
    assert torch.equal(b, want)


# 128x128 tiles: the last 49 of 561 as 64x64 quarters (too shallow to split), and split over K
@pytest.mark.parametrize("n,k", [(4097, 21), (4099, 1031)])
@pytest.mark.parametrize("uplo", "UL")
@pytest.mark.parametrize("trans", "NT")
@pytest.mark.parametrize("rank2", [False, True])
def test_ssyrk_and_ssyr2k_on_large_tiles(torch_cuda, n, k, uplo, trans, rank2):
    torch = torch_cuda
    from zynum_amd import _lib

    lib = _lib.load()
    rows, cols = (n, k) if trans == "N" else (k, n)
    lda, ldb, ldc = rows + 1, rows + 2, n + 3
    a, b, c = integers(torch, rows, cols, lda, 1), integers(torch, rows, cols, ldb, 2), integers(torch, n, n, ldc, 3)
    X, Y = a[:, :rows].T, b[:, :rows].T
    if trans == "T":
        X, Y = X.T, Y.T
    product = X @ (Y if rank2 else X).T.contiguous()
    if rank2:
        product = product + product.T
    want = c.clone()
    mask = stored_mask(torch, n, uplo)
    want[:, :n].T[mask] = (2.0 * product - 3.0 * c[:, :n].T)[mask]
    a, b, c = a.float(), b.float(), c.float()
    two, three = C.byref(C.c_float(2.0)), C.byref(C.c_float(-3.0))
    if rank2:
        lib.ssyr2k_(uplo.encode(), trans.encode(), i32(n), i32(k), two, a.data_ptr(), i32(lda), b.data_ptr(), i32(ldb), three, c.data_ptr(), i32(ldc))
    else:
        lib.ssyrk_(uplo.encode(), trans.encode(), i32(n), i32(k), two, a.data_ptr(), i32(lda), three, c.data_ptr(), i32(ldc))
    assert lib.zynum_gpu_last_status() == _lib.OK
    torch.cuda.synchronize()
    assert torch.equal(c.double(), want)


@pytest.mark.parametrize("single", [False, True])
@pytest.mark.parametrize("side,uplo,trans", [("L", "L", "N"), ("L", "L", "T"), ("R", "U", "N"), ("R", "U", "T")])
@pytest.mark.parametrize("nvec", [1, 100, 257])
def test_trsm_updates_split_over_k(torch_cuda, single, side, uplo, trans, nvec):
    """Few vectors against many unknowns: the updates have few output tiles and are
    split over K.  |op(A) X - B| <= 2 (K + 2) u |op(A)| |X| entrywise."""
    torch = torch_cuda
    from zynum_amd import _lib

    lib = _lib.load()
    dt, scalar, u = (torch.float32, C.c_float, 2.0**-24) if single else (torch.float64, C.c_double, 2.0**-53)
    na = 3347
    m, n = (na, nvec) if side == "L" else (nvec, na)
    g = torch.Generator(device="cuda").manual_seed(nvec)
    A = ((torch.rand((na, na), generator=g, device="cuda", dtype=dt) * 2 - 1) / math.sqrt(na)).contiguous()
    A.diagonal().copy_(1 + torch.rand(na, generator=g, device="cuda", dtype=dt))
    B = torch.rand((n, m), generator=g, device="cuda", dtype=dt) * 2 - 1
    X = B.clone()
    fn = lib.strsm_ if single else lib.dtrsm_
    fn(side.encode(), uplo.encode(), trans.encode(), b"N", i32(m), i32(n), C.byref(scalar(1.0)), A.data_ptr(), i32(na), X.data_ptr(), i32(m))
    assert lib.zynum_gpu_last_status() == _lib.OK
    torch.cuda.synchronize()
    T = torch.where(stored_mask(torch, na, uplo), A.T, torch.zeros((), device="cuda", dtype=dt)).double()
    T = T.T.contiguous() if trans == "T" else T
    x, b = X.T.double(), B.T.double()
    # (the residual's own rounding in 64 bits: as much again)
    resid, mag = (T @ x - b, T.abs() @ x.abs()) if side == "L" else (x @ T - b, x.abs() @ T.abs())
    assert bool((resid.abs() <= (2 * (na + 2) * u + na * 2.0**-53) * mag).all())

"""FP32 products on the bf16 matrix cores at the ends of their range: entries and
sums that leave it, and subnormal entries, which do not.
"""
import pytest

from test_gemm_f32_split_gpu import FP32_TILE, call, draw

pytestmark = pytest.mark.gpu
U = 2.0**-24
# whole 256x256 tiles (16 x 16 of them) and whole 128x128 tiles, k % 16 of 0, 1 and 13
WHOLE = [(4096, 4096, 333), (4096, 4090, 336), (2048, 2048, 2049)]


def product(torch, m, n, k, ta, tb, A, B, tile, alpha=1.0, beta=0.0):
    """C^T; A (k, m) and B (n, k) hold op(A)^T and op(B)^T."""
    a, lda = (A, m) if ta == "N" else (A.T.contiguous(), k)
    b, ldb = (B, k) if tb == "N" else (B.T.contiguous(), n)
    c = torch.ones((n, m), device="cuda")
    call(m, n, k, ta, tb, a, lda, b, ldb, c, m, alpha, beta, tile=tile)
    return c


@pytest.mark.parametrize("shape", WHOLE)
@pytest.mark.parametrize("ta,tb", [("N", "N"), ("T", "T"), ("N", "T")])
@pytest.mark.parametrize("where", ["first", "second", "middle", "last", "every", "b_first", "b_last", "product"])
def test_every_tile_out_of_range_is_the_fp32_tile(torch_cuda, shape, ta, tb, where):
    """Each output tile meets an infinity (or a huge product), at its first stage,
    its last or between: bit for bit the FP32 instruction's results."""
    torch = torch_cuda
    m, n, k = shape
    A, B = draw(torch, "uniform", (k, m), 3), draw(torch, "uniform", (n, k), 4)
    inf = float("inf")
    if where == "product":  # finite sums past 2^80
        A[:, 5::128] = 1.0e19
        B *= 1.0e19
    elif where == "every":
        A[:, 5::128] = float("nan")
    elif where[0] == "b":
        B[7::128, 0 if where == "b_first" else k - 1] = -inf
    else:
        A[{"first": 0, "second": 16, "middle": k // 2, "last": k - 1}[where], 5::128] = inf
    got, want = (product(torch, m, n, k, ta, tb, A, B, t, 1.5, -1.0) for t in (0, FP32_TILE))
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(torch.nan_to_num(got, nan=7.0, posinf=3e38, neginf=-3e38),
                       torch.nan_to_num(want, nan=7.0, posinf=3e38, neginf=-3e38))


@pytest.mark.parametrize("shape", [(4096, 4096, 333), (2048, 2048, 2049), (1024, 1024, 8192)])
@pytest.mark.parametrize("scale", [1e-39, 3e-38, 1e-42])
def test_subnormal_entries_stay_on_the_bf16_cores(torch_cuda, shape, scale):
    """Not the FP32 tile's bits, and at least as exact."""
    torch = torch_cuda
    m, n, k = shape
    A, B = draw(torch, "uniform", (k, m), 3) * scale, draw(torch, "uniform", (n, k), 4) * 1e3
    ref = B.double() @ A.double()
    got, fp32 = (product(torch, m, n, k, "N", "N", A, B, t) for t in (0, FP32_TILE))
    assert not torch.equal(got, fp32)
    assert (got.double() - ref).norm() <= (fp32.double() - ref).norm()
    mag = B.double().abs() @ A.double().abs()
    assert bool(((got.double() - ref).abs() <= 2 * (k + 2) * U * mag + 2.0**-149).all())


@pytest.mark.parametrize("shape", [(1024, 1024, 8192), (1000, 1031, 8177)])
@pytest.mark.parametrize("where", ["first", "last", "b_middle", "product"])
def test_k_ranges_out_of_range(torch_cuda, shape, where):
    """Tiles split over K, some of whose ranges leave the range: the same NaNs and
    infinities as the FP32 instruction, every other entry within its bound."""
    torch = torch_cuda
    m, n, k = shape
    A, B = draw(torch, "uniform", (k, m), 3), draw(torch, "uniform", (n, k), 4)
    if where == "product":
        A[:1000, 700] = 1.0e19
        B[300, :1000] = 1.0e19
    elif where == "b_middle":
        B[300, k // 2] = float("-inf")
    else:
        A[0 if where == "first" else k - 1, 700] = float("nan")
    got, fp32 = (product(torch, m, n, k, "N", "N", A, B, t, 1.5, -1.0) for t in (0, FP32_TILE))
    assert not torch.equal(torch.nan_to_num(got), torch.nan_to_num(fp32))  # (another order of the sums)
    assert torch.equal(torch.isnan(got), torch.isnan(fp32))
    assert torch.equal(torch.isinf(got), torch.isinf(fp32))
    fine = fp32.isfinite()
    A, B = torch.nan_to_num(A, nan=0.0, posinf=0.0, neginf=0.0), torch.nan_to_num(B, nan=0.0, posinf=0.0, neginf=0.0)
    ref = 1.5 * (B.double() @ A.double()) - 1.0
    mag = 1.5 * (B.double().abs() @ A.double().abs()) + 1.0
    assert bool(((got.double() - ref).abs() <= 2 * (k + 2) * U * mag)[fine].all())

"""The loop over a batch sums every element over K in one chain, whatever tile a
problem's size picks: bitwise the forced 64x64 tile's result (random operands,
so another order of a sum would show)."""
import pytest

pytestmark = pytest.mark.gpu

# 64x64; 128x64, 64x128 and 128x128 tiles in one round and in several; edges; many 128x128 tiles (FP32: register-staged)
SHAPES = [(16, 16, 16), (64, 64, 64), (1, 70, 33), (70, 1, 129), (130, 61, 250), (1024, 1024, 72), (61, 8200, 40),
          (8200, 61, 40), (2047, 2049, 65), (3001, 2900, 47), (4096, 4100, 20)]


@pytest.mark.parametrize("dtype_name", ["float64", "float32"])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("pad", [0, 1])
def test_loop_walks_one_chain(torch_cuda, dtype_name, ta, tb, pad):
    torch = torch_cuda
    from zynum_amd import _lib, blas, grouped

    b = grouped.Batch(torch, SHAPES, getattr(torch, dtype_name), seed=9, transa=ta, transb=tb, alpha=0.75, beta=-0.25, pad=pad)
    b.loop()
    torch.cuda.synchronize()
    got = b.C.clone()
    b.reset_c()
    for (m, n, k), p in zip(SHAPES, b.problems):
        _lib.check(blas.gemm_request(ta, tb, m, n, k, 0.75, p.a, p.lda, p.b, p.ldb, -0.25, p.c, p.ldc, b.scalar, tile=1), "gemm")
    torch.cuda.synchronize()
    for i, (m, n, k) in enumerate(SHAPES):
        end = b.offs[2][i] + b.lds[i][2] * n
        assert torch.equal(got[b.offs[2][i]: end], b.C[b.offs[2][i]: end]), (m, n, k)

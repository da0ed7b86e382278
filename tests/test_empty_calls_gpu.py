"""A call on an empty result returns at once: it does not wait for work queued on
the null stream.  The writer keeps that stream busy for tens of milliseconds,
and is still at work when every empty call has returned."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


def empty_calls(lib, _lib, blas, p):
    """Every symbol with one extent zero, on the operand p."""
    i = lambda v: C.byref(C.c_int32(v))  # noqa: E731
    n, z, ld = i(64), i(0), i(64)
    for t, scalar in (("s", C.c_float), ("d", C.c_double)):
        one = C.byref(scalar(1.0))
        fn = lambda name: getattr(lib, t + name + "_")  # noqa: E731
        fn("gemm")(b"N", b"N", z, n, n, one, p, ld, p, ld, one, p, ld)
        fn("syrk")(b"L", b"N", z, n, one, p, ld, one, p, ld)
        fn("syr2k")(b"L", b"N", z, n, one, p, ld, p, ld, one, p, ld)
        fn("symm")(b"L", b"L", n, z, one, p, ld, p, ld, one, p, ld)
        fn("trmm")(b"L", b"L", b"N", b"N", n, z, one, p, ld, p, ld)
        fn("trsm")(b"L", b"L", b"N", b"N", n, z, one, p, ld, p, ld)
    pair = C.cast((C.c_double * 2)(1.0, 0.0), C.c_void_p)
    lib.zgemm_(b"N", b"N", n, z, n, pair, p, ld, p, ld, pair, p, ld)
    lib.cgemm_(b"N", b"N", z, n, n, pair, p, ld, p, ld, pair, p, ld)
    for scalar in (_lib.F32, _lib.F64, _lib.C64):
        _lib.check(blas.gemm_request("N", "N", 64, 0, 64, 1.0, p, 64, p, 64, 1.0, p, 64, scalar), "gemm")
    _lib.check(lib.zynum_gpu_dtrsm(b"L", b"L", b"N", b"N", 64, 0, 1.0, p, 64, p, 64, None, 0, 0, 0), "dtrsm")
    _lib.check(lib.zynum_gpu_dsyrk(b"L", b"N", 0, 64, 1.0, p, 64, 1.0, p, 64, None, 0, 0, 0), "dsyrk")
    _lib.check(lib.zynum_gpu_dsymm(b"L", b"L", 0, 64, 1.0, p, 64, p, 64, 1.0, p, 64, None, 0), "dsymm")
    _lib.check(lib.zynum_gpu_dtrmm(b"L", b"L", b"N", b"N", 0, 64, 1.0, p, 64, p, 64, None, 0), "dtrmm")
    _lib.check(lib.zynum_gpu_dsyr2k(b"L", b"N", 0, 64, 1.0, p, 64, p, 64, 1.0, p, 64, None, 0), "dsyr2k")


def test_empty_calls_do_not_wait(torch_cuda):
    torch = torch_cuda
    from zynum_amd import _lib, blas

    lib = _lib.load()
    big = torch.zeros((8192, 8192), dtype=torch.float64, device="cuda")
    empty_calls(lib, _lib, blas, big.data_ptr())  # first uses (device probe) behind us
    torch.cuda.synchronize()
    done = torch.cuda.Event()
    with torch.cuda.stream(torch.cuda.default_stream()):
        for _ in range(400):  # at least 0.13 ms each (1 GiB at 8 TB/s)
            big.add_(1)
        done.record()
    empty_calls(lib, _lib, blas, big.data_ptr())
    still_busy = not done.query()
    torch.cuda.synchronize()
    assert still_busy
    assert bool((big == 400).all())

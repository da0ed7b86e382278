"""An asynchronous call that needs scratch for partial sums waits for its stream,
which a stream under capture refuses: the call says so instead of reporting
success for work that will not run."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu
RELAXED = 2  # hipStreamCaptureModeRelaxed


@pytest.fixture()
def hip_stream():
    hip = C.CDLL("libamdhip64.so")
    s = C.c_void_p()
    assert hip.hipStreamCreateWithFlags(C.byref(s), 1) == 0
    yield hip, s
    assert hip.hipStreamDestroy(s) == 0
    hip.hipGetLastError()


@pytest.mark.parametrize("dtype_name", ["float64", "float32", "complex128"])
def test_scratch_under_capture_is_an_error(torch_cuda, hip_stream, dtype_name):
    torch = torch_cuda
    from zynum_amd import _lib, blas

    hip, s = hip_stream
    scalar = {"float64": _lib.F64, "float32": _lib.F32, "complex128": _lib.C64}[dtype_name]
    m, k = 64, 4096  # one 64 x 64 tile (complex: two), split over K
    dt = getattr(torch, dtype_name)
    a = torch.ones((k, m), dtype=dt, device="cuda")
    c = torch.zeros((m, m), dtype=dt, device="cuda")

    def call(stream):
        return blas.gemm_request("N", "T", m, m, k, 1.0, a.data_ptr(), m, a.data_ptr(), m, 0.0, c.data_ptr(), m,
                                 scalar, stream=stream, flags=_lib.FLAG_ASYNC)

    _lib.check(call(s.value), "eager")
    torch.cuda.synchronize()
    assert bool((c == k).all())
    assert hip.hipStreamBeginCapture(s, RELAXED) == 0
    status = call(s.value)
    graph = C.c_void_p()
    ended = hip.hipStreamEndCapture(s, C.byref(graph))
    hip.hipGetLastError()
    if graph.value:
        hip.hipGraphDestroy(graph)
    assert ended != 0  # the wait ended the capture
    assert status == _lib.ERR_LAUNCH
    # no error is left behind for the next call
    c.zero_()
    torch.cuda.synchronize()
    _lib.check(call(None), "after the capture")
    torch.cuda.synchronize()
    assert bool((c == k).all())

"""A complex call that waits for its own work does not hold up other threads'
calls meanwhile: thread A's synchronous product of split tiles sits behind long
work on its stream; an asynchronous call from this thread on another stream
returns while that work still runs."""
import threading

import pytest

pytestmark = pytest.mark.gpu


def test_synchronous_split_product_waits_outside_the_workspace_lock(torch_cuda):
    torch = torch_cuda
    from zynum_amd import _lib, blas

    m, k = 64, 2048  # two 64 x 64 real tiles, split over K
    a = torch.ones((k, m), dtype=torch.complex128, device="cuda")
    c = torch.zeros((2, m, m), dtype=torch.complex128, device="cuda")
    big = torch.zeros((8192, 8192), dtype=torch.float64, device="cuda")
    sa, sb = torch.cuda.Stream(), torch.cuda.Stream()

    def product(i, stream, flags, size=k):
        return blas.gemm_request("N", "T", m, m, size, 1.0, a.data_ptr(), m, a.data_ptr(), m, 0.0, c[i].data_ptr(), m,
                                 _lib.C64, stream=stream.cuda_stream, flags=flags)

    _lib.check(product(0, sa, 0), "warm")
    _lib.check(product(1, sb, _lib.FLAG_ASYNC, 64), "warm")
    c.zero_()
    torch.cuda.synchronize()
    done = torch.cuda.Event()
    with torch.cuda.stream(sa):
        for _ in range(1000):  # at least 0.13 ms each
            big.add_(1)
        done.record()
    started, status = threading.Event(), []

    def other():
        started.set()
        status.append(product(0, sa, 0))  # waits for sa

    t = threading.Thread(target=other)
    t.start()
    started.wait()
    t.join(0.02)  # it is inside its wait by now
    assert t.is_alive()
    status.append(product(1, sb, _lib.FLAG_ASYNC, 64))
    still_busy = not done.query()
    t.join()
    torch.cuda.synchronize()
    assert status == [_lib.OK, _lib.OK]
    assert still_busy
    assert bool((c[0] == k).all()) and bool((c[1] == 64).all())

"""Device-pointer factorizations do not wait for their stream.

The first look-ahead call on a stream chooses a pair of the library's own
streams by timing; it may not wait for what is queued on the caller's stream,
which can depend on something that the calling thread does later.
"""
import time

import pytest

import oracle as O

pytestmark = pytest.mark.gpu

N = 2304


@pytest.fixture(scope="module")
def G():
    import torch
    assert torch.cuda.is_available()
    import atlas_gpu
    return atlas_gpu


def matrix(torch):
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    a = torch.rand((N, N), generator=g, device="cuda", dtype=torch.float64) * 2 - 1
    return a + a.t() + 4 * N * torch.eye(N, device="cuda", dtype=torch.float64)


@pytest.mark.parametrize("routine", ["dpotrf", "dgetrf"])
def test_first_call_on_a_busy_stream_returns(G, routine):
    import torch

    def call(a, n):
        if routine == "dpotrf":
            G.dpotrf(O.Lower, n, a, N, info)
        else:
            G.dgetrf(n, n, a, N, piv, info)

    a0 = matrix(torch)
    info = torch.zeros(1, dtype=torch.int32, device="cuda")
    piv = torch.zeros(N, dtype=torch.int32, device="cuda")
    a = a0.clone()
    call(a, N)  # code and the library's streams are loaded
    want = a.clone()
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        b = a0.clone()
        call(b, 1920)  # workspace, without the look-ahead
        b.copy_(a0)
        torch.cuda.synchronize()
        # the stream busy for about a second
        t0 = torch.cuda.Event(enable_timing=True)
        t1 = torch.cuda.Event(enable_timing=True)
        t0.record()
        torch.cuda._sleep(10 ** 6)
        t1.record()
        torch.cuda.synchronize()
        torch.cuda._sleep(int(10 ** 6 * 1000.0 / t0.elapsed_time(t1)))
        busy = torch.cuda.Event()
        busy.record()
        before = time.monotonic()
        call(b, N)
        took = time.monotonic() - before
        assert not busy.query(), "the call waited for its stream"
        assert took < 0.5
    torch.cuda.synchronize()
    assert int(info.item()) == 0
    with torch.cuda.stream(s):
        G.check_stream()
    assert torch.equal(b, want)

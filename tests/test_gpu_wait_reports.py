"""Waits that give up inside a factorization are reported to its caller.

The look-ahead LU and Cholesky queue their triangular solves on streams of
the library's own; a wait that gives up there (forced from the host as in
test_gpu_failure.py: the bound is one poll) has to reach the failure word of
the stream that the caller passed, and the info word, since nobody asks the
library's streams.
"""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import torch
    assert torch.cuda.is_available()
    import atlas_gpu
    assert atlas_gpu.lib().atlg_init() == 0
    yield atlas_gpu
    atlas_gpu.set_wait_limit(0)


def spd(n):
    rng = np.random.default_rng(n)
    a = rng.uniform(-1, 1, (n, n))
    return np.asfortranarray(a + a.T + 4 * n * np.eye(n))


# 1100: the recursion on the caller's stream (its 384-column blocks take one-launch
# solves; below order 769 there are none); 2304: the look-ahead's streams
@pytest.mark.parametrize("n", [1100, 2304])
@pytest.mark.parametrize("uplo", [O.Lower, O.Upper])
def test_potrf_failed_solve_reported(G, uplo, n):
    import torch
    a0 = spd(n)
    info = torch.zeros(1, dtype=torch.int32, device="cuda")
    st = torch.cuda.Stream()
    G.set_wait_limit(1)
    try:
        with torch.cuda.stream(st):
            da = G.from_fortran(a0)
            G.dpotrf(uplo, n, da, n, info)
            assert G.stream_status() == G.FAIL_TRSV
            assert int(info.item()) == -2 ** 31
            assert G.stream_status() == 0
        with pytest.raises(G.AtlgWaitError) as ei:
            G.clapack_dpotrf(G.ColMajor, uplo, n, a0.copy(order="F"), n)
        assert ei.value.bits == G.FAIL_TRSV
    finally:
        G.set_wait_limit(0)
    with torch.cuda.stream(st):
        da = G.from_fortran(a0)
        G.dpotrf(uplo, n, da, n, info, check=True)
        assert int(info.item()) == 0
        assert O.llt_resid(uplo, n, a0, G.to_fortran(da)) <= 16


def test_getrf_failed_solve_reported(G):
    import torch
    n = 2304
    a0 = O.gegen(n, n, 2304)
    ipiv = torch.zeros(n, dtype=torch.int32, device="cuda")
    info = torch.zeros(1, dtype=torch.int32, device="cuda")
    G.set_wait_limit(1)
    try:
        da = G.from_fortran(a0)
        G.dgetrf(n, n, da, n, ipiv, info)
        assert G.stream_status() & G.FAIL_TRSV
        assert int(info.item()) == -2 ** 31
    finally:
        G.set_wait_limit(0)
    da = G.from_fortran(a0)
    G.dgetrf(n, n, da, n, ipiv, info, check=True)
    assert int(info.item()) == 0
    assert O.lu_resid(n, n, a0, G.to_fortran(da), ipiv.cpu().numpy()) <= 100


def test_noalloc_failure_stays_with_its_stream(G):
    import torch
    n, k = 1500, 40
    rng = np.random.default_rng(4)
    a = G.from_fortran(np.asfortranarray(np.tril(rng.uniform(-1, 1, (n, n))) / n + 2 * np.eye(n)))
    b = G.from_fortran(np.asfortranarray(rng.uniform(-1, 1, (n, k))))
    s = [torch.cuda.Stream() for _ in range(3)]
    torch.cuda.synchronize()

    def solve(stream):
        with torch.cuda.stream(stream):
            x = b.clone()
            G.dtrsm_noalloc(G.Left, G.Lower, G.NoTrans, G.NonUnit, n, k, 1.0, a, n, x, n)
        torch.cuda.synchronize()  # (such solves on different streams may not overlap)
        return x

    def status(stream):
        with torch.cuda.stream(stream):
            return G.stream_status()

    want = solve(s[1])
    G.set_wait_limit(1)
    try:
        solve(s[0])
    finally:
        G.set_wait_limit(0)
    assert status(s[1]) == 0  # a stream with such solves of its own
    assert status(s[2]) == 0  # and one without
    assert torch.equal(solve(s[1]), want) and status(s[1]) == 0
    assert status(s[0]) == G.FAIL_TRSV
    assert status(s[0]) == 0
    assert torch.equal(solve(s[0]), want) and status(s[0]) == 0

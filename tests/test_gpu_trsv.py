"""Triangular solves with few right-hand sides (one launch up to order 2048,
1024 or 512, halves above; one right-hand side above 4096 by the sync-free launch):
orders around the 64-row blocks and the 128-row inverses, right-hand sides
around the 16-column groups, every side, triangle, transpose and diagonal.

Accepted residual: with op(A)'s diagonal in [1, 2] and the sum of a row's
other entries at most 1/2 in magnitude, a solve through inverted blocks errs
by at most a few sums of n terms: 4 n eps (|op(A)| max|x| + max|alpha b|).
"""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -53


@pytest.fixture(scope="module")
def G():
    import torch
    assert torch.cuda.is_available()
    import atlas_gpu
    return atlas_gpu


def system(n, k, seed):
    rng = np.random.default_rng(seed)
    a = rng.uniform(-0.5, 0.5, (n + 1, n)) / n
    a[np.arange(n), np.arange(n)] = rng.uniform(1, 2, n)
    return np.asfortranarray(a), np.asfortranarray(rng.uniform(-1, 1, (n + 2, k)))


def op(a, n, uplo, trans, diag):
    t = np.tril(a[:n]) if uplo == O.Lower else np.triu(a[:n])
    if diag == O.Unit:
        t[np.arange(n), np.arange(n)] = 1
    return t.T if trans == O.Trans else t


def close(n, t, x, b, alpha):
    r = np.abs(t @ x - alpha * b).max()
    return r <= 4 * n * EPS * (np.abs(t).sum(1).max() * np.abs(x).max() + np.abs(alpha * b).max())


@pytest.mark.parametrize("uplo", [O.Lower, O.Upper])
@pytest.mark.parametrize("trans", [O.NoTrans, O.Trans])
@pytest.mark.parametrize("n,k", [(129, 1), (191, 16), (192, 17), (193, 3), (256, 128), (257, 129),
                                 (500, 5), (1000, 33), (2047, 2), (2048, 1), (2049, 1), (4097, 1),
                                 (1024, 385), (1025, 400), (2049, 384), (300, 3073), (200, 4097)])
def test_few_rhs(G, uplo, trans, n, k):
    a, b = system(n, k, n + k)
    for diag, alpha in ((O.NonUnit, 1.0), (O.Unit, -0.7)):
        da, db = G.from_fortran(a), G.from_fortran(b)
        G.dtrsm(G.Left, uplo, trans, diag, n, k, alpha, da, n + 1, db, n + 2, check=True)
        x = G.to_fortran(db)
        assert np.array_equal(x[n:], b[n:])
        assert close(n, op(a, n, uplo, trans, diag), x[:n], b[:n], alpha)


@pytest.mark.parametrize("uplo", [O.Lower, O.Upper])
@pytest.mark.parametrize("trans", [O.NoTrans, O.Trans])
@pytest.mark.parametrize("n,k", [(129, 1), (192, 17), (500, 5), (1000, 200), (2049, 3)])
def test_right(G, uplo, trans, n, k):
    # X op(A) = alpha B is op(A)^T X^T = alpha B^T
    a, b = system(n, k, n + k)
    b = np.asfortranarray(b.T)
    for diag, alpha in ((O.NonUnit, 1.0), (O.Unit, -0.7)):
        da, db = G.from_fortran(a), G.from_fortran(b)
        G.dtrsm(G.Right, uplo, trans, diag, k, n, alpha, da, n + 1, db, k, check=True)
        x = G.to_fortran(db)
        assert np.array_equal(x[:, n:], b[:, n:])
        assert close(n, op(a, n, uplo, trans, diag).T, x[:, :n].T, b[:, :n].T, alpha)


def test_not_finite(G):
    # a right-hand side's infinities and NaN stay in its column, from its row on
    n, k = 300, 18
    a, b = system(n, k, 5)
    b[70, 3] = np.inf
    b[200, 17] = np.nan
    da, db = G.from_fortran(a), G.from_fortran(b)
    G.dtrsm(G.Left, G.Lower, G.NoTrans, G.NonUnit, n, k, 1.0, da, n + 1, db, n + 2, check=True)
    x = G.to_fortran(db)[:n]
    rest = [c for c in range(k) if c not in (3, 17)]
    assert close(n, op(a, n, O.Lower, O.NoTrans, O.NonUnit), x[:, rest], b[:n, rest], 1.0)
    assert not np.isfinite(x[70:, 3]).any() and not np.isfinite(x[200:, 17]).any()
    assert np.isfinite(x[:64, 3]).all() and np.isfinite(x[:128, 17]).all()


def test_captured_without_workspace(G):
    # on a stream that has only seen a wide solve, a captured narrow one
    # allocates nothing; the eager one between the replays may
    import torch
    n, k = 500, 3
    a, b = system(n, k, 9)
    wide = np.asfortranarray(np.ones((n, 200)))
    t = op(a, n, O.Lower, O.NoTrans, O.NonUnit)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        da, b0, dw = G.from_fortran(a), G.from_fortran(b), G.from_fortran(wide)
        db = b0.clone()
        G.dtrsm(G.Left, G.Lower, G.NoTrans, G.NonUnit, n, 200, 1.0, da, n + 1, dw, n)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        db.copy_(b0)
        G.dtrsm(G.Left, G.Lower, G.NoTrans, G.NonUnit, n, k, 1.0, da, n + 1, db, n + 2)
    for _ in range(3):
        db.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert close(n, t, G.to_fortran(db)[:n], b[:n], 1.0)
        with torch.cuda.stream(s):
            db.copy_(b0)
            G.dtrsm(G.Left, G.Lower, G.NoTrans, G.NonUnit, n, k, 1.0, da, n + 1, db, n + 2)
        torch.cuda.synchronize()
        assert close(n, t, G.to_fortran(db)[:n], b[:n], 1.0)


def test_noalloc_same_bits_and_failure(G):
    # the allocation-free entry takes the same launches in its own memory, and
    # a wait that runs over is reported the same way
    n, k = 1500, 40
    a, b = system(n, k, 11)
    da, x, y = G.from_fortran(a), G.from_fortran(b), G.from_fortran(b)
    G.dtrsm(G.Left, G.Lower, G.NoTrans, G.NonUnit, n, k, 1.0, da, n + 1, x, n + 2, check=True)
    G.dtrsm_noalloc(G.Left, G.Lower, G.NoTrans, G.NonUnit, n, k, 1.0, da, n + 1, y, n + 2)
    G.check_stream()
    assert np.array_equal(G.to_fortran(x), G.to_fortran(y))
    G.set_wait_limit(1)
    try:
        G.dtrsm_noalloc(G.Left, G.Lower, G.NoTrans, G.NonUnit, n, k, 1.0, da, n + 1, y, n + 2)
        with pytest.raises(G.AtlgWaitError) as e:
            G.check_stream()
        assert e.value.bits & G.FAIL_TRSV
    finally:
        G.set_wait_limit(0)
    y.copy_(G.from_fortran(b))
    G.dtrsm_noalloc(G.Left, G.Lower, G.NoTrans, G.NonUnit, n, k, 1.0, da, n + 1, y, n + 2)
    G.check_stream()
    assert np.array_equal(G.to_fortran(x), G.to_fortran(y))

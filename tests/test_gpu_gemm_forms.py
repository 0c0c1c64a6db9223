"""DGEMM/SGEMM at the edges of the tile forms the dispatch chooses between
(128x128 tiles, 64x64 and 32x32 waves, the in-place 128-wide sides), against
the oracle's refgemm (FP64) with gemmtst's element bound, or an FP64 product
(FP32) with the bound 2 K eps32 sum|a||b| of any order of summation.
"""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

TR = [O.NoTrans, O.Trans]


@pytest.fixture(scope="module")
def G():
    import torch
    assert torch.cuda.is_available()
    import atlas_gpu
    return atlas_gpu


def operands(ta, tb, m, n, k, gap):
    sa = (m, k) if ta == O.NoTrans else (k, m)
    sb = (k, n) if tb == O.NoTrans else (n, k)
    a = O.gegen(sa[0], sa[1], m * k + 7, lda=sa[0] + gap)
    b = O.gegen(sb[0], sb[1], n * k + 3, lda=sb[0] + gap)
    return a, b, O.gegen(m, n, m * n + 1, lda=m + gap)


# tile edges of 32 and 64, chunks of 16 k with every remainder class, K
# shorter than the four slices of the 32x32 form
SMALL = [(1, 1, 1), (31, 33, 15), (32, 32, 16), (33, 31, 17), (63, 65, 31), (64, 64, 64),
         (65, 63, 66), (100, 7, 130), (5, 129, 200)]
# 64x64 waves (one round of tiles with a short K), 128x128 tiles with even,
# odd and register-path K
LARGE = [(1023, 1025, 70), (1023, 1025, 21), (2050, 2047, 33), (2048, 2050, 64)]


@pytest.mark.parametrize("ta", TR)
@pytest.mark.parametrize("tb", TR)
@pytest.mark.parametrize("gap", [0, 3])
@pytest.mark.parametrize("m,n,k", SMALL + LARGE)
def test_dgemm(G, ta, tb, m, n, k, gap):
    alpha, beta = (0.7, 1.3) if gap else (1.0, 0.0)
    a, b, c0 = operands(ta, tb, m, n, k, gap)
    if beta == 0.0:
        c0[:m] = np.nan  # never read
    da, db, dc = G.from_fortran(a), G.from_fortran(b), G.from_fortran(c0)
    G.dgemm(ta, tb, m, n, k, alpha, da, a.shape[0], db, b.shape[0], beta, dc, c0.shape[0])
    c = G.to_fortran(dc)
    ref = c0.copy(order="F")
    O.lib().orc_refgemm(ta, tb, m, n, k, alpha, O._p(a), a.shape[0], O._p(b), b.shape[0], beta,
                        O._p(ref), c0.shape[0])
    assert O.gechkgap(c, m) == 0
    nbad, worst = O.gemm_elem_check(m, n, k, alpha, beta, c, ref)
    assert nbad == 0, worst


@pytest.mark.parametrize("ta", TR)
@pytest.mark.parametrize("tb", TR)
@pytest.mark.parametrize("m,n,k", [(33, 31, 17), (65, 63, 66), (1023, 1025, 21), (2050, 2047, 33)])
def test_sgemm(G, ta, tb, m, n, k):
    import torch
    a, b, _ = operands(ta, tb, m, n, k, 1)
    da, db = (torch.from_numpy(np.ascontiguousarray(x.T)).float().cuda() for x in (a, b))
    dc = torch.full((n, m), float("nan"), device="cuda")
    G.sgemm(ta, tb, m, n, k, 1.0, da, a.shape[0], db, b.shape[0], 0.0, dc, m)
    sa, sb = da.double().cpu().numpy().T, db.double().cpu().numpy().T
    sa = sa[:m, :k] if ta == O.NoTrans else sa[:k, :m].T
    sb = sb[:k, :n] if tb == O.NoTrans else sb[:n, :k].T
    err = np.abs(dc.double().cpu().numpy().T - sa @ sb)
    assert np.all(err <= 2 * k * 2.0 ** -24 * (np.abs(sa) @ np.abs(sb)))


@pytest.mark.parametrize("uplo", [O.Upper, O.Lower])
@pytest.mark.parametrize("trans", TR)
@pytest.mark.parametrize("n,k", [(33, 17), (97, 40), (700, 50), (1100, 96)])
def test_syrk_triangles(G, uplo, trans, n, k):
    a = O.gegen(*((n, k) if trans == O.NoTrans else (k, n)), n * k)
    c0 = O.gegen(n, n, n + 5)
    dc = G.from_fortran(c0)
    G.dsyrk(uplo, trans, n, k, -1.0, G.from_fortran(a), a.shape[0], 1.0, dc, n)
    c, ref = G.to_fortran(dc), c0.copy(order="F")
    O.refsyrk(uplo, trans, n, k, -1.0, a, 1.0, ref)
    nbad, worst = O.gemm_elem_check(n, n, k, -1.0, 1.0, c, ref)
    assert nbad == 0, worst
    other = np.tril_indices(n, -1) if uplo == O.Upper else np.triu_indices(n, 1)
    assert np.array_equal(c[other], c0[other])


@pytest.mark.parametrize("side", [O.Left, O.Right])
@pytest.mark.parametrize("ta", TR)
@pytest.mark.parametrize("n,r", [(1, 33), (31, 1), (100, 65), (128, 31), (127, 2049)])
def test_in_place_side(G, side, ta, n, r):
    # TRSM of one diagonal block: the whole solve is the in-place product
    a = np.asfortranarray(O.gegen(n, n, n * 31) / max(1, n))
    a[np.arange(n), np.arange(n)] = 1.5 + 0.25 * np.cos(np.arange(n))
    b0 = O.gegen(*((n, r) if side == O.Left else (r, n)), n * r)
    db = G.from_fortran(b0)
    G.dtrsm(side, O.Lower, ta, O.NonUnit, b0.shape[0], b0.shape[1], 0.7, G.from_fortran(a), n, db,
            b0.shape[0])
    b, ref = G.to_fortran(db), b0.copy(order="F")
    O.reftrsm(side, O.Lower, ta, O.NonUnit, b0.shape[0], b0.shape[1], 0.7, a, ref)
    # a well-conditioned triangle (off-diagonal row sums below 1.25): two
    # orders of summation and the inverse's rounding, n eps each, scaled by
    # ||X|| times a condition of at most 6
    assert np.abs(b - ref).max() <= 32 * (n + 4) * np.finfo(float).eps * np.abs(ref).max()

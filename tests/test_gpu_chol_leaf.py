"""The Cholesky leaf (one diagonal block of order at most 128, with its
inverse) against the oracle: orders around its 4-column blocks and 16x16
tiles, both triangles, failing minors, tiny and huge scales.  Accepted:
ATLAS's llttst residual (16) and the oracle's info; two blocks (order above
128) exercise the leaf's inverse through the panel solve.
"""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

UPLO = [O.Lower, O.Upper]


@pytest.fixture(scope="module")
def G():
    import torch
    assert torch.cuda.is_available()
    import atlas_gpu
    return atlas_gpu


def potrf(G, uplo, a):
    import torch
    d = G.from_fortran(a)
    info = torch.zeros(1, dtype=torch.int32, device="cuda")
    G.dpotrf(uplo, a.shape[1], d, a.shape[0], info)
    return G.to_fortran(d), int(info.item())


def other(uplo, n):
    return np.triu_indices(n, 1) if uplo == O.Lower else np.tril_indices(n, -1)


@pytest.mark.parametrize("uplo", UPLO)
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 15, 16, 17, 31, 33, 63, 64, 65, 100, 127, 128, 129,
                               144, 255])
def test_leaf(G, uplo, n):
    s = O.lltgen(uplo, n, n * 1029 + n, lda=n + 3)
    f, info = potrf(G, uplo, s)
    assert info == 0
    assert O.llt_resid(uplo, n, s, f) <= 16
    assert np.array_equal(f[:n][other(uplo, n)], s[:n][other(uplo, n)])
    assert np.array_equal(f[n:], s[n:])


@pytest.mark.parametrize("uplo", UPLO)
@pytest.mark.parametrize("scale", [2.0 ** -1060, 2.0 ** -1000, 2.0 ** 900])
def test_leaf_scales(G, uplo, scale):
    # a power of two: the factor scales by its root exactly while nothing is
    # subnormal; subnormal entries keep an absolute error of their spacing
    n = 40
    s = O.lltgen(uplo, n, 77)
    f1, _ = potrf(G, uplo, s)
    f, info = potrf(G, uplo, np.asfortranarray(s * scale))
    assert info == 0
    tri = np.tril_indices(n) if uplo == O.Lower else np.triu_indices(n)
    root = np.sqrt(scale)
    eps = np.finfo(float).eps
    tol = 64 * n * (eps + 5e-324 / scale) * np.abs(f1[tri]).max()
    assert np.abs(f[tri] / root - f1[tri]).max() <= tol


@pytest.mark.parametrize("uplo", UPLO)
@pytest.mark.parametrize("n,bad", [(1, 0), (20, 0), (20, 3), (20, 4), (64, 15), (64, 16), (128, 97),
                                   (128, 127), (150, 149)])
@pytest.mark.parametrize("value", [0.0, -1.0, np.nan])
def test_leaf_failing_minor(G, uplo, n, bad, value):
    s = O.lltgen(uplo, n, n * 7 + 1)
    ref = s.copy(order="F")
    O.potf2(uplo, ref)
    # the pivot of column `bad` becomes `value`: its diagonal less what the
    # factor's column says is subtracted from it
    col = ref[bad, :bad] if uplo == O.Lower else ref[:bad, bad]
    s[bad, bad] = value + float(col @ col) - (1.0 if value == 0.0 else 0.0)
    f, info = potrf(G, uplo, s)
    assert info == bad + 1
    assert np.array_equal(f[other(uplo, n)], s[other(uplo, n)])


@pytest.mark.parametrize("uplo", UPLO)
@pytest.mark.parametrize("n, q", [(5, 1), (20, 2), (20, 7), (64, 17), (64, 63), (128, 98),
                                  (150, 131), (400, 390), (2304, 1301)])
def test_leading_factor_of_a_failing_matrix(G, uplo, n, q):
    # the leading minor of order info - 1 has its factor in place
    s = O.lltgen(uplo, n, n * 7 + q)
    s[q, q] = -1.0
    f, info = potrf(G, uplo, s)
    assert info == q + 1
    lead = np.asfortranarray(s[:q, :q])
    assert O.llt_resid(uplo, q, lead, np.asfortranarray(f[:q, :q])) <= 16
    assert np.array_equal(f[other(uplo, n)], s[other(uplo, n)])

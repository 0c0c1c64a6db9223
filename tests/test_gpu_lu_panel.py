"""The LU leaf panel of one XCD (csrc/lu_panel.hpp) against the oracle's getf2.

Sizes at its edges: waves (64 rows), the single-workgroup panel (512 rows),
several workgroups up to its tallest (8192 rows) and one row past it (the
other panel kernel), one column to a full leaf, panels wider than tall.
Accepted: the oracle's pivots, and ATLAS's LU residual (lutst: 100 in units
of ||A|| eps max(M, N)).
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
    return atlas_gpu


def factor(G, a):
    import torch
    m, n = a.shape
    d = G.from_fortran(a)
    piv = torch.full((min(m, n),), -7, dtype=torch.int32, device="cuda")
    info = torch.zeros(1, dtype=torch.int32, device="cuda")
    G.dgetrf(m, n, d, m, piv, info, check=True)
    return G.to_fortran(d), piv.cpu().numpy(), int(info.item())


def oracle(a):
    ref = a.copy(order="F")
    piv, info = O.getf2(ref)
    return ref, piv, info


@pytest.mark.parametrize("n", [1, 2, 5, 31, 32])
@pytest.mark.parametrize("m", [1, 3, 31, 33, 63, 64, 65, 511, 512, 513, 1025, 4096, 4097, 8191,
                               8192, 8193])
def test_panel(G, m, n):
    a = O.gegen(m, n, m * n + 17 * m)
    lu, piv, info = factor(G, a)
    _, rpiv, rinfo = oracle(a)
    assert np.array_equal(piv, rpiv) and info == rinfo
    assert O.lu_resid(m, n, a, lu, piv) <= 100


@pytest.mark.parametrize("m", [40, 512, 700])
def test_panel_ties_and_zero_columns(G, m):
    # equal magnitudes within a lane, a wave, a workgroup and across them:
    # the first row wins; a zero column is reported and passed over
    n = 32
    a = np.zeros((m, n), order="F")
    for j in range(n):
        a[j::7, j] = 1.0 if j % 2 else -1.0
    a += np.eye(m, n) * 1.0
    a[:, 11] = 0.0
    lu, piv, info = factor(G, a)
    ref, rpiv, rinfo = oracle(a)
    assert np.array_equal(piv, rpiv) and info == rinfo
    # entries of size O(1): each is a sum of at most n products, so the two
    # orders of summation differ by at most n eps max|L| max|U| per entry
    tol = 2 * n * np.finfo(float).eps * max(1.0, np.abs(ref).max()) ** 2
    assert np.abs(lu - ref).max() <= tol


@pytest.mark.parametrize("m", [100, 513])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_panel_nonfinite(G, m, bad):
    # one infinity or NaN spreads exactly as in the textbook elimination: a
    # NaN is never chosen while a number is left, finished rows stay finite
    n = 32
    rng = np.random.default_rng(m)
    a = np.asfortranarray(rng.uniform(-1, 1, (m, n)))
    a[m // 3, n // 2] = bad
    lu, piv, _ = factor(G, a)
    ref, rpiv, _ = oracle(a)
    assert np.array_equal(piv, rpiv)
    fin = np.isfinite(ref)
    assert np.array_equal(fin, np.isfinite(lu))
    tol = 2 * n * np.finfo(float).eps * max(1.0, np.abs(ref[fin]).max()) ** 2
    assert np.abs(lu[fin] - ref[fin]).max() <= tol


def test_panel_subnormal_pivots(G):
    # pivots below the smallest normal number divide instead of multiplying
    # by a reciprocal that would overflow: multipliers of at most one
    m, n = 200, 4
    rng = np.random.default_rng(3)
    a = np.asfortranarray(rng.uniform(-1, 1, (m, n)))
    a[:, 0] *= 2.0 ** -1040
    lu, piv, info = factor(G, a)
    p0 = int(np.argmax(np.abs(a[:, 0])))
    assert info == 0 and piv[0] == p0
    b = a[:, 0].copy()
    b[[0, p0]] = b[[p0, 0]]
    exact = (b[1:] * 2.0 ** 500) / (b[0] * 2.0 ** 500)
    # column 0 of L in its final row order
    for j in range(1, n):
        exact[[j - 1, piv[j] - 1]] = exact[[piv[j] - 1, j - 1]]
    assert np.abs(lu[1:, 0] - exact).max() <= np.finfo(float).eps

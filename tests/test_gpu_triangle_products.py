"""Triangular inverse, LAUUM, POTRI and the likelihood gradient over it at the orders where their products
change form: one 128-row block, the dense copy's smallest orders, ragged last
blocks, levels of several blocks in one launch (FP64).

Accepted: residuals of 4 n eps, the sums of n terms of each product, relative
to the norms of the factors they are taken over (largest row sums)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -53
SIZES = [1, 33, 47, 48, 64, 127, 128, 129, 160, 255, 256, 257, 385, 511, 640, 777, 1024, 1055, 1300, 2049]


@pytest.fixture(scope="module")
def G():
    import torch
    assert torch.cuda.is_available()
    import atlas_gpu
    return atlas_gpu


def norm(a):
    return np.abs(a).sum(1).max(initial=0.0)


def triangle(n, uplo):
    """A triangle with diagonal in [1, 2], a marker in the other one, padding."""
    rng = np.random.default_rng(n)
    a = rng.uniform(-1, 1, (n + 3, n)) / n
    a[np.arange(n), np.arange(n)] = rng.uniform(1, 2, n)
    other = np.triu_indices(n, 1) if uplo == O.Lower else np.tril_indices(n, -1)
    a[:n][other] = 9.0
    return np.asfortranarray(a), other


def run(G, f, a, *args):
    import torch
    d = G.from_fortran(a)
    info = torch.full((1,), -7, dtype=torch.int32, device="cuda")
    f(*args, a.shape[1], d, a.shape[0], *(() if f is G.dlauum else (info,)))
    assert f is G.dlauum or int(info.item()) == 0
    return G.to_fortran(d)


@pytest.mark.parametrize("uplo", [O.Lower, O.Upper])
@pytest.mark.parametrize("n", SIZES)
def test_inverse_and_product(G, uplo, n):
    a, other = triangle(n, uplo)
    part = np.tril if uplo == O.Lower else np.triu
    t = part(a[:n])

    x = run(G, G.dtrtri, a, uplo, G.NonUnit)
    assert np.array_equal(x[:n][other], a[:n][other]) and np.array_equal(x[n:], a[n:])
    x = part(x[:n])
    assert norm(t @ x - np.eye(n)) <= 4 * n * EPS * norm(t) * norm(x)

    p = run(G, G.dlauum, a, uplo)
    assert np.array_equal(p[:n][other], a[:n][other]) and np.array_equal(p[n:], a[n:])
    want = t.T @ t if uplo == O.Lower else t @ t.T
    assert norm(part(p[:n] - want)) <= 4 * n * EPS * norm(t) * norm(t.T)

    q = run(G, G.dpotri, a, uplo)
    assert np.array_equal(q[:n][other], a[:n][other]) and np.array_equal(q[n:], a[n:])
    q = part(q[:n])
    q = q + q.T - np.diag(q.diagonal())
    assert norm(want_full(t, uplo) @ q - np.eye(n)) <= 4 * n * EPS * (norm(t) * norm(t.T)
                                                                    * norm(x) * norm(x.T))


def want_full(t, uplo):
    return t @ t.T if uplo == O.Lower else t.T @ t


@pytest.mark.parametrize("n,zero", [(48, 47), (100, 0), (300, 130), (777, 776)])
def test_zero_diagonal(G, n, zero):
    import torch
    a, _ = triangle(n, O.Lower)
    a[zero, zero] = 0.0
    for f in (lambda d, i: G.dtrtri(O.Lower, G.NonUnit, n, d, n + 3, i),
              lambda d, i: G.dpotri(O.Lower, n, d, n + 3, i)):
        d = G.from_fortran(a)
        info = torch.zeros(1, dtype=torch.int32, device="cuda")
        f(d, info)
        assert int(info.item()) == zero + 1
        assert np.array_equal(G.to_fortran(d), a)


@pytest.mark.parametrize("n,k,same", [(1, 1, False), (20, 2, False), (47, 0, False), (48, 3, True), (65, 16, False),
                                      (100, 17, True), (129, 1, False), (300, 40, False), (513, 2, True)])
def test_loglik_grad(G, n, k, same):
    # g/2 (A A^T - k inv(L L^T)), symmetric to the bit; the sums as above
    import torch
    a, _ = triangle(n, O.Lower)
    t = np.tril(a[:n])
    rng = np.random.default_rng(k)
    x = np.asfortranarray(rng.standard_normal((n + 1, max(k, 1))))
    d, dx = G.from_fortran(a), G.from_fortran(x)
    w = d if same else G.from_fortran(np.full((n + 3, n), np.nan, order="F"))
    g = torch.tensor(-1.7, dtype=torch.float64, device="cuda")
    info = torch.full((1,), -7, dtype=torch.int32, device="cuda")
    G.dloglik_grad(n, k, d, n + 3, dx, n + 1, g, w, n + 3, info)
    assert int(info.item()) == 0
    got = G.to_fortran(w)[:n]
    assert np.array_equal(got, got.T)
    if not same:
        assert np.array_equal(G.to_fortran(d), a)
    ti = np.linalg.inv(t)
    aa = x[:n, :k] @ x[:n, :k].T
    want = -0.85 * (aa - k * (ti.T @ ti))
    scale = norm(t) * norm(t.T) * norm(ti) ** 2 * norm(ti.T) ** 2
    assert norm(got - want) <= 4 * max(n, k, 1) * EPS * (norm(x[:n, :k]) * norm(x[:n, :k].T) + k * scale)


@pytest.mark.parametrize("routine, n", [("dlauum", 48), ("dlauum", 100), ("dtrtri", 200),
                                        ("dpotri", 100), ("dpotri", 128)])
def test_captured_without_workspace(G, routine, n):
    # a stream that has only seen a triangular solve holds no space for the
    # dense copy: a captured call does without it, an eager one may make it
    import torch
    rng = np.random.default_rng(n)
    t = np.asfortranarray(np.tril(rng.uniform(-1, 1, (n, n))) / n + 2 * np.eye(n))
    inv = np.linalg.inv(t)
    want = {"dlauum": t.T @ t, "dtrtri": inv, "dpotri": inv.T @ inv}[routine]
    low = np.tril_indices(n)
    # each entry: sums of at most n products in each of the (at most two)
    # products and the inversion, entries of |L^-1||L||L^-1| of order one
    tol = 8 * n * np.finfo(float).eps * np.abs(want).max()
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        a0 = G.from_fortran(t)
        a = a0.clone()
        info = torch.zeros(1, dtype=torch.int32, device="cuda")
        G.dtrsm(G.Left, G.Lower, G.NoTrans, G.NonUnit, n, n, 1.0, a0, n, a.clone(), n)

        def call():
            a.copy_(a0)
            if routine == "dlauum":
                G.dlauum(G.Lower, n, a, n)
            elif routine == "dtrtri":
                G.dtrtri(G.Lower, G.NonUnit, n, a, n, info)
            else:
                G.dpotri(G.Lower, n, a, n, info)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        call()
    for _ in range(3):
        a.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert int(info.item()) == 0
        assert np.abs(G.to_fortran(a)[low] - want[low]).max() <= tol
        with torch.cuda.stream(s):
            call()
        torch.cuda.synchronize()
        assert np.abs(G.to_fortran(a)[low] - want[low]).max() <= tol

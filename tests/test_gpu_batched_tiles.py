"""Batched Cholesky systems at the sizes where their tiles can go wrong: orders
around the 16x16 tiles and 64-wide block columns, the orders from which the
right-hand sides no longer fit in LDS, right-hand sides around the groups of
four, failing minors in every tile of a block column.

Accepted: backward error ||A X - B|| <= 4 n eps ||A|| ||X|| for the solvers
(sums of n terms and a backward-stable factor, both norms the largest row
sum), ||A - L L^T|| <= 4 n eps ||A|| for the factor.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 3, 15, 16, 17, 33, 48, 63, 64, 65, 79, 81, 127, 128, 129, 191, 200, 257, 320]
EPS = {np.float64: 2.0 ** -53, np.float32: 2.0 ** -24}


@pytest.fixture(scope="module")
def G():
    import torch
    assert torch.cuda.is_available()
    import atlas_gpu
    return atlas_gpu


def spd(n, rng):
    b = rng.standard_normal((n, n))
    return b @ b.T / n + np.eye(n)


def norm(m):
    return np.abs(m).sum(1).max() if m.size else 0.0


class Systems:
    """Column-major matrices with two rows of padding, the upper triangle
    filled with a marker."""

    def __init__(self, mats, rhs, dt):
        import torch
        self.n = [m.shape[0] for m in mats]
        self.ld = [n + 2 for n in self.n]
        self.host, self.rhs = [], []
        for m, b, n in zip(mats, rhs, self.n):
            a = np.full((n + 2, n), -77.0, dt)
            a[:n][np.tril_indices(n)] = m[np.tril_indices(n)]
            x = np.full((n + 2, b.shape[1]), 55.0, dt)
            x[:n] = b
            self.host.append(a)
            self.rhs.append(x)
        self.a = [torch.tensor(np.ascontiguousarray(h.T), device="cuda") for h in self.host]
        self.b = [torch.tensor(np.ascontiguousarray(h.T), device="cuda") for h in self.rhs]
        self.pa = [t.data_ptr() for t in self.a]
        self.pb = [t.data_ptr() for t in self.b]
        self.info = torch.full((len(mats),), -7, dtype=torch.int32, device="cuda")

    def factor(self, k):
        got = self.a[k].cpu().numpy().T
        n = self.n[k]
        up = np.triu_indices(n, 1)
        assert np.array_equal(got[:n][up], self.host[k][:n][up])
        assert np.array_equal(got[n:], self.host[k][n:])
        return np.tril(got[:n]).astype(np.float64)

    def sol(self, k):
        got = self.b[k].cpu().numpy().T
        n = self.n[k]
        assert np.array_equal(got[n:], self.rhs[k][n:])
        return got[:n].astype(np.float64)


def check(s, mats, rhs, eps):
    for k, (m, b) in enumerate(zip(mats, rhs)):
        n, x, f = s.n[k], s.sol(k), s.factor(k)
        low = lambda t: np.tril(t) + np.tril(t, -1).T
        m = low(s.host[k][:n].astype(np.float64))
        b = s.rhs[k][:n].astype(np.float64)
        assert norm(m - f @ f.T) <= 4 * n * eps * norm(m), n
        assert norm(m @ x - b) <= 4 * n * eps * norm(m) * norm(x), n


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("nrhs", [1, 4, 5, 9])
def test_posv(G, dt, nrhs):
    import torch
    rng = np.random.default_rng(nrhs)
    sizes = SIZES + ([1536, 1537] if nrhs in (4, 5) else [])
    mats = [spd(n, rng) for n in sizes]
    rhs = [rng.standard_normal((n, nrhs)) for n in sizes]
    s = Systems(mats, rhs, dt)
    f = G.dposv_batched if dt == np.float64 else G.sposv_batched
    f(s.n, s.pa, s.ld, s.pb, s.ld, nrhs, s.info)
    torch.cuda.synchronize()
    assert not s.info.any()
    check(s, mats, rhs, EPS[dt])


@pytest.mark.parametrize("nrhs", [2, 6])
def test_potrf_potrs(G, nrhs):
    import torch
    rng = np.random.default_rng(30 + nrhs)
    sizes = SIZES + [1537]
    mats = [spd(n, rng) for n in sizes]
    rhs = [rng.standard_normal((n, nrhs)) for n in sizes]
    s = Systems(mats, rhs, np.float64)
    G.dpotrf_batched(s.n, s.pa, s.ld, s.info)
    G.dpotrs_batched(s.n, s.pa, s.ld, s.pb, s.ld, nrhs)
    torch.cuda.synchronize()
    assert not s.info.any()
    check(s, mats, rhs, EPS[np.float64])


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("value", [0.0, -1.0, np.nan])
def test_failing_minor(G, dt, value):
    import torch
    rng = np.random.default_rng(8)
    cases = [(1, 0), (20, 0), (20, 15), (20, 16), (64, 31), (64, 32), (64, 63), (100, 47), (100, 64),
             (150, 81), (150, 149)]
    mats, rhs = [], []
    for n, j in cases:
        m = spd(n, rng)
        m[j, j] = value
        mats.append(m)
        rhs.append(rng.standard_normal((n, 3)))
    s = Systems(mats, rhs, dt)
    f = G.dposv_batched if dt == np.float64 else G.sposv_batched
    f(s.n, s.pa, s.ld, s.pb, s.ld, 3, s.info)
    torch.cuda.synchronize()
    assert s.info.cpu().tolist() == [j + 1 for _, j in cases]
    for k in range(len(cases)):
        s.factor(k)  # the upper triangle and the padding stay
        assert np.array_equal(s.b[k].cpu().numpy().T, s.rhs[k])


@pytest.mark.parametrize("nrhs", [1, 4, 5])
def test_mixed(G, nrhs):
    import torch
    rng = np.random.default_rng(60 + nrhs)
    sizes = [8] + SIZES[2:] + [1024, 1025]
    mats = [spd(n, rng) for n in sizes]
    rhs = [rng.standard_normal((n, nrhs)) for n in sizes]
    s = Systems(mats, rhs, np.float64)
    x = [torch.zeros_like(t) for t in s.b]
    it = torch.full((len(sizes),), 99, dtype=torch.int32, device="cuda")
    G.dsposv_batched(s.n, s.pa, s.ld, s.pb, s.ld, [t.data_ptr() for t in x], s.ld, nrhs, s.info, it)
    torch.cuda.synchronize()
    assert not s.info.any()
    assert all(0 <= v <= 5 for v in it.cpu().tolist())
    for k, n in enumerate(sizes):
        got = x[k].cpu().numpy().T[:n]
        assert norm(mats[k] @ got - rhs[k]) <= 4 * n * EPS[np.float64] * norm(mats[k]) * norm(got)

"""LU panels whose workgroups cannot all be resident at once.

A panel of several workgroups on one XCD waits for them to start, and where
other work keeps one out, a single workgroup factors it in memory.  Forced
here (set_gather_limit(-1)) at the panel's edges, against the oracle's getf2
as test_gpu_lu_panel.py does, and met in earnest by several streams whose
panels together want more compute units than an XCD has: nobody's call may
fail, whoever gets the units.
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
    yield atlas_gpu
    atlas_gpu.set_gather_limit(0)


@pytest.fixture
def alone(G):
    G.set_gather_limit(-1)
    yield
    G.set_gather_limit(0)


def factor(G, a, single=False):
    import torch
    m, n = a.shape
    d = G.from_fortran(a)
    d = d.float() if single else d
    piv = torch.full((min(m, n),), -7, dtype=torch.int32, device="cuda")
    info = torch.zeros(1, dtype=torch.int32, device="cuda")
    (G.sgetrf if single else G.dgetrf)(m, n, d, m, piv, info)
    G.check_stream()
    return G.to_fortran(d), piv.cpu().numpy(), int(info.item())


def oracle(a):
    ref = a.copy(order="F")
    piv, info = O.getf2(ref)
    return ref, piv, info


@pytest.mark.parametrize("n", [1, 7, 32])
@pytest.mark.parametrize("m", [513, 1025, 4097, 8192])
def test_panel(G, alone, m, n):
    a = O.gegen(m, n, m * n + 17 * m)
    lu, piv, info = factor(G, a)
    _, rpiv, rinfo = oracle(a)
    assert np.array_equal(piv, rpiv) and info == rinfo
    assert O.lu_resid(m, n, a, lu, piv) <= 100


def test_panel_single(G, alone):
    # entries of at most 1 times 32 pivots: 32 products of entries of at most
    # max|U|, each rounded in 24 bits
    m, n = 3000, 32
    a = O.gegen(m, n, 5).astype(np.float32).astype(np.float64)
    lu, piv, info = factor(G, a, single=True)
    ref, rpiv, rinfo = oracle(a)
    assert np.array_equal(piv, rpiv) and info == rinfo
    tol = 2 * n * np.finfo(np.float32).eps * max(1.0, np.abs(ref).max()) ** 2
    assert np.abs(lu - ref).max() <= tol


def test_panel_ties_and_zero_columns(G, alone):
    m, n = 700, 32
    a = np.zeros((m, n), order="F")
    for j in range(n):
        a[j::7, j] = 1.0 if j % 2 else -1.0
    a += np.eye(m, n) * 1.0
    a[:, 11] = 0.0
    lu, piv, info = factor(G, a)
    ref, rpiv, rinfo = oracle(a)
    assert np.array_equal(piv, rpiv) and info == rinfo
    tol = 2 * n * np.finfo(float).eps * max(1.0, np.abs(ref).max()) ** 2
    assert np.abs(lu - ref).max() <= tol


@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_panel_nonfinite(G, alone, bad):
    m, n = 700, 32
    a = np.asfortranarray(np.random.default_rng(m).uniform(-1, 1, (m, n)))
    a[m // 3, n // 2] = bad
    lu, piv, _ = factor(G, a)
    ref, rpiv, _ = oracle(a)
    assert np.array_equal(piv, rpiv)
    fin = np.isfinite(ref)
    assert np.array_equal(fin, np.isfinite(lu))
    tol = 2 * n * np.finfo(float).eps * max(1.0, np.abs(ref[fin]).max()) ** 2
    assert np.abs(lu[fin] - ref[fin]).max() <= tol


def test_panel_subnormal_pivot(G, alone):
    m = 600
    a = np.asfortranarray(np.random.default_rng(3).uniform(-1, 1, (m, 2)))
    a[:, 0] *= 2.0 ** -1040
    lu, piv, info = factor(G, a)
    p0 = int(np.argmax(np.abs(a[:, 0])))
    assert info == 0 and piv[0] == p0
    b = a[:, 0].copy()
    b[[0, p0]] = b[[p0, 0]]
    exact = (b[1:] * 2.0 ** 500) / (b[0] * 2.0 ** 500)
    exact[[0, piv[1] - 1]] = exact[[piv[1] - 1, 0]]
    assert np.abs(lu[1:, 0] - exact).max() <= np.finfo(float).eps


@pytest.mark.parametrize("n", [1500, 2304])  # the recursion, the look-ahead
def test_whole_factorization(G, alone, n):
    a = O.gegen(n, n, n)
    lu, piv, info = factor(G, a)
    assert info == 0
    assert O.lu_resid(n, n, a, lu, piv) <= 100
    G.set_gather_limit(0)
    _, together, _ = factor(G, a)
    assert np.array_equal(piv, together)


def test_streams_together(G):
    # tall panels on four streams and two look-aheads (of different widths of
    # reserved units, a Cholesky between them): panels of up to sixteen whole
    # compute units each, all in flight at once
    import torch
    dev = "cuda"
    g = torch.Generator(device=dev)
    g.manual_seed(1)
    shapes = [(8192, 640), (7000, 512), (6500, 640), (8000, 512), (4200, 4200), (8320, 2304)]
    a = [torch.rand((n, m), generator=g, device=dev, dtype=torch.float64) * 2 - 1
         for m, n in shapes]
    spd = torch.eye(2304, dtype=torch.float64, device=dev) * 4.0 + 1.0 / 2304

    def run(streams):
        lu = [x.clone() for x in a]
        ch = spd.clone()
        piv = [torch.full((min(s),), -7, dtype=torch.int32, device=dev) for s in shapes]
        info = torch.full((len(shapes) + 1,), -7, dtype=torch.int32, device=dev)
        torch.cuda.synchronize()
        for i in (4, 0, 1, -1, 2, 3, 5):
            with torch.cuda.stream(streams[i]):
                if i < 0:
                    G.dpotrf(O.Lower, 2304, ch, 2304, info[len(shapes):])
                else:
                    m, n = shapes[i]
                    G.dgetrf(m, n, lu[i], m, piv[i], info[i:])
        for s in streams:
            with torch.cuda.stream(s):
                G.check_stream()
        torch.cuda.synchronize()
        assert (info == 0).all()
        return [p.cpu().numpy() for p in piv], ch

    one = torch.cuda.Stream()
    want, ch0 = run([one] * (len(shapes) + 1))
    for _ in range(2):
        got, ch = run([torch.cuda.Stream() for _ in range(len(shapes) + 1)])
        for w, x in zip(want, got):
            assert np.array_equal(w, x)
        assert torch.equal(ch0, ch)


def test_lookaheads_in_turn(G):
    # look-ahead LUs of both widths of reserved units (order 12000: 64, order
    # 2304: 128), whose panels would share units, run one after the other, also
    # with a Cholesky between them
    import torch
    dev = "cuda"
    g = torch.Generator(device=dev)
    g.manual_seed(2)
    big, small = (torch.rand((n, n), generator=g, device=dev, dtype=torch.float64) * 2 - 1
                  for n in (12000, 2304))
    spd = torch.eye(2304, dtype=torch.float64, device=dev) * 4.0 + 1.0 / 2304
    piv = [torch.zeros(n, dtype=torch.int32, device=dev) for n in (12000, 2304)]
    info = torch.zeros(3, dtype=torch.int32, device=dev)
    s = [torch.cuda.Stream() for _ in range(3)]
    end = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    for _ in range(2):  # the first pass makes streams and workspaces
        a, b, c = big.clone(), small.clone(), spd.clone()
        torch.cuda.synchronize()
        with torch.cuda.stream(s[0]):
            G.dgetrf(12000, 12000, a, 12000, piv[0], info)
            end[0].record()
        with torch.cuda.stream(s[1]):
            G.dpotrf(O.Lower, 2304, c, 2304, info[1:])
        with torch.cuda.stream(s[2]):
            G.dgetrf(2304, 2304, b, 2304, piv[1], info[2:])
            end[1].record()
        torch.cuda.synchronize()
    assert (info == 0).all()
    for x in s:
        with torch.cuda.stream(x):
            G.check_stream()
    assert end[0].elapsed_time(end[1]) > 0

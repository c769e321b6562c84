"""The mixed-precision contractions on the bfloat16 matrix cores (split3.hpp) against FP64.

Every FP32 operand is split exactly into three bfloat16 pieces and the six partial products above
2^-24 are summed in FP32.  The result differs from the FP64 sum of the FP32-rounded operands by
at most (S = sum |a b|, u = 2^-24, G = ceil(K / 32) groups):
  * the partial products left out: |a1 b2| + |a2 b1| + |a2 b2| <= (2^-8 2^-16 2 + 2^-32) |a b| < 3 u S
  * the FP32 additions: within a group at most 192 roundings of a partial sum of that group, one
    of the accumulator per group: (192 + G) u S
  * K slices summed in FP64 and rounded once, the scale factor's product: 2 u |result|
so |error| <= (200 + G) u S, element by element.  That is the worst case of every rounding; whether
a partial product is lost shows in the 2-norm of the error, which is held to 10 u of the result
(test_split_accuracy).  The sizes put walkers, pairs, vectors and k values
on and off the 16-row, 32/16 x 64..96 tile and 32-k group edges.
"""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from safire_amd.synthetic import make_problem  # noqa: E402
from test_split_accuracy import PRODUCT, U, f32, rel2  # noqa: E402


@pytest.fixture(scope="module")
def gpu():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from safire_amd import afq
    return afq, afq.Context(0), torch


def bound(A, B, K):
    """(200 + G) u sum |a b| of each output, A [W][K] complex, B [n][K] real."""
    g = (200 + (K + 31) // 32) * U
    return g * (np.abs(A.real) @ np.abs(B).T), g * (np.abs(A.imag) @ np.abs(B).T)


# tile edges: 16 and 32 walkers, 64 / 80 / 96 columns, 32 k values; the smallest and ragged sizes
@pytest.mark.parametrize("N,M,W", [(2, 1, 1), (8, 31, 15), (9, 32, 16), (13, 33, 17), (16, 64, 33),
                                   (24, 96, 64), (31, 155, 65), (97, 487, 301), (200, 160, 130)])
def test_vhs(gpu, N, M, W):
    afq, ctx, torch = gpu
    print(f"case: split vHS N={N} M={M} W={W}", flush=True)
    p = make_problem(N, 1, M, 3)
    ham = afq.HamiltonianOperations(ctx, p.h1, p.Likn, p.PsiT, 1, precision=afq.AFQ_MIXED)
    rng = np.random.default_rng(W)
    X = f32(rng.normal(size=(W, M)) + 1j * rng.normal(size=(W, M)))
    V = afq.empty((W, N, N), torch.complex64)
    ham.vHS(afq.device_tensor(X), V, 1.0)
    V = afq.host(V)
    assert np.array_equal(V, np.transpose(V, (0, 2, 1)))
    B = f32(p.Likn).reshape(N * N, M).astype(np.float64)
    A = X.astype(np.complex128)
    ref, (br, bi) = A @ B.T, bound(A, B, M)
    d = V.reshape(W, -1) - ref
    assert rel2(V.reshape(W, -1), ref) <= PRODUCT
    assert np.all(np.abs(d.real) <= br) and np.all(np.abs(d.imag) <= bi)


@pytest.mark.parametrize("N,n,nd,M,W", [(2, 1, 0, 1, 1), (9, 2, 0, 33, 17), (16, 3, 2, 95, 31),
                                        (40, 7, 0, 161, 64), (33, 8, 0, 165, 129),
                                        (120, 30, 28, 97, 160)])
def test_vbias(gpu, N, n, nd, M, W):
    afq, ctx, torch = gpu
    print(f"case: split vbias N={N} n={n}+{nd} M={M} W={W}", flush=True)
    p = make_problem(N, n, M, 4)
    wt = afq.AFQ_COLLINEAR if nd else afq.AFQ_CLOSED
    rows = np.concatenate([p.PsiT, p.PsiT[:nd]])
    ham = afq.HamiltonianOperations(ctx, p.h1, p.Likn, rows, n, nd, walker_type=wt,
                                    precision=afq.AFQ_MIXED)
    rng = np.random.default_rng(N)
    G = rng.normal(size=(W, n + nd, N)) + 1j * rng.normal(size=(W, n + nd, N))
    v = afq.empty((W, M), torch.complex128)
    ham.vbias(afq.device_tensor(G), v, 1.0)
    v = afq.host(v)
    L = ham.tensors()[0].real
    c = 1.0 if nd else 2.0
    ref, br, bi, g0, l0 = 0, 0, 0, 0, 0
    for ns in (n, nd):
        if not ns:
            continue
        A = f32(G[:, g0:g0 + ns].reshape(W, -1)).astype(np.complex128)
        B = f32(L[l0:l0 + M * ns * N].reshape(M, -1)).astype(np.float64)
        r, i = bound(A, B, ns * N)
        ref, br, bi = ref + c * (A @ B.T), br + c * r, bi + c * i
        g0, l0 = g0 + ns, l0 + M * ns * N
    d = v - ref
    assert rel2(v, ref) <= PRODUCT
    assert np.all(np.abs(d.real) <= br) and np.all(np.abs(d.imag) <= bi)


def test_infinities_and_nan(gpu):
    """A walker with an infinite or NaN field gives the infinities and NaN of the FP32 products
    (AFQ_CRGEMM=0); the other walkers keep their bits."""
    afq, ctx, torch = gpu
    N, M, W = 12, 40, 21
    print(f"case: split vHS with infinities N={N} M={M} W={W}", flush=True)
    p = make_problem(N, 1, M, 5)
    ham = afq.HamiltonianOperations(ctx, p.h1, p.Likn, p.PsiT, 1, precision=afq.AFQ_MIXED)
    rng = np.random.default_rng(1)
    X = f32(rng.normal(size=(W, M)) + 1j * rng.normal(size=(W, M)))

    def vhs(x):
        V = afq.empty((W, N, N), torch.complex64)
        ham.vHS(afq.device_tensor(x), V, 1.0)
        return afq.host(V)
    clean = vhs(X)
    Y = X.copy()
    Y[3, 7] = np.inf
    Y[16, 39] = complex(0.5, -np.inf)
    Y[18, 0] = np.nan
    Y[20, 5], Y[20, 6] = np.inf, -np.inf
    got = vhs(Y)
    os.environ["AFQ_CRGEMM"] = "0"
    try:
        ref = vhs(Y)
    finally:
        del os.environ["AFQ_CRGEMM"]
    rest = [w for w in range(W) if w not in (3, 16, 18, 20)]
    assert np.array_equal(got[rest], clean[rest])
    for part in (np.real, np.imag):
        g, r = part(got), part(ref)
        assert np.array_equal(np.isnan(g), np.isnan(r))
        inf = np.isinf(r)
        assert np.array_equal(np.isinf(g), inf) and np.array_equal(g[inf], r[inf])


def test_tensors_outside_the_split_keep_the_fp32_product(gpu):
    """A Cholesky tensor with an infinity is contracted as before (no split operand is built)."""
    afq, ctx, torch = gpu
    N, M, W = 10, 33, 5
    print("case: infinite Cholesky entry", flush=True)
    p = make_problem(N, 1, M, 6)
    L = p.Likn.copy()
    L[2, 4, 9] = L[4, 2, 9] = np.inf
    ham = afq.HamiltonianOperations(ctx, p.h1, L, p.PsiT, 1, precision=afq.AFQ_MIXED)
    X = f32(np.ones((W, M)) * (1 + 2j))

    def vhs():
        V = afq.empty((W, N, N), torch.complex64)
        ham.vHS(afq.device_tensor(X), V, 1.0)
        return afq.host(V)
    V = vhs()
    os.environ["AFQ_CRGEMM"] = "0"
    try:
        ref = vhs()
    finally:
        del os.environ["AFQ_CRGEMM"]
    assert np.array_equal(V, ref, equal_nan=True)
    assert not np.any(np.isfinite(V[:, 2, 4])) and not np.any(np.isfinite(V[:, 4, 2]))
    V[:, 2, 4] = V[:, 4, 2] = 0
    assert np.all(np.isfinite(V))


# one K slice and several; both parts, one walker past FP32's range
@pytest.mark.parametrize("N,n,nd,M,W", [(12, 3, 0, 40, 21), (33, 8, 0, 165, 40), (40, 9, 7, 96, 21)])
def test_vbias_infinities_and_nan(gpu, N, n, nd, M, W):
    """As test_infinities_and_nan for a density matrix."""
    afq, ctx, torch = gpu
    print(f"case: split vbias with infinities N={N} n={n}+{nd} M={M} W={W}", flush=True)
    p = make_problem(N, n, M, 5)
    ham = afq.HamiltonianOperations(
        ctx, p.h1, p.Likn, np.concatenate([p.PsiT, p.PsiT[:nd]]), n, nd,
        walker_type=afq.AFQ_COLLINEAR if nd else afq.AFQ_CLOSED, precision=afq.AFQ_MIXED)
    rng = np.random.default_rng(1)
    G = rng.normal(size=(W, n + nd, N)) + 1j * rng.normal(size=(W, n + nd, N))

    def vbias(g):
        v = afq.empty((W, M), torch.complex128)
        ham.vbias(afq.device_tensor(g), v, 1.0)
        return afq.host(v)
    clean = vbias(G)
    H = G.copy()
    H[3, n - 1, 7] = np.inf
    H[16, 0, N - 1] = complex(0.5, -1e39)
    H[18, n + nd - 1, 0] = np.nan
    H[20, 0, 0], H[20, n + nd - 1, N - 1] = np.inf, -np.inf
    got = vbias(H)
    os.environ["AFQ_CRGEMM"] = "0"
    try:
        ref = vbias(H)
    finally:
        del os.environ["AFQ_CRGEMM"]
    rest = [w for w in range(W) if w not in (3, 16, 18, 20)]
    assert np.array_equal(got[rest], clean[rest])
    for part in (np.real, np.imag):
        g, r = part(got), part(ref)
        assert np.array_equal(np.isnan(g), np.isnan(r))
        inf = np.isinf(r)
        assert np.array_equal(np.isinf(g), inf) and np.array_equal(g[inf], r[inf])


@pytest.mark.parametrize("which", ["vHS", "vbias"])
def test_captured_without_a_first_call(gpu, which):
    """The first vHS or vbias of a context inside a HIP graph capture is recorded (a capture cannot
    allocate: it takes the FP32 engine), and a graph that was captured after a first call keeps
    giving its result when later calls with more walkers have made the workspace grow."""
    afq, _, torch = gpu
    N, n, M, W = 24, 5, 30, 8
    print(f"case: captured {which}", flush=True)
    p = make_problem(N, n, M, 8)
    rng = np.random.default_rng(2)

    def inputs(w):
        s = (w, M) if which == "vHS" else (w, n, N)
        x = afq.device_tensor(rng.normal(size=s) + 1j * rng.normal(size=s))
        if which == "vHS":
            return x.to(torch.complex64), afq.empty((w, N, N), torch.complex64)
        return x, afq.empty((w, M), torch.complex128)

    for warm in (False, True):
        ctx = afq.Context(0)
        ham = afq.HamiltonianOperations(ctx, p.h1, p.Likn, p.PsiT, n, precision=afq.AFQ_MIXED)
        x, out = inputs(W)
        if warm:
            getattr(ham, which)(x, out, 0.01)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=ctx.stream):
            getattr(ham, which)(x, out, 0.01)
        for grow in (1, 5, 40):
            y, big = inputs(W * grow)
            getattr(ham, which)(y, big, 0.01)
            eager = torch.empty_like(out)
            getattr(ham, which)(x, eager, 0.01)
            out.zero_()
            g.replay()
            torch.cuda.synchronize()
            a, b = afq.host(out), afq.host(eager)
            if warm:
                assert np.array_equal(a, b)
            else:  # other kernels: 30 or 120 FP32 products of N(0, 1) numbers
                assert np.max(np.abs(a - b)) < 1e-5 * np.max(np.abs(b))


@pytest.mark.parametrize("N,n,nd,M,W", [(37, 9, 7, 150, 96), (64, 16, 16, 320, 256)])
def test_two_spins_take_the_launches_of_one(gpu, N, n, nd, M, W):
    """A two-spin vbias packs both density matrices in one launch and forms one product whose K slices
    keep the spins apart: three launches at most (pack, product, sum of the slices)."""
    import ctypes
    afq, ctx, torch = gpu
    print(f"case: launches of a two-spin vbias N={N} n={n}+{nd} M={M} W={W}", flush=True)
    p = make_problem(N, n, M, 4)
    ham = afq.HamiltonianOperations(ctx, p.h1, p.Likn, np.concatenate([p.PsiT, p.PsiT[:nd]]), n, nd,
                                    walker_type=afq.AFQ_COLLINEAR, precision=afq.AFQ_MIXED)
    G = torch.randn(W, n + nd, N, dtype=torch.complex128, device="cuda")
    v = afq.empty((W, M), torch.complex128)
    ham.vbias(G, v, 1.0)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(g, stream=ctx.stream):
        ham.vbias(G, v, 1.0)
    hip = ctypes.CDLL("libamdhip64.so")
    nodes = ctypes.c_size_t(0)
    assert hip.hipGraphGetNodes(ctypes.c_void_p(g.raw_cuda_graph()), None,
                                ctypes.byref(nodes)) == 0
    print("  nodes", nodes.value, flush=True)
    assert 2 <= nodes.value <= 3


def test_fields_past_2_gib(gpu):
    """Packed fields of more than 2 GiB (unsigned 32-bit offsets): the last walkers' V."""
    afq, ctx, torch = gpu
    N, M, W = 8, 1024, 180_000
    print(f"case: split vHS, fields past 2 GiB N={N} M={M} W={W}", flush=True)
    p = make_problem(N, 1, M, 3)
    ham = afq.HamiltonianOperations(afq.Context(0), p.h1, p.Likn, p.PsiT, 1,
                                    precision=afq.AFQ_MIXED)
    g = torch.Generator(device="cuda").manual_seed(5)
    X = torch.randn(W, M, generator=g, dtype=torch.complex64, device="cuda")
    V = afq.empty((W, N, N), torch.complex64)
    ham.vHS(X, V, 1.0)
    L = f32(p.Likn).reshape(N * N, M).astype(np.float64)
    for rows in (slice(0, 40), slice(W - 40, W)):
        ref = afq.host(X[rows]).astype(np.complex128) @ L.T
        assert rel2(afq.host(V[rows]).reshape(40, -1), ref) <= PRODUCT


def test_walkers_in_runs(gpu):
    """A density matrix whose packed form passes 4 GiB is taken in runs of walkers."""
    afq, ctx, torch = gpu
    N, n, M, W = 64, 32, 5, 180_000
    print(f"case: split vbias, walker runs N={N} n={n} M={M} W={W}", flush=True)
    p = make_problem(N, n, M, 3)
    ham = afq.HamiltonianOperations(afq.Context(0), p.h1, p.Likn, p.PsiT, n,
                                    precision=afq.AFQ_MIXED)
    g = torch.Generator(device="cuda").manual_seed(6)
    G = torch.randn(W, n, N, generator=g, dtype=torch.complex128, device="cuda")
    v = afq.empty((W, M), torch.complex128)
    ham.vbias(G, v, 1.0)
    L = f32(ham.tensors()[0].real.reshape(M, -1)).astype(np.float64)
    for w0 in (0, 100_000, 170_000, W - 40):
        ref = 2.0 * f32(afq.host(G[w0:w0 + 40]).reshape(40, -1)).astype(np.complex128) @ L.T
        assert rel2(afq.host(v[w0:w0 + 40]), ref) <= PRODUCT


def test_vectors_in_runs(gpu):
    """Two spins' half-rotated rows of more than 4 GiB packed (each below it) are taken in runs of
    vectors."""
    afq, ctx, torch = gpu
    N = n = 33
    M, W = 350_000, 3
    print(f"case: split vbias, vector runs N={N} n={n}+{n} M={M} W={W}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(9)
    L = torch.randn(N, N, M, generator=g, dtype=torch.float64, device="cuda") / N
    L = 0.5 * (L + L.transpose(0, 1))
    rng = np.random.default_rng(9)
    h1 = rng.normal(size=(N, N))
    P = np.linalg.qr(rng.normal(size=(N, N)))[0]
    ham = afq.HamiltonianOperations(afq.Context(0), 0.5 * (h1 + h1.T), L.cpu().numpy(),
                                    np.concatenate([P, P]).astype(np.complex128), n, n,
                                    walker_type=afq.AFQ_COLLINEAR, precision=afq.AFQ_MIXED)
    G = afq.device_tensor(rng.normal(size=(W, 2 * n, N)) + 1j * rng.normal(size=(W, 2 * n, N)))
    v = afq.empty((W, M), torch.complex128)
    ham.vbias(G, v, 1.0)
    # sum over a, k of G[a][k] sum_i P[a][i] L[i][k][m], both spins with the same P
    F = torch.einsum("ai,wak->wik", afq.device_tensor(P).to(torch.complex128), G[:, :n] + G[:, n:])
    F, L = F.reshape(W, -1), L.reshape(N * N, M)
    ref = torch.complex(F.real.contiguous() @ L, F.imag.contiguous() @ L)
    # (two more roundings to FP32, of G and of the half-rotated rows, are in the result)
    for m in (slice(0, 1000), slice(M // 2, M // 2 + 1000), slice(M - 1000, M)):
        assert rel2(afq.host(v[:, m]), afq.host(ref[:, m])) <= PRODUCT + 2 * U

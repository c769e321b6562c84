"""The mixed-precision propagation on the bfloat16 matrix cores (prop_split.hip) against FP64.

Phi <- P1 (sum_k (iV)^k / k!) P1 Phi with FP32 products.  Every product of N terms carries at most
(200 + ceil(N / 32)) u relative to sum |a||b| (see test_gpu_split3; u = 2^-24), so with
A = |P1|, B = |V| the error is bounded, entry by entry, by
    c u A (sum_k B^k / k!) A |Phi|,   c = (order + 2) (200 + ceil(N / 32) + 4),
the 4 covering the rounding of the tile to FP32, the factor 1/k, the running sum and the operand
stored as FP32.  That is the worst case of every rounding; whether a partial product is lost shows in
the 2-norm of the error, which is held to 8 u of the result (test_split_accuracy).  Sizes: one stripe to sixteen (every remainder of the rows of four stripes), 1 to 64
columns (pairs, the mixed block, several workgroups per walker), odd N (rows not 16-byte
aligned), and every number of workgroups per walker, which must not change a bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from test_split_accuracy import PROPAGATION, U, rel2  # noqa: E402


@pytest.fixture(scope="module")
def gpu():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from safire_amd import afq
    return afq, afq.Context(0), torch


def inputs(N, n, W, complex_p1=True):
    rng = np.random.default_rng(N * 100 + n)

    def z(*s):
        return rng.normal(size=s) + 1j * rng.normal(size=s)
    P1 = np.eye(N) + 0.1 * (z(N, N) if complex_p1 else rng.normal(size=(N, N))) / N
    V = (0.3 / np.sqrt(N) * z(W, N, N)).astype(np.complex64)
    Phi = z(W, N, n) * np.exp(rng.normal(size=(W, 1, 1)))
    return P1.astype(np.complex64).astype(np.complex128), V, Phi


def propagate(afq, ctx, P1, V, Phi, order=6):
    d = afq.device_tensor(Phi)
    afq.det_ops.Propagate(ctx, afq.device_tensor(P1), afq.device_tensor(V), d, order, "N",
                          afq.AFQ_MIXED)
    return afq.host(d)


@pytest.mark.parametrize("N,n,W", [(1, 1, 2), (15, 2, 3), (16, 8, 3), (17, 9, 3), (33, 16, 3),
                                   (48, 17, 2), (49, 24, 2), (64, 25, 2), (65, 32, 2), (96, 33, 2),
                                   (97, 23, 3), (113, 40, 2), (128, 41, 2), (129, 64, 2),
                                   (160, 40, 2), (177, 12, 2), (200, 40, 3), (210, 7, 2),
                                   (225, 40, 2), (256, 48, 2)])
def test_against_fp64(gpu, N, n, W):
    afq, ctx, torch = gpu
    print(f"case: split propagation N={N} n={n} W={W}", flush=True)
    P1, V, Phi = inputs(N, n, W)
    got = propagate(afq, ctx, P1, V, Phi)
    T = P1 @ Phi
    S = T.copy()
    Ta = np.abs(P1) @ np.abs(Phi)
    Sa = Ta.copy()
    for k in range(1, 7):
        T = (1j / k) * (V.astype(np.complex128) @ T)
        Ta = (np.abs(V).astype(np.float64) @ Ta) / k
        S, Sa = S + T, Sa + Ta
    c = 8 * (200 + (N + 31) // 32 + 4) * U
    assert rel2(got, P1 @ S) <= PROPAGATION
    # (a complex product's real part has two real ones, both within |a||b|)
    assert np.all(np.abs(got - P1 @ S) <= 2 * c * (np.abs(P1) @ Sa))


# The FP32 kernel: beyond sixteen stripes, and below with the three-product form or without a V
# product.  A sum of N terms takes N roundings, N u in the worst case and about the square root of it
# (17 u) in the 2-norm, of each term falling by k!; three products lose up to another factor of four
# (sums of two operands and of three results).
@pytest.mark.parametrize("N,n,W,order,m3", [(257, 9, 2, 6, False), (300, 40, 2, 6, False),
                                            (300, 17, 2, 6, True), (97, 23, 2, 6, True),
                                            (200, 40, 2, 6, True), (50, 11, 2, 0, False),
                                            (128, 40, 2, 0, False), (270, 20, 2, 0, False)])
def test_fp32_kernel(gpu, monkeypatch, N, n, W, order, m3):
    afq, ctx, torch = gpu
    print(f"case: FP32 propagation N={N} n={n} W={W} order={order} m3={m3}", flush=True)
    if m3:
        monkeypatch.setenv("AFQ_PROP_M3", "1")
    P1, V, Phi = inputs(N, n, W)
    got = propagate(afq, ctx, P1, V, Phi, order)
    T = P1 @ Phi
    S = T.copy()
    Ta = np.abs(P1) @ np.abs(Phi)
    Sa = Ta.copy()
    for k in range(1, order + 1):
        T = (1j / k) * (V.astype(np.complex128) @ T)
        Ta = (np.abs(V).astype(np.float64) @ Ta) / k
        S, Sa = S + T, Sa + Ta
    c = (order + 2) * (N + 4) * U
    assert np.all(np.abs(got - P1 @ S) <= (8 if m3 else 2) * c * (np.abs(P1) @ Sa))
    assert rel2(got, P1 @ S) <= (4 if m3 else 1) * 2 * PROPAGATION


@pytest.mark.parametrize("N,n,W", [(40, 40, 3), (97, 23, 5), (200, 40, 4), (70, 64, 3)])
def test_workgroups_per_walker_keep_the_bits(gpu, N, n, W):
    afq, ctx, torch = gpu
    print(f"case: split propagation, every candidate N={N} n={n} W={W}", flush=True)
    P1, V, Phi = inputs(N, n, W)
    ref = propagate(afq, ctx, P1, V, Phi)
    # fewer and fewer of the n8 groups of 8 columns a workgroup, from five on, four candidates at most
    n8 = -(-n // 8)
    widths = sorted({-(-n8 // k) for k in range(-(-n8 // 5), n8 + 1)}, reverse=True)[:4]
    for i in range(len(widths) + 1):
        afq.tune_force("prop_fused:f32", i)
        try:
            if i == len(widths):
                with pytest.raises(afq.AfqError):
                    propagate(afq, ctx, P1, V, Phi)
            else:
                assert np.array_equal(propagate(afq, ctx, P1, V, Phi), ref), i
        finally:
            afq.tune_force("prop_fused:f32", -1)


@pytest.mark.parametrize("N,n", [(45, 11), (97, 24), (200, 40)])
@pytest.mark.parametrize("complex_p1", [False, True])
def test_diagonals_of_p1(gpu, N, n, complex_p1):
    """Diagonal entries around one are reduced by it and the row added back; others are not.  The
    added rows are one more rounding of a term of the bound."""
    afq, ctx, torch = gpu
    print(f"case: split propagation, diagonals N={N} n={n} complex={complex_p1}", flush=True)
    P1, V, Phi = inputs(N, n, 2, complex_p1)
    diag = np.resize([1.0, 0.5, 2.0, 0.4999, 2.001, 0.0, -1.0, 0.75, 1.5], N).astype(np.float32)
    P1[np.arange(N), np.arange(N)] = diag
    got = propagate(afq, ctx, P1, V, Phi, order=1)
    T = P1 @ Phi
    S = T + 1j * (V.astype(np.complex128) @ T)
    Ta = np.abs(P1) @ np.abs(Phi)
    Sa = Ta + np.abs(V).astype(np.float64) @ Ta
    c = 3 * (200 + (N + 31) // 32 + 5) * U
    # |P1_ii - 1| + 1 is at most 3 |P1_ii| for entries of at least 1/2
    assert np.all(np.abs(got - P1 @ S) <= 6 * c * (np.abs(P1) @ Sa))


def test_walkers_past_fp32_range(gpu):
    """A walker of size 2^130 and one of 2^-130 give the scaled result of the others exactly."""
    afq, ctx, torch = gpu
    N, n = 45, 11
    print(f"case: split propagation, scaled walkers N={N} n={n}", flush=True)
    P1, V, Phi = inputs(N, n, 1)
    V3, s = np.repeat(V, 3, axis=0), np.array([1.0, 2.0 ** 130, 2.0 ** -130])[:, None, None]
    got = propagate(afq, ctx, P1, V3, np.repeat(Phi, 3, axis=0) * s)
    assert np.array_equal(got[1] / 2.0 ** 130, got[0])
    assert np.array_equal(got[2] * 2.0 ** 130, got[0])


def plain(P1, V, Phi, order):
    """The recurrence in float64 with every complex product as four real ones, k by k, so that an
    infinity times a zero part is the NaN that the FP32 products give."""
    def mul(a, b, sign=1.0):
        ar, ai, br, bi = a.real, a.imag, b.real, b.imag

        def dot(x, y):
            return (x[:, :, None] * y[None]).sum(axis=1)
        with np.errstate(all="ignore"):
            return dot(ar, br) - dot(ai, bi), dot(ar, bi) + dot(ai, br)

    def z(re, im):
        out = np.empty(re.shape, np.complex128)
        out.real, out.imag = re, im
        return out
    T = z(*mul(P1, Phi))
    S = T.copy()
    for k in range(1, order + 1):
        re, im = mul(V, T)
        T = z(-(im / k), re / k)
        with np.errstate(all="ignore"):
            S = z(S.real + T.real, S.imag + T.imag)
    return z(*mul(P1, S))


@pytest.mark.parametrize("N,n", [(1, 1), (7, 3), (40, 21), (97, 23), (150, 12), (200, 40)])
@pytest.mark.parametrize("order", [1, 2, 6])
def test_infinities_and_nan(gpu, N, n, order):
    """Infinities and NaN in the walkers, in V and in P1: infinite and NaN where the products in
    FP32 are.  The other walkers keep their bits, the other columns of a walker with such a column
    their values (1e-5 of the largest: FP32 products of at most 200 terms, four to eight of them)."""
    afq, ctx, torch = gpu
    print(f"case: split propagation with infinities N={N} n={n} order={order}", flush=True)
    P1, V, Phi = inputs(N, n, 6)
    Phi[:] /= np.abs(Phi).max(axis=(1, 2), keepdims=True)
    clean = propagate(afq, ctx, P1, V, Phi, order)
    inf, nan = np.inf, np.nan
    A, B = V.copy(), Phi.copy()
    B[0, N - 1, n - 1] = complex(inf, 0.5)
    B[1, 0, 0] = complex(0.5, nan)
    A[2, N // 2, 0] = complex(-inf, 0.5)
    A[3, 0, N - 1] = complex(0.5, nan)
    got = propagate(afq, ctx, P1, A, B, order)
    assert np.array_equal(got[4:], clean[4:])
    if n > 1:
        for w, cols in ((0, np.s_[:n - 1]), (1, np.s_[1:])):
            assert np.max(np.abs(got[w][:, cols] - clean[w][:, cols])) < 1e-5 * np.max(np.abs(clean[w]))
    for w in range(4):
        ref = plain(P1, A[w].astype(np.complex128), B[w], order)
        for x, y in ((got[w].real, ref.real), (got[w].imag, ref.imag)):
            assert np.array_equal(np.isnan(x), np.isnan(y)), w
            m = np.isinf(y)
            assert np.array_equal(np.isinf(x), m) and np.array_equal(x[m], y[m]), w
    Q = P1.copy()
    Q[N // 3, N // 2] = complex(inf, 1.0)
    got = propagate(afq, ctx, Q, V, Phi, order)
    for w in range(6):
        ref = plain(Q, V[w].astype(np.complex128), Phi[w], order)
        for x, y in ((got[w].real, ref.real), (got[w].imag, ref.imag)):
            assert np.array_equal(np.isnan(x), np.isnan(y)), w
            m = np.isinf(y)
            assert np.array_equal(np.isinf(x), m) and np.array_equal(x[m], y[m]), w


def test_overflow(gpu):
    """A Taylor term past FP32's range: T_0 = 1.5, T_1 = (0, 4.5e38) becomes (0, inf) and leaves
    P1 (1.5, inf) = (1.5 - 0 inf, inf + 0) = (NaN, inf)."""
    afq, ctx, torch = gpu
    print("case: split propagation past FP32's range", flush=True)
    got = propagate(afq, ctx, np.ones((1, 1), np.complex128),
                    np.full((1, 1, 1), 3e38, np.complex64), np.full((1, 1, 1), 1.5 + 0j), 1)[0, 0, 0]
    assert np.isnan(got.real) and got.imag == np.inf


def test_tuned_choices_are_not_shared_between_candidate_lists(gpu):
    """48 and 64 columns have three and four candidates: each keeps a choice of its own."""
    afq, ctx, torch = gpu
    print("case: split propagation, tuning keys", flush=True)
    for n in (48, 64):
        propagate(afq, ctx, *inputs(190, n, 9))
    lines = [x for x in afq.tuning_report().splitlines() if x.startswith("prop_fused:f32:16x256x64x")]
    assert sorted(x.rsplit(" of ", 1)[1] for x in lines) == ["3", "4"]

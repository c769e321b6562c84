"""The mixed-precision propagation on the bfloat16 matrix cores (prop_split.hip) against FP64.

Phi <- P1 (sum_k (iV)^k / k!) P1 Phi with FP32 products.  Every product of N terms carries at most
(200 + ceil(N / 32)) u relative to sum |a||b| (see test_gpu_split3; u = 2^-24), so with
A = |P1|, B = |V| the error is bounded, entry by entry, by
    c u A (sum_k B^k / k!) A |Phi|,   c = (order + 2) (200 + ceil(N / 32) + 4),
the 4 covering the rounding of the tile to FP32, the factor 1/k, the running sum and the operand
stored as FP32.  Sizes: one stripe to sixteen (every remainder of the rows of four stripes), 1 to 64
columns (pairs, the mixed block, several workgroups per walker), odd N (rows not 16-byte
aligned), and every number of workgroups per walker, which must not change a bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


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
    # (a complex product's real part has two real ones, both within |a||b|)
    assert np.all(np.abs(got - P1 @ S) <= 2 * c * (np.abs(P1) @ Sa))


@pytest.mark.parametrize("N,n,W", [(40, 40, 3), (97, 23, 5), (200, 40, 4)])
def test_workgroups_per_walker_keep_the_bits(gpu, N, n, W):
    afq, ctx, torch = gpu
    print(f"case: split propagation, every candidate N={N} n={n} W={W}", flush=True)
    P1, V, Phi = inputs(N, n, W)
    ref = propagate(afq, ctx, P1, V, Phi)
    for i in range(3):
        afq.tune_force("prop_fused:f32", i)
        try:
            got = propagate(afq, ctx, P1, V, Phi)
        finally:
            afq.tune_force("prop_fused:f32", -1)
        assert np.array_equal(got, ref), i


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

"""The batched inverse and log det at the edges of its row lengths (8, 16, 24, 32, 40, 48, 64 columns;
two wavefronts above 48) against numpy.

The matrices are row permutations of n I plus unit noise, so partial pivoting has to find every
row and their condition number k is small; both inverses carry an error of at most
16 n u k relative (u = 2^-53; Gauss-Jordan with pivot growth at most 2 on such matrices), and the log
det n times the relative error of a pivot.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -53


@pytest.fixture(scope="module")
def gpu():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from safire_amd import afq
    return afq, afq.Context(0), torch


def run(afq, ctx, torch, A):
    inv, ld = afq.empty(A.shape, torch.complex128), afq.empty(A.shape[0], torch.complex128)
    ld.zero_()
    afq.det_ops.inverse_logdet(ctx, afq.device_tensor(A), ld, inv)
    return afq.host(inv), afq.host(ld)


@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 16, 17, 23, 24, 25, 32, 33, 40, 41, 47, 48, 49, 63, 64])
def test_inverse_logdet(gpu, n):
    afq, ctx, torch = gpu
    print(f"case: inverse and log det n={n}", flush=True)
    rng = np.random.default_rng(n)
    B = n * np.eye(n) + (rng.normal(size=(5, n, n)) + 1j * rng.normal(size=(5, n, n))) / np.sqrt(2)
    A = np.stack([b[rng.permutation(n)] for b in B])
    got, ld = run(afq, ctx, torch, A)
    ref = np.linalg.inv(A)
    sign, mag = np.linalg.slogdet(A)
    for g, r, a in zip(got, ref, A):
        k = np.linalg.cond(a)
        assert np.linalg.norm(g - r) <= 16 * n * U * k * np.linalg.norm(r)
    assert np.all(np.abs(ld.real - mag) <= 32 * n * n * U * np.maximum(1.0, np.abs(mag)))
    assert np.all(np.abs(np.exp(1j * ld.imag) - sign) <= 32 * n * n * U)


@pytest.mark.parametrize("n", [3, 24, 48, 50, 64])
def test_ties_and_singular(gpu, n):
    """Equal magnitudes take the first row (a permutation matrix of 1, -1, i, -i has exact results);
    a zero column gives a zero inverse."""
    afq, ctx, torch = gpu
    print(f"case: inverse and log det, ties n={n}", flush=True)
    rng = np.random.default_rng(n)
    A = np.zeros((3, n, n), np.complex128)
    for a in A:
        a[np.arange(n), rng.permutation(n)] = rng.choice([1, -1, 1j, -1j], size=n)
    A[1, :, n // 2] = 0.0
    A[2] += 2.0 * (np.add.outer(np.arange(n), np.arange(n)) % 2 == 0)  # ties in every column
    A[2] += 4.0 * n * np.eye(n)
    got, ld = run(afq, ctx, torch, A)
    assert np.array_equal(got[0], A[0].conj().T)
    assert abs(ld[0].real) <= n * U
    assert np.all(got[1] == 0.0)
    r = np.linalg.inv(A[2])
    assert np.linalg.norm(got[2] - r) <= 16 * n * U * np.linalg.cond(A[2]) * np.linalg.norm(r)


def test_many_matrices_keep_the_bits(gpu):
    """Above 48 columns many matrices take a kernel with fewer registers: the same arithmetic."""
    afq, ctx, torch = gpu
    print("case: inverse and log det, 3 and 900 matrices n=52", flush=True)
    rng = np.random.default_rng(52)
    A = rng.normal(size=(3, 52, 52)) + 1j * rng.normal(size=(3, 52, 52))
    few, many = run(afq, ctx, torch, A), run(afq, ctx, torch, np.tile(A, (300, 1, 1)))
    assert np.array_equal(np.tile(few[0], (300, 1, 1)), many[0])
    assert np.array_equal(np.tile(few[1], 300), many[1])

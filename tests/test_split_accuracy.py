"""What the accuracy bounds of the split bfloat16 products can see, on the CPU.

An FP32 product is formed from the pieces a0 + a1 + a2 and b0 + b1 + b2 of its factors as the six
partial products a0 b0, a0 b1, a1 b0, a1 b1, a0 b2, a2 b0 (split3.hpp).  The GPU tests bound the
2-norm of the error, relative to that of the result, by
  * PRODUCT = 10 u for a product (u = 2^-24): what is left out is 0.1 u, and the FP32 additions of
    1600 falling terms, one after the other, come to 7 u (the kernels round less often);
  * PROPAGATION = 8 u for the recurrence of the propagation: a rounding to FP32 of the tile, of every
    term and of the sum, each about u / 3 rms, beside the products' own.
Here the six products are emulated in 64 bits: with all of them the error is far below the bounds,
and with any one of them lost it is above.
"""
import numpy as np
import pytest

U = 2.0 ** -24
PRODUCT = 10 * U
PROPAGATION = 8 * U

SIX = ((0, 0), (0, 1), (1, 0), (1, 1), (0, 2), (2, 0))
KEPT = {"six": SIX, "two pieces": SIX[:4], **{f"without a{i} b{j}": tuple(k for k in SIX if k != (i, j))
                                               for i, j in SIX[1:]}}


def rel2(a, b):
    return float(np.linalg.norm(np.asarray(a) - b) / np.linalg.norm(b))


def f32(x):
    return np.asarray(x).astype(np.complex64 if np.iscomplexobj(x) else np.float32)


def bfloat16(x):
    """Rounded to nearest, ties to even."""
    u = x.astype(np.float32).view(np.uint32).astype(np.uint64)
    return ((u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000).astype(np.uint32).view(np.float32)


def pieces(x):
    out, x = [], np.asarray(x, np.float32)
    for _ in range(3):
        h = bfloat16(x)
        out.append(h.astype(np.float64))
        x = x - h
    return out


def product(A, B, kept):
    a, b = pieces(A), pieces(B)
    return sum(a[i] @ b[j] for i, j in kept)


def complex_product(A, B, kept):
    return (product(A.real, B.real, kept) - product(A.imag, B.imag, kept)
            + 1j * (product(A.real, B.imag, kept) + product(A.imag, B.real, kept)))


def test_pieces_are_exact():
    x = np.random.default_rng(0).normal(size=4096).astype(np.float32)
    assert np.array_equal(sum(pieces(x)), x.astype(np.float64))


@pytest.mark.parametrize("K", [1, 31, 97, 1600])
@pytest.mark.parametrize("kept", list(KEPT))
def test_product(K, kept):
    rng = np.random.default_rng(K)
    A = f32(rng.normal(size=(40, K)))
    B = f32(rng.normal(size=(K, 50)) * np.exp(-np.arange(K) / 20)[:, None])
    e = rel2(product(A, B, KEPT[kept]), A.astype(np.float64) @ B.astype(np.float64))
    assert (e < PRODUCT / 20) if kept == "six" else (e > 2 * PRODUCT), e


@pytest.mark.parametrize("N,n", [(17, 9), (48, 17), (97, 23), (200, 40)])
@pytest.mark.parametrize("kept", list(KEPT))
def test_propagation(N, n, kept):
    rng = np.random.default_rng(N)

    def z(*s):
        return rng.normal(size=s) + 1j * rng.normal(size=s)
    P1 = f32(np.eye(N) + 0.1 * z(N, N) / N).astype(np.complex128)
    V, Phi = f32(0.3 / np.sqrt(N) * z(N, N)).astype(np.complex128), z(N, n)

    def run(mul):
        def p1(x):  # the diagonal enters reduced by one
            return mul(P1 - np.eye(N), x) + x
        T = p1(Phi)
        S = T.copy()
        for k in range(1, 7):
            T = (1j / k) * mul(V, T)
            S = S + T
        return p1(S)
    e = rel2(run(lambda a, b: complex_product(f32(a), f32(b), KEPT[kept])), run(np.matmul))
    assert (e < PROPAGATION / 20) if kept == "six" else (e > 1.5 * PROPAGATION), e

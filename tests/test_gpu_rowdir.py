"""The direct-index row kernel (the exact engine's for all but very wide
matrices) against the oracle, bit for bit: values, column order, counts.

Sizes sit at the edges of its parts: rows of B around a multiple of the
lanes of a step (8, 16, 32, 64 and several chunks), column counts around the
32 columns of an index word and the 2^16 columns above which the list of
touched columns changes form, rows without entries, products that are -0.0,
blocks that form their rows in several passes, and batches of systems much
smaller than a block."""
import numpy as np
import pytest

import orc
from bml_amd import generators as G
from bml_amd.ell import Ell
from helpers import assert_ell_identical

pytestmark = pytest.mark.gpu

DTYPES = [np.float32, np.float64, np.complex64, np.complex128]


def square(hip, A, M2, thr):
    ref, rtr = orc.x2(A, M2, thr)
    dA = hip.from_ell(A)
    for _ in range(2):  # without and with the hint of a previous product
        X2 = hip.zero_matrix(A.precision, A.N, M2)
        tr = hip.multiply_x2(dA, X2, thr)
        assert_ell_identical(X2.get(), ref, f"x2 N={A.N}")
    np.testing.assert_allclose(tr, rtr, rtol=1e-5 if A.dtype.itemsize < 8 or
                               A.dtype == np.complex64 else 1e-12, atol=1e-6)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("N,fill", [(1, 1), (31, 6), (32, 8), (33, 9), (64, 17), (97, 32),
                                    (130, 33), (300, 63), (301, 64), (700, 65), (900, 129),
                                    (1100, 193), (1500, 321), (2100, 330)])
def test_square_at_edges(hip, dtype, N, fill):
    square(hip, G.random_ell(N, min(N, fill + 1), fill, 7, dtype), min(N, 2100), 0.05)


@pytest.mark.parametrize("dtype", [np.float32, np.complex128])
def test_several_passes_per_block(hip, dtype):
    """Wide products: what a block's rows touch does not fit beside the rows
    themselves, so they are formed a few at a time (and the first product,
    without a hint, guesses low)."""
    square(hip, G.random_ell(6000, 90, 80, 3, dtype), 5200, 0.9)


def test_many_columns(hip):
    """Above 2^16 columns the list holds slots instead of columns."""
    for N in (65535, 65536, 65537, 70001):
        A = G.random_banded(N=N, M=32, draws=4, band=N // 2, decay=1e9, seed=3)
        ref, _ = orc.x2(A, 256, 1e-3)
        X2 = hip.zero_matrix(A.precision, N, 256)
        hip.multiply_x2(hip.from_ell(A), X2, 1e-3)
        assert_ell_identical(X2.get(), ref, f"x2 N={N}")


@pytest.mark.parametrize("dtype", DTYPES)
def test_negative_zero_products_and_empty_rows(hip, dtype):
    """Stored zeros times negative values give -0.0: such a column is touched
    once and starts as 0.0 + (-0.0) = +0.0.  The matrix starts with rows
    without entries, so a row's first steps can be empty."""
    rng = np.random.default_rng(5)
    N = 333
    A = G.random_ell(N, 24, 20, 11, dtype)
    z = rng.random(A.value.shape) < 0.4
    A.value[z & A.live_mask()] = 0
    A.value[A.live_mask() & (rng.random(A.value.shape) < 0.5)] *= -1
    A.nnz[:70] = 0
    A.nnz[200:203] = 0
    square(hip, A, N, -1.0)
    B = A.copy()
    B.nnz[:] = 0
    ref = orc.ab(A, B, 8, 0.0)
    C = hip.zero_matrix(A.precision, N, 8)
    hip.multiply_AB(hip.from_ell(A), hip.from_ell(B), C, 0.0)
    assert_ell_identical(C.get(), ref, "AB with an empty B")


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_infinities_and_nan(hip, dtype):
    A = G.random_ell(200, 20, 15, 4, dtype)
    A.value[3, 0] = np.inf
    A.value[50, 1] = -np.inf
    A.value[100, 0] = np.nan
    ref, _ = orc.x2(A, 200, 0.01)
    X2 = hip.zero_matrix(A.precision, A.N, 200)
    hip.multiply_x2(hip.from_ell(A), X2, 0.01)
    got = X2.get()
    np.testing.assert_array_equal(got.nnz, ref.nnz)
    m = ref.live_mask()
    np.testing.assert_array_equal(got.index[m], ref.index[m])
    np.testing.assert_array_equal(got.value[m], ref.value[m])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (-2.0, 1.0), (0.0, 0.5), (0.75, -0.5)])
def test_fused_multiply(hip, dtype, alpha, beta):
    for N, fill in ((65, 9), (500, 40), (1300, 150)):
        A = G.random_ell(N, fill + 1, fill, 21, dtype)
        B = G.random_ell(N, fill + 1, fill, 22, dtype)
        C = G.random_ell(N, N, min(N - 1, 90), 23, dtype)
        ref = orc.multiply(A, B, C, alpha, beta, 0.02)
        dC = hip.from_ell(C)
        hip.multiply(hip.from_ell(A), hip.from_ell(B), dC, alpha, beta, 0.02)
        assert_ell_identical(dC.get(), ref, f"multiply N={N} alpha={alpha} beta={beta}")


def test_batch_of_systems_smaller_than_a_block(hip):
    """Rows of one block from several systems, and systems that end early:
    each system's density matrix equals its own solve's."""
    shapes = [(1, 1, 1), (2, 2, 2), (3, 3, 1), (4, 4, 4), (1, 1, 2), (5, 5, 4), (2, 2, 1),
              (9, 9, 9), (3, 3, 3), (2, 2, 2)]
    Hs = [G.lattice_hamiltonian(*s, M=16, hopping=-0.1, disorder=0.01, seed=k)
          for k, s in enumerate(shapes)]
    dH = [hip.from_ell(H) for H in Hs]
    X = [hip.zero_matrix(H.precision, H.N, 512) for H in Hs]
    nocc = [float(H.N // 2) for H in Hs]
    res = hip.sp2_batch(dH, X, nocc, threshold=1e-6, tol=1e-5, maxit=25)
    for H, h, x, n, r in zip(Hs, dH, X, nocc, res):
        Y = hip.zero_matrix(H.precision, H.N, 512)
        one, _ = hip.sp2(h, Y, n, threshold=1e-6, tol=1e-5, maxit=25)
        assert one.iterations == r.iterations
        assert_ell_identical(x.get(), Y.get(), f"system of {H.N}")


def test_overflow_is_reported(hip):
    A = Ell.from_dense(np.ones((40, 40)), 40)
    X2 = hip.zero_matrix(A.precision, 40, 39)
    with pytest.raises(hip.BmlError, match="Number of non-zeroes per row > M"):
        hip.multiply_x2(hip.from_ell(A), X2, 0.0)


@pytest.mark.parametrize("N", [65535, 65536, 65537, 70001])
@pytest.mark.parametrize("dtype", [np.float64, np.complex64])
def test_many_columns_long_rows(hip, dtype, N):
    """Above 2^16 columns the list holds slots instead of columns: rows long
    enough for the direct kernel there."""
    A = G.random_banded(N=N, M=90, draws=36, band=60, seed=3, dtype=dtype)
    assert A.nnz.max() > 64
    square(hip, A, 260, 1e-3)

"""bml_add / bml_add_norm against the oracle, bit for bit, at the sizes where
the row kernel's parts meet: rows around a wavefront's 64 entries, unions
around the width M, widths whose hash table just changes size, rows that are
empty on either side, zero coefficients, and B = A; and temporaries handed
out again between calls of different sizes."""
import numpy as np
import pytest

import orc
from bml_amd import generators as G
from helpers import assert_ell_identical

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.complex64, np.complex128])
@pytest.mark.parametrize("N,fa,fb,M", [(1, 1, 1, 2), (40, 5, 9, 21), (65, 20, 40, 65),
                                       (300, 63, 64, 149), (300, 64, 65, 150), (500, 130, 100, 320),
                                       (900, 200, 3, 321), (700, 1, 300, 700)])
def test_add_at_edges(hip, dtype, N, fa, fb, M):
    A = G.random_ell(N, M, min(fa, N - 1) if N > 1 else 0, 3, dtype)
    B = G.random_ell(N, min(fb, N) + 1, min(fb, N), 4, dtype)
    A.nnz[:: 7] = 0
    B.nnz[:: 5] = 0
    for alpha, beta in ((1.0, 1.0), (2.0, -1.0), (0.0, 1.5), (0.7, 0.0)):
        ref = orc.add(A, B, alpha, beta, 0.1)
        dA = hip.from_ell(A)
        hip.add(dA, hip.from_ell(B), alpha, beta, 0.1)
        assert_ell_identical(dA.get(), ref, f"add {alpha} {beta}")
        ref, n = orc.add_norm(A, B, alpha, beta, 0.1)
        dA = hip.from_ell(A)
        got = hip.add_norm(dA, hip.from_ell(B), alpha, beta, 0.1)
        assert_ell_identical(dA.get(), ref, f"add_norm {alpha} {beta}")
        # the oracle sums in double over rows in turn
        np.testing.assert_allclose(got, n, rtol=1e-12, atol=1e-12)


def test_add_to_itself(hip):
    A = G.random_ell(300, 130, 100, 9)
    ref = orc.add(A, A.copy(), 1.0, -0.25, 0.1)
    dA = hip.from_ell(A)
    hip.add(dA, dA, 1.0, -0.25, 0.1)
    assert_ell_identical(dA.get(), ref, "A + A")


def test_temporaries_between_sizes(hip):
    """A multiply whose output is an operand forms its product in a temporary;
    small and large ones in turn give the same as alone."""
    first = {}
    for rep in range(3):
        for N, f in ((400, 10), (60, 20), (1500, 30), (400, 12)):
            A = G.random_ell(N, min(N, 900), f, N + f)
            ref = first.get((N, f))
            dA = hip.from_ell(A)
            hip.multiply(dA, hip.from_ell(A), dA, 1.0, 0.5, 0.01)
            got = dA.get()
            if ref is None:
                first[(N, f)] = got
            else:
                assert_ell_identical(got, ref, f"N={N} rep {rep}")

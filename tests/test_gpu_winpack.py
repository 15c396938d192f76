"""Order of a packed row's entries inside a window.

The pack deals a row's entries over the 16 column classes mod 16 in turn.  At
its edges: rows whose entries all lie in one class, rows with every column,
rows of one entry, empty rows, and a last window that is not full.  Elements
are small integers, so every sum is exact and the result equal to the
oracle's, entry for entry.
"""
import numpy as np
import pytest

import orc
from bml_amd.ell import Ell
from helpers import DTYPES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 2, 4])
@pytest.mark.parametrize("dtype", DTYPES)
def test_packed_classes(hip, monkeypatch, dtype, rows):
    N = 1100
    rng = np.random.default_rng(5)
    A = Ell.zeros(N, N, dtype)
    for i in range(N):
        cols = [np.arange(3, N, 16), np.arange(N), np.array([i]), np.array([], int),
                np.sort(rng.choice(N, 37, replace=False))][i % 5]
        n = len(cols)
        v = rng.choice([-2.0, -1.0, 1.0, 2.0], n)
        if np.issubdtype(np.dtype(dtype), np.complexfloating):
            v = v + 1j * rng.choice([-1.0, 0.0, 1.0], n)
        A.index[i, :n], A.value[i, :n], A.nnz[i] = cols, v, n
    ref, rtr = orc.x2(A, N, 0.5)
    monkeypatch.setenv("BML_HIP_WIN_ROWS", str(rows))
    hip.set_row_engine(hip.ROW_ENGINE_WINDOW)
    try:
        X2 = hip.zero_matrix(A.precision, N, N)
        tr = hip.multiply_x2(hip.from_ell(A), X2, 0.5)
    finally:
        hip.set_row_engine(hip.ROW_ENGINE_EXACT)
    np.testing.assert_array_equal(X2.get().to_dense(), ref.to_dense())
    assert tuple(tr) == tuple(rtr)

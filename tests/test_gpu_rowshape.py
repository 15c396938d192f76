"""The product's device entry with launch shapes that no host rule gives: a
direct-index shape whose LDS holds no row, or whose index has too few words
for the matrix, hands its rows to the global-table pass and the product is
still whole."""
import ctypes as C

import numpy as np
import pytest

import orc
from bml_amd import generators as G
from helpers import assert_ell_identical

pytestmark = pytest.mark.gpu


class Args(C.Structure):
    """bmlhip_spgemm_args (csrc/bmlhip_abi.h)."""
    _fields_ = ([(n, C.c_int) for n in ("prec", "kind", "N", "MA", "MB", "MC")] +
                [(n, C.c_void_p) for n in ("Av", "Ai", "An", "Bv", "Bi", "Bn", "Cv", "Ci", "Cn")] +
                [("threshold", C.c_double)] +
                [(n, C.c_int) for n in ("group", "table", "bucket", "remap", "waves", "engine",
                                        "sym", "wbits", "wrows")] +
                [("skip", C.c_void_p), ("batch", C.c_void_p), ("ws", C.c_void_p),
                 ("ws_bytes", C.c_size_t), ("fuse", C.c_int), ("alpha", C.c_double),
                 ("beta", C.c_double), ("sp2", C.c_void_p)])


DIRECT, LIST, DENSE, OWN = 3, 0, 1, 2


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("mode,table,words_of", [(DENSE, 6144, 1000), (DENSE, 40960, 500),
                                                 (DENSE, 40960, 1000), (LIST, 6144, 1000),
                                                 (OWN, 6144, 1000), (LIST, 40960, 500)])
def test_rows_without_room_go_to_the_global_pass(hip, dtype, mode, table, words_of):
    A = G.random_ell(1000, 40, 33, 5, dtype)
    ref, _ = orc.x2(A, 1000, 1e-3)
    X, X2 = hip.from_ell(A), hip.zero_matrix(A.precision, 1000, 1000)
    x, y = X._s, X2._s
    a = Args(prec=A.precision, kind=0, N=1000, MA=x.M, MB=x.M, MC=y.M, Av=x.value, Ai=x.index,
             An=x.nnz, Bv=x.value, Bi=x.index, Bn=x.nnz, Cv=y.value, Ci=y.index, Cn=y.nnz,
             threshold=1e-3, group=64, table=table, bucket=1, waves=1, engine=DIRECT,
             wbits=mode, wrows=words_of)
    assert hip.lib().bmlhip_spgemm(C.byref(a)) == 0
    hip.synchronize()
    assert_ell_identical(X2.get(), ref, f"mode {mode}, {table} bytes, index of {words_of}")

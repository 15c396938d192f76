"""The status block between operations.  An operation that begins (it may end
in an error before its last launch) leaves the block in use: the next one
starts on a cleared block, and a fetch reads what the block holds, not the
copy that an earlier operation handed to the host."""
import ctypes as C

import numpy as np
import pytest

import orc
from bml_amd import generators as G
from helpers import assert_ell_identical

pytestmark = pytest.mark.gpu

MAX_NNZ = 12  # byte offset in bmlhip_status (csrc/bmlhip_abi.h)


def _begin_and_stop(lib, value):
    """What an operation leaves that stops after filling in its longest row."""
    assert lib.bmlhip_status_ready() == 0
    lib.bmlhip_status_dev.restype = C.c_void_p
    v = C.c_int(value)
    assert lib.bmlhip_h2d(C.c_void_p(lib.bmlhip_status_dev() + MAX_NNZ), C.byref(v),
                          C.c_size_t(4)) == 0


def test_operation_after_one_that_stopped_half_way(hip):
    lib = hip.lib()
    A = G.random_banded(N=700, M=64, draws=8, band=64, seed=2)
    ref, _ = orc.x2(A, 400, 1e-5)
    X = hip.from_ell(A)
    for k in range(2):
        X2 = hip.zero_matrix(A.precision, A.N, 400)
        hip.multiply_x2(X, X2, 1e-5)  # ends with a clear block and a copy on the host
        _begin_and_stop(lib, 4567)
        st = (C.c_int * 256)()
        assert lib.bmlhip_status_fetch(st) == 0
        assert st[MAX_NNZ // 4] == 4567
        _begin_and_stop(lib, 4567)
        X2 = hip.zero_matrix(A.precision, A.N, 400)
        if k:
            hip.multiply_AB(X, X, X2, 1e-5)
        else:
            hip.multiply_x2(X, X2, 1e-5)
        assert X2.row_stats()[0] == int(np.max(ref.nnz))
        assert_ell_identical(X2.get(), ref, "after a stopped operation")

"""The device memory that calls keep for their temporaries: it can be given
back, and calls before and after give the same result."""
import ctypes as C

import numpy as np
import pytest

import orc
from bml_amd import generators as G
from helpers import assert_ell_identical

pytestmark = pytest.mark.gpu


def _free_bytes(hip):
    hip.synchronize()
    free, total = C.c_size_t(), C.c_size_t()
    rt = C.CDLL("libamdhip64.so")
    assert rt.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_kept_memory_is_given_back(hip):
    """C <- A C into its operand at N x M = 512 MB of values: the temporary's
    arrays stay with the library until they are released."""
    N, M = 1 << 16, 1 << 10
    A = G.random_banded(N=N, M=32, draws=4, band=100, seed=1)
    dA = hip.from_ell(A)
    got = []
    for k in range(3):  # the first product sizes the library's scratch as well
        Cm = hip.from_ell(A, M)
        hip.release_temporaries()
        before = _free_bytes(hip)
        hip.multiply(dA, Cm, Cm, 1.0, 0.0, 1e-6)
        if k:
            assert before - _free_bytes(hip) >= 8 * N * M  # its values at least
            hip.release_temporaries()
            assert _free_bytes(hip) >= before
        got.append(Cm.get())
        Cm.free()
    for g in got[1:]:
        assert_ell_identical(g, got[0], "before and after the release")
    ref = orc.ab(A, A, M, 1e-6)
    np.testing.assert_array_equal(got[0].nnz, ref.nnz)


def test_more_blocks_than_are_kept(hip):
    """Temporaries past the number that is kept (64) are freed; those kept are
    handed out again, each to one caller."""
    lib = hip.lib()
    for _ in range(2):
        held = []
        for k in range(80):
            p = C.c_void_p()
            assert lib.bmlhip_temp_malloc(C.byref(p), C.c_size_t(1000 * (k % 7) + k)) == 0
            held.append(p.value)
        assert len(set(held)) == 80
        for p in held:
            lib.bmlhip_temp_free(C.c_void_p(p))
    hip.release_temporaries()

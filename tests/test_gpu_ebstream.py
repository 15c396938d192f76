"""FP64 block products on the matrix cores at the edges of their work queues.

The block rows' batches are found through a prefix over at most 2048 groups of
rows and dealt from 8 queues: fewer block rows than queues, a last group that
is not full, two and three rows in a group, empty rows between full ones, and
rows whose dropped blocks are compacted.  Against the exact oracle: a sum has
at most 64 terms of at most 1, so its two orders differ by less than
64 * 64 * 2^-53 = 4.6e-13, and the largest element is above 1.
"""
import numpy as np
import pytest

import orc
from bml_amd import generators as G
from helpers import rel_close
from test_gpu_ellblock import blocks_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("NB", [1, 5, 67, 2047, 2049, 4100])
def test_queues_and_row_groups(hip, NB):
    bsize = np.resize([32, 1, 3, 17, 2, 1, 1], NB)
    M, MC = min(NB, 2), min(NB, 4)
    A = G.random_blk(bsize, M, 1, NB, bmax=32)
    B = G.random_blk(bsize, M, 1, NB + 1, bmax=32)
    if NB > 60:
        for X in (A, B):
            X.nnzb[20:60] = 0
            X.nnzb[-1] = 0
    hip.set_block_engine(1)
    try:
        dA, dB = hip.from_blk(A), hip.from_blk(B)
        X2 = hip.block_matrix(A.precision, A.bsize, MC)
        C = hip.block_matrix(A.precision, A.bsize, MC)
        tr = hip.eb_multiply_x2(dA, X2, 0.5)
        hip.eb_multiply_AB(dA, dB, C, 0.5)
    finally:
        hip.set_block_engine(hip.BLOCK_ENGINE_AUTO)
    ref, otr = orc.eb_x2(A, MC, 0.5)
    blocks_close(X2.get(32), ref, 1e-12, "x2")
    assert rel_close(tr[0], otr[0], 1e-12) and rel_close(tr[1], otr[1], 1e-12)
    blocks_close(C.get(32), orc.eb_ab(A, B, MC, 0.5), 1e-12, "ab")

"""The search for a launch shape of the direct-index row product, and the
shapes it reads back from its cache (host logic, no GPU): the measurement is
replaced by one that times nothing and notes the candidates."""
import ctypes as C
import os
import subprocess
import sys

import pytest

from bml_amd import hip

EXACT, DIRECT = 0, 3  # engines of a launch shape
SINGLE, DOUBLE, SINGLE_C, DOUBLE_C = 1, 2, 3, 4
ELEM = {SINGLE: 4, DOUBLE: 8, SINGLE_C: 8, DOUBLE_C: 16}
SQUARE = 1


class Shape(C.Structure):
    _fields_ = [(n, C.c_int) for n in ("group", "table", "bucket", "remap", "waves", "engine",
                                       "wbits", "wrows")]

    def key(self):
        return tuple(getattr(self, n) for n, _ in self._fields_)


MEASURE = C.CFUNCTYPE(C.c_int, C.POINTER(Shape), C.c_void_p, C.POINTER(C.c_double))


def copy_of(sh):
    out = Shape()
    C.pointer(out)[0] = sh
    return out


def search(prec, N, n, touched=0, ms=lambda sh: 1.0):
    """bmlh_tuned_spgemm for an N x N square of rows of n entries: the shape
    taken and the candidates measured."""
    tried = []

    @MEASURE
    def measure(sh, ctx, out):
        tried.append(copy_of(sh[0]))
        out[0] = ms(sh[0])
        return 0

    out = Shape()
    hip.lib().bmlh_tuned_spgemm(prec, N, n, n, touched, n if touched else 0, SQUARE, C.byref(out),
                                measure, None)
    return out, tried


def analytic(prec, N, n, touched=0):
    out = Shape()
    hip.lib().bmlh_pick_spgemm(prec, N, N, n, n, touched, n if touched else 0, SQUARE, C.byref(out))
    return out


@pytest.fixture
def tuner():
    hip.autotune_clear()
    hip.set_autotune(True, "")
    yield
    hip.set_autotune(False, "")
    hip.autotune_clear()


def test_search_from_one_wavefront_ends():
    """Shapes of one wavefront (few rows, or long ones) are searched too."""
    code = ("import test_autotune_direct as t\n"
            "t.hip.set_autotune(True, '')\n"
            "for N in (100, 300, 500, 511, 4096):\n"
            "    t.hip.autotune_clear()\n"
            "    sh, tried = t.search(t.DOUBLE, N, 33)\n"
            "    assert sh.engine == t.DIRECT and tried, N\n"
            "    assert {1, 2} <= {s.waves for s in tried}, N\n")
    here = os.path.dirname(os.path.abspath(__file__))
    env = dict(os.environ, PYTHONPATH=os.pathsep.join([here, os.path.dirname(here)]))
    subprocess.run([sys.executable, "-c", code], check=True, timeout=60, env=env)


def rows_held(prec, sh, D):
    """Rows of D columns that the kernel's LDS holds at once: the index words
    and 48 bytes, the columns' list (2^16 columns or more), a spare slot per
    lane, and per row its sums and its 16-bit list."""
    def up(b):
        return (b + 15) // 16 * 16
    head = up(8 * (sh.wrows // 32 + 2)) + 48
    fixed = (up(4 * D) if sh.wrows > 65536 else 0) + 64 * sh.waves * ELEM[prec]
    per_row = up(D * ELEM[prec]) + up(2 * D)
    return max(0, sh.table - head - fixed) // per_row


DENSE = 1  # numbering: a column is its own slot


@pytest.mark.parametrize("prec", sorted(ELEM))
def test_every_candidate_holds_a_row(tuner, prec):
    """A shape whose LDS holds no row hands every row to the global-table
    pass; it must not be measured, however fast that is."""
    for N in list(range(60, 3000, 97)) + [870, 946, 1000, 1072, 1716, 2817, 2892, 4096, 30000]:
        for n, touched in ((9, 0), (9, 60), (33, 0), (33, 300), (63, 0), (63, min(N, 1500))):
            hip.autotune_clear()
            sh, tried = search(prec, N, n, touched, ms=lambda s: float(s.waves))
            for c in tried:
                if c.engine != DIRECT:
                    continue
                D = N if c.wbits == DENSE else min(touched or 1, N)
                assert rows_held(prec, c, D) >= 1, (N, n, touched, c.key())
                assert c.table <= 160 * 1024 and c.wrows == N


@pytest.mark.parametrize("prec,N,N2,n", [(SINGLE, 1300, 1400, 33), (DOUBLE, 900, 1000, 33),
                                         (DOUBLE, 870, 1020, 40), (SINGLE, 1500, 1700, 33),
                                         (DOUBLE_C, 900, 1000, 33), (DOUBLE, 20000, 22000, 33)])
def test_cached_shape_fits_the_call(tuner, prec, N, N2, n):
    """An entry of the table serves sizes near its own; the shape taken from
    it is the call's own size's, in both orders."""
    for first, second in ((N, N2), (N2, N)):
        hip.autotune_clear()
        assert search(prec, first, n, ms=lambda s: float(s.waves))[1]
        sh, tried = search(prec, second, n)
        assert not tried, "not the same key"
        assert sh.engine == DIRECT and sh.wrows == second
        D = second if sh.wbits == DENSE else min(1000, second)
        assert rows_held(prec, sh, D) >= 1


def test_direct_entry_of_a_file_is_not_taken_as_it_stands(tmp_path):
    """Wavefronts that do not fit, an index for other columns or an LDS size
    from a cache file never reach the kernel."""
    p = tmp_path / "tune.txt"
    hip.autotune_clear()
    hip.set_autotune(True, str(p))
    try:
        search(DOUBLE, 1000, 33)
        key = p.read_text().split()[0]
        for waves in (0, 1, 2, 7, 9, 4096, -3):
            p.write_text(f"{key} 64 2048 1 0 {waves} 3 1 17 0.001\n")
            hip.autotune_clear()
            hip.set_autotune(True, str(p))
            sh, tried = search(DOUBLE, 1000, 33)
            assert not tried
            assert sh.engine == DIRECT and sh.wrows == 1000 and 1 <= sh.waves <= 8
            assert rows_held(DOUBLE, sh, 1000) >= 1
    finally:
        hip.set_autotune(False, "")
        hip.autotune_clear()


@pytest.mark.parametrize("prec", sorted(ELEM))
def test_a_work_queue_gets_the_hash_kernels(prec):
    """Rows taken from a batch's work queue (BML_HIP_BATCH_QUEUE=1): the
    direct kernel, whose blocks form consecutive rows, does not read it."""
    queue = 4
    for N, span, n, touched in ((3000, 900, 7, 0), (38394, 8190, 63, 500), (512, 64, 9, 30)):
        sh, out = Shape(), Shape()
        hip.lib().bmlh_pick_spgemm(prec, N, span, n, n, touched, n, SQUARE, C.byref(sh))
        assert sh.engine == DIRECT
        hip.lib().bmlh_pick_spgemm(prec, N, span, n, n, touched, n, SQUARE | queue, C.byref(out))
        assert out.engine == EXACT and out.group in (8, 16, 32, 64) and out.table >= 64


# (precision, N, entries a row, distinct columns a row of an earlier product
# or 0, direct kernel): the sides of each line of the rule
CROSSOVER = [
    (DOUBLE, 16384, 7, 0, True), (DOUBLE, 16385, 7, 0, False), (DOUBLE, 16385, 32, 0, False),
    (DOUBLE, 17150, 7, 25, True), (DOUBLE, 17151, 7, 25, False), (DOUBLE, 17151, 7, 43, False),
    (DOUBLE, 110592, 25, 87, True), (DOUBLE, 262144, 25, 87, False), (DOUBLE, 262144, 7, 25, False),
    (DOUBLE, 32000, 12, 133, False), (DOUBLE, 32000, 12, 99, True),
    (DOUBLE, 65536, 33, 0, True), (DOUBLE, 65537, 33, 0, False), (DOUBLE, 65537, 64, 0, False),
    (DOUBLE, 131072, 45, 639, True), (DOUBLE, 131073, 45, 639, False),
    (DOUBLE, 262144, 45, 1981, True), (SINGLE, 262144, 45, 1981, False),
    (DOUBLE_C, 100000, 64, 0, False), (DOUBLE_C, 100000, 64, 949, True),
    (DOUBLE, 70001, 65, 0, True), (DOUBLE, 262144, 87, 260, False), (DOUBLE, 262144, 87, 0, True),
    (DOUBLE, 262144, 185, 1177, True), (DOUBLE_C, 262144, 322, 2300, False),
    (DOUBLE_C, 175616, 322, 2300, True), (SINGLE_C, 262144, 322, 2300, True),
]


@pytest.mark.parametrize("prec,N,n,touched,direct", CROSSOVER)
def test_crossover_of_the_two_exact_kernels(prec, N, n, touched, direct):
    """Large matrices of short rows, and short rows all over the matrix, stay
    on the hash kernels."""
    assert (analytic(prec, N, n, touched).engine == DIRECT) == direct


@pytest.mark.parametrize("prec", sorted(ELEM))
def test_lds_for_rows_not_known_to_share_columns(prec):
    """Rows of more than 64 entries whose product is not known: LDS for 6500
    columns (or all that they can touch), or as many as fit beside the
    index.  Short rows: for the columns of every row of the block."""
    for N, n in ((3500, 100), (8000, 100), (16384, 80), (25000, 140), (100000, 90)):
        sh = analytic(prec, N, n)
        room = (160 * 1024 - 8 * (N // 32 + 2)) // (ELEM[prec] + 2) - 200
        if N > 65536:
            room = room * 2 // 3
        assert sh.engine == DIRECT
        assert rows_held(prec, sh, min(N, n * n, 6500, room)) >= 1, (N, n, sh.key())
    for N, n, touched in ((12000, 7, 0), (16384, 12, 133), (16384, 16, 241), (9000, 9, 75)):
        sh = analytic(prec, N, n, touched)
        rb = sh.waves * (64 // sh.group)
        assert sh.engine == DIRECT and sh.group <= 16
        assert rows_held(prec, sh, rb * (touched or n * n)) >= rb, (N, n, sh.key())


@pytest.mark.parametrize("prec", sorted(ELEM))
@pytest.mark.parametrize("N,n", [(576, 256), (20000, 9), (48000, 7), (110592, 256), (3000, 8)])
def test_first_iterate_of_a_solve(prec, N, n):
    """A solve's iterate before its first product is known: the direct kernel
    up to 2^17 columns, with LDS for 3000 columns at most, and the cache key
    of any other square."""
    solve = 8
    sh, x2 = Shape(), analytic(prec, N, n)
    hip.lib().bmlh_pick_spgemm(prec, N, N, n, n, 0, 0, SQUARE | solve, C.byref(sh))
    assert sh.engine == DIRECT and sh.wrows == N
    if x2.engine == DIRECT:
        assert sh.table <= x2.table
    hip.lib().bmlh_pick_spgemm(prec, 262144, 262144, 9, 9, 0, 0, SQUARE | solve, C.byref(sh))
    assert sh.engine == EXACT


def test_count_of_the_matrix_it_was_made_from():
    """A negative count is an earlier matrix's (before an add, or the factor
    of a square): LDS for the columns to expect by it, and the crossover's side
    of rows that share columns."""
    def pick(prec, N, n, touched, hint):
        sh = Shape()
        hip.lib().bmlh_pick_spgemm(prec, N, N, n, n, touched, hint, SQUARE, C.byref(sh))
        return sh

    never, seen = pick(DOUBLE, 32768, 148, 0, 0), pick(DOUBLE, 32768, 148, -1100, 140)
    assert never.engine == seen.engine == DIRECT
    assert rows_held(DOUBLE, never, 6500) >= 1
    # rows in flight per CU: the LDS is not kept for 6500 columns a row
    assert seen.waves * (160 * 1024 // seen.table) > never.waves * (160 * 1024 // never.table)
    wide = pick(DOUBLE, 16384, 80, -5300, 80)
    assert wide.engine == DIRECT and rows_held(DOUBLE, wide, 5300) >= 1
    grown = pick(DOUBLE, 16384, 88, -5300, 80)
    assert grown.engine == DIRECT and rows_held(DOUBLE, grown, 5830) >= 1
    assert pick(DOUBLE, 32768, 25, 0, 0).engine == EXACT
    assert pick(DOUBLE, 32768, 25, -90, 25).engine == DIRECT
    assert pick(DOUBLE, 32768, 25, -600, 25).engine == EXACT

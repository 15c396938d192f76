/*
 * Launch-shape choice for the ELLPACK row-product kernels.  The exact engine
 * takes the direct-index kernel where it is the faster one and its index fits
 * (direct_wins and pick_direct below); what follows is the hash kernels'
 * choice.
 *
 * group (lanes per output row) follows the length of the rows of B that a
 * step streams: a step holds three GROUP-wide chunks of a row of B in
 * registers, so GROUP is the smallest power of two with 3*GROUP >= max_b and
 * a 64-lane wavefront carries 64/GROUP output rows.
 *
 * The LDS table holds a row's distinct columns.  est, the largest distinct
 * count per row, comes from the previous product of the same matrix when
 * known (scaled by the growth of its rows since), else from the bound
 * min(N, max_a*max_b).
 * The table gets max(3/2 est, est + max_b) + 64 slots in 4-slot buckets: a
 * row stops (and goes to the global-table pass) once count + (row length of
 * B) could pass the table, and at ~2/3 load the probe rounds per step (the
 * longest probe among the 3*64 lanes of a step) stay low; a smaller table
 * buys occupancy but costs more rounds (on the 32^3 lattice X^2, 1177
 * distinct columns per row, 1792 slots ran 1.4x faster than 1536 and as
 * fast as 2048).  One wavefront's tables are capped at 32 KiB so at least
 * five wavefronts share a CU.  Rows that outgrow the table are finished by the global-table
 * pass, so the cap costs speed, never correctness.
 *
 * Environment overrides: BML_HIP_GROUP, BML_HIP_TABLE, BML_HIP_BUCKET,
 * BML_HIP_LDS_BUDGET (bytes per wavefront), BML_HIP_XCD_REMAP (0/1).
 */
#include "bml_hip_tune.h"
#include "bml_hip_host.h"

#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

/* Where the direct-index kernel is the faster one.  Every block of it pays
 * for an index of all reachable columns (8 bytes of LDS and a share of a scan
 * per 32 of them), and rows that share a block hold a sum for each column
 * that any of them touches; the hash kernels pay per product.  Measured with
 * both kernels on random rows near the diagonal and all over the matrix, on
 * lattice Hamiltonians and iterates, in three element types (us, double
 * unless said, hash and direct):
 *
 * - up to 2^14 columns the index is small: direct, 2 to 4 times as fast from
 *   9 entries a row on (N = 16384: 31 near the diagonal 444 and 121, all
 *   over 590 and 323), level on shorter ones;
 * - rows of more than 64 entries: direct (N = 25000, 100 near the diagonal
 *   9878 and 2540; 64^3 lattice, 185 a row 48500 and 31100).  Above 2^17
 *   columns the index leaves few rows per CU: with the counts of an earlier
 *   product known, so that the hash table has its right size, it wins below
 *   span / 32 products a row (64^3, 87 a row: 8920 and 9400) and where less
 *   than two and a half rows fit beside the index (complex, 322 a row, 64^3:
 *   179 ms and 243, 56^3: 181 and 84);
 * - 33 to 64 entries: direct up to 2^16 columns (N = 65000, 45 near the
 *   diagonal 1560 and 850, all over 10000 and 6950), above that on rows known
 *   to share columns, up to 2^17 (N = 262144, 45: 6160 and 6290; not known,
 *   complex, N = 100000, 64: 7530 and 11430), and where the row does not fit
 *   the hash kernel's table (all over, N = 262144, 45: 42400 and 32800);
 * - up to 32 entries, several rows to a wavefront: only on rows known to
 *   share columns (fewer distinct ones than 7/10 of the products), up to
 *   2^17 columns and 350 for each product of a row (48^3 lattice: 25 a row
 *   875 and 690, 7 a row 151 and 333; all over, N = 32000, 12: 148 and 269).
 *
 * A solve's iterate that has not been squared yet: direct up to 2^17 columns.
 * The shape serves until the counts are polled, and the rows grow meanwhile
 * (five systems of up to 27000 rows, a poll every 3 iterations: 117 ms, with
 * the hash kernels until the first poll 167). */
static int direct_wins(size_t es, int span, int max_a, int max_b, long long est, int known,
                       int solve)
{
    const long long products = (long long) max_a * max_b;
    if (span <= 16384 || (solve && !known && span <= 131072))
        return 1;
    const int shared = known && 10 * est <= 7 * products;
    if (max_b > 64)
        return !known || span <= 131072 ||
               (32 * products >= span &&
                5 * est * (long long) (es + 2) <= 2 * (160 * 1024 - span / 4));
    if (max_b > 32) {
        if (span <= 65536 || (known && est * 5 / 4 * (long long) (es + 6) > 32 * 1024))
            return 1;
        return shared && span <= 131072;
    }
    return shared && span <= 131072 && 350 * products >= span;
}

/* Shape of the direct-index kernel (hip/rowdir.hip), 0 when its LDS cannot
 * hold one row.
 *
 * GROUP lanes per row: enough for a row of B in one chunk (rows of up to 8,
 * 16 or 32 entries share a wavefront), wider while the matrix has too few
 * rows to fill the GPU's 1024 SIMDs twice over; up to five 64-lane chunks a
 * step.  W wavefronts per block and the blocks per CU follow the LDS: the
 * block needs 8 bytes per 32 reachable columns, and each row sizeof(T) + 2 per
 * column that any row of the block touches (15% more for each further row: on
 * a lattice a step along the fast axis adds the ball's cross-section, near
 * the diagonal less; as many again where up to 16 entries share a wavefront
 * with other rows and are not known to share columns with them); the W with the most wavefronts per CU is
 * taken, the larger of equals (its rows share more of the index).  A block
 * whose rows touch more than that forms them in several passes; a row that
 * does not fit alone is left to the global-table pass.  Without a hint the
 * bound min(span, max_a * max_b) is mostly far above the truth: 3000 columns
 * are provided for, 6500 for rows of more than 64 entries, whose hash tables
 * held as many (double, N = 16384, 80 entries all over: 20.8 ms with 3000,
 * 4.2 with 6500, the hash kernel 8.7; near the diagonal 0.99, 1.75, 5.3).
 * seen: the distinct columns to expect from the count of the matrix that this
 * one was made from (a client's loop of x2 and add_norm), 0 without one; the
 * LDS is for 9/8 of them, or 3000.  solve: the rows are a solve's first iterate, far shorter than max_a, and
 * 3000 columns serve them and what grows from them until they are known (32^3
 * lattice, M = 256: 334 us, with 6500 606).
 * Rows so short that all columns fit are indexed by the column itself.
 * waves != 0 asks for the shape of that many wavefronts per block (the
 * autotuner's candidates; fewer rows than CUs then do not rule it out). */
static int pick_direct(size_t es, int N, int span, int max_a, int max_b, long long est,
                       int known, long long seen, int grows, int solve, int waves,
                       bmlh_spgemm_shape *out)
{
    if (N <= 0 || span <= 0)
        return 0;
    if (!direct_wins(es, span, max_a, max_b, est, known, solve) &&
        !(seen && max_b <= 64 && direct_wins(es, span, max_a, max_b, seen, 1, solve)))
        return 0;
    int g = 8;
    while (g < 64 && (g < max_b || (long long) N * g < 64 * 2048))
        g <<= 1;
    int nch = (max_b + g - 1) / g;
    if (nch > 5) {
        /* several steps a row: as many as rows a tenth shorter than the
         * longest take (24^3 complex square, 279 entries a row, 322 at most:
         * one step of five chunks 6.8 ms, two of three 7.7) */
        const int most = (max_b * 9 / 10 + g - 1) / g, parts = (most + 4) / 5;
        nch = (most + parts - 1) / parts;
    }
    if (nch < 1)
        nch = 1;
    if (est > span)
        est = span;
    const long long per = (long long) es + 2;
    const int dense = span * per <= 6 * 1024 || (2 * est >= span && span * per <= 20 * 1024);
    const int shared = known || seen ? 10 * (known ? est : seen) <= 7 * (long long) max_a * max_b
                                     : solve;
    const long long words = span / 32 + 2;
    const long long cu = 160 * 1024;
    if (!known) {
        /* at most what the LDS holds beside the index */
        const long long room = (cu - 8 * words - 64 * (long long) es - 192) /
                                   (per + (span > 65536 ? 4 : 0)) - 40;
        long long most = seen ? seen * 9 / 8 : (max_b > 64 && !solve ? 6500 : 3000);
        if (most > room)
            most = room;
        if (most < 3000)
            most = 3000;
        if (est > most)
            est = most;
    }
    /* growing rows touch more columns for their length each time (a ball of
     * radius r squared has radius 2r) */
    if (grows && est + est / 2 <= span)
        est += est / 2;
    const int more = g <= 16 && !shared ? 100 : 15;
    int best = 0, best_waves = 0;
    long long best_lds = 0;
    for (int w = 8; w >= 1; w--) {
        const int rb = w * (64 / g);
        if (waves ? w != waves : w > 1 && (long long) N < 256ll * rb)
            continue; /* fewer blocks than CUs */
        long long D = est + est * more * (rb - 1) / 100 + 32;
        if (dense || D > span)
            D = span;
        long long need = 8 * words + 64 + (span > 65536 ? 4 * D + 16 : 0) + 64ll * w * (long long) es +
                         rb * (D * per + 32);
        /* the lists of the symbolic phase */
        const long long list = (long long) rb * max_a < span ? (long long) rb * max_a : span;
        const long long low = 12 * words + 128 + 4 * list + 1024;
        if (need < low)
            need = low;
        if (need > cu)
            continue;
        long long k = cu / ((need + 1279) / 1280 * 1280);
        if (k * w > 16)
            k = 16 / w;
        if (k * w > best_waves) {
            best = w;
            best_waves = (int) (k * w);
            /* the whole share of the CU (allocated in 1280 bytes): est may
             * be low, above all while rows grow */
            best_lds = cu / k / 1280 * 1280;
        }
    }
    if (!best)
        return 0;
    out->engine = BMLHIP_ROW_DIRECT;
    out->group = g;
    out->bucket = nch;
    out->waves = best;
    out->table = (int) best_lds;
    out->wrows = span;
    /* two rows share too few rows of B to pay for listing them */
    out->wbits = dense ? BMLHIP_DIR_DENSE
                       : (best * (64 / g) <= 2 && max_a <= 96 ? BMLHIP_DIR_OWN : BMLHIP_DIR_LIST);
    if (best * (64 / g) == 1 && !dense)
        out->wbits = BMLHIP_DIR_OWN;
    return 1;
}

static int shape_from_env(void)
{
    static const char *const names[] = { "BML_HIP_GROUP", "BML_HIP_TABLE", "BML_HIP_BUCKET",
                                         "BML_HIP_WAVES", "BML_HIP_LDS_BUDGET" };
    for (size_t k = 0; k < sizeof names / sizeof names[0]; k++)
        if (getenv(names[k]))
            return 1;
    return 0;
}

/* The distinct columns of a row when rows of up to hint_max_a entries had
 * `touched`: they grow about as the rows' length does. */
static long long distinct(int touched, int max_a, int hint_max_a, long long bound)
{
    const double grow = hint_max_a > 0 && max_a > hint_max_a ? (double) max_a / hint_max_a : 1.0;
    const long long est = (long long) (touched * grow) + 1;
    return est > bound ? bound : est;
}

/* bmlh_pick_spgemm; direct_waves != 0: where it takes the direct kernel, its
 * shape of that many wavefronts per block */
static void pick(int precision, int N, int span, int max_a, int max_b, int touched_hint,
                 int hint_max_a, int flags, int direct_waves, bmlh_spgemm_shape *out)
{
    const int square = flags & BMLH_PICK_SQUARE;
    int g = 8;
    while (g < 64 && 3 * g < max_b)
        g <<= 1;
    long long bound = (long long) max_a * (long long) max_b;
    if (bound > N)
        bound = N;
    long long est = bound;
    if (touched_hint > 0)
        est = distinct(touched_hint, max_a, hint_max_a, bound);
    long long need = est * 3 / 2;
    if (need < est + max_b)
        need = est + max_b;
    need = (need + 64 + 63) & ~63ll;
    const long long slot = (long long) bmlh_elem_size(precision) + 4 + 2;
    const char *eb = getenv("BML_HIP_LDS_BUDGET");
    const long long budget = eb ? atoll(eb) : 32 * 1024;
    /* more rows per wavefront only while their tables fit */
    while (g < 64 && (64 / g) * (need + 8 + g) * slot > budget)
        g <<= 1;
    /* The kernel is latency bound, so its speed follows the wavefronts
     * resident per CU, which the LDS sets (160 KiB per CU, allocated in
     * 1 KiB granules here).  Take the largest table that still keeps the
     * most wavefronts with at least `need` slots: on the 32^3 lattice X^2
     * (1177 distinct columns per row, need 1856) 1792 slots (6 wavefronts
     * per CU) ran 4.8 ms, 1856 slots (5) 5.4 ms. */
    const int R = 64 / g;
    const long long pad = 8 + g;
    long long t = 0;
    for (int k = 8; k >= 5 && !t; k--) {
        const long long per = (160 * 1024 / k) / 1024 * 1024;
        const long long tk = (per / (R * slot) - pad) / 64 * 64;
        if (tk >= need - 64)
            t = tk;
    }
    if (!t) {
        t = need;
        while (t > 64 && R * (t + pad) * slot > budget)
            t -= 64;
    }
    /* A row whose table does not fit one wavefront's budget: several
     * wavefronts (at most 3 chunks of the rows of B each) share one table
     * of up to 120 KB, so the row still fits in LDS.  When the table fits,
     * one wavefront is faster: on the 32^3 lattice X^2, 6.3 ms against
     * 16 ms with three wavefronts (a step's fixed work and the barrier
     * outweigh the occupancy gain).  On the 64^3 complex X^2 (73 KB tables,
     * 5 chunks) two wavefronts ran in 203 ms, 3 in 211, 5 in 243, one
     * wavefront with the whole table in 323, and the capped table (rows in
     * the global-table pass) in 3200. */
    const int nch = (max_b + 63) / 64;
    int waves = 1;
    if (g == 64 && nch >= 2 && (need + 72) * slot > budget) {
        waves = (nch + 2) / 3;
        if (waves < 2)
            waves = 2;
        if (waves == 7)
            waves = 8;
        if (waves > 8)
            waves = 8;
        long long tm = need;
        const long long mw_budget = 120 * 1024;
        while (tm > 64 && (tm + 72) * slot > mw_budget)
            tm -= 64;
        t = tm;
    }
    const int sel =
        flags & BMLH_PICK_EXACT ? BML_HIP_ROW_ENGINE_EXACT : bml_hip_get_row_engine();
    int engine = (sel == BML_HIP_ROW_ENGINE_UNORDERED || sel == BML_HIP_ROW_ENGINE_WINDOW) &&
                         g == 64
                     ? BMLHIP_ROW_UNORDERED
                     : BMLHIP_ROW_EXACT;
    const char *e;
    if (engine == BMLHIP_ROW_UNORDERED) {
        /* W wavefronts share a row's table; no first-touch list is kept
         * (key + double-component accumulator per slot).  Insertions are
         * counted as they are claimed, so the table needs the row's
         * distinct columns plus slack against growth: max(3/2 est, est +
         * 256) + 64 slots.  For W = 4 and 8, take the largest table that
         * keeps the most blocks per CU (at most 20 wavefronts per CU), and
         * the W with the most wavefronts per CU (ties: the larger table).
         * 32^3 lattice X^2 (FP64, 1177 distinct columns per row): 4 x 2560
         * slots (5 blocks) 2.01 ms, the exact engine 4.76 ms; 64^3 complex
         * X^2 (2139 distinct): 8 wavefronts 101-107 ms, 4 wavefronts 153 ms.
         */
        long long nu = est * 3 / 2;
        if (nu < est + 256)
            nu = est + 256;
        nu = (nu + 64 + 63) & ~63ll;
        /* double-component accumulators (8 or 16 bytes) + key */
        const long long su = (precision == 3 || precision == 4 ? 16 : 8) + 4;
        long long best_waves = -1;
        for (int wv = 4; wv <= 8; wv *= 2) {
            long long tw = 0, kw = 0;
            for (int k = 32 / wv; k >= 1 && !tw; k--) {
                const long long per = (160 * 1024 / k) / 1024 * 1024 - 1024;
                const long long tk = (per / su - 72) / 64 * 64;
                if (tk >= nu - 64) {
                    tw = tk;
                    kw = k;
                }
            }
            if (!tw) {
                tw = nu;
                while (tw > 64 && (tw + 72) * su > 159 * 1024)
                    tw -= 64;
                kw = 1;
            }
            /* beyond ~20 wavefronts per CU the table's load and the
             * epilogue's idle wavefronts cost more than the occupancy buys
             * (lattice X^2: 8 x 3200 slots, 32 per CU, 2.33 ms) */
            while (kw * wv > 20) {
                kw--;
                const long long per = (160 * 1024 / kw) / 1024 * 1024 - 1024;
                tw = (per / su - 72) / 64 * 64;
            }
            if (kw * wv > best_waves || (kw * wv == best_waves && tw > t)) {
                best_waves = kw * wv;
                t = tw;
                waves = wv;
            }
        }
    }
    /* Window engine (squares): forced by the WINDOW setting, or on the
     * unordered setting when a row's distinct columns would pass what an
     * LDS hash table holds at two blocks per CU (beyond that the hash
     * engine's rows fall to the global-table pass).  Windows of 2^11
     * columns (10% faster than 2^12 on the 32^3 lattice at hopping -0.5:
     * smaller windows keep more blocks per CU), eight wavefronts per row;
     * at most 64 windows.  Blocks of 4 consecutive output rows share each
     * streamed row of X (the launcher takes fewer when 4 rows' columns
     * would not fit its LDS union table), with windows of 2^10 columns. */
    out->wbits = 0;
    out->wrows = 1;
    if (square && (sel == BML_HIP_ROW_ENGINE_WINDOW ||
                   (sel == BML_HIP_ROW_ENGINE_UNORDERED && engine == BMLHIP_ROW_UNORDERED))) {
        int wr = (e = getenv("BML_HIP_WIN_ROWS")) ? atoi(e) : 4;
        if (wr != 1 && wr != 2)
            wr = 4;
        int wb = (e = getenv("BML_HIP_WINDOW_BITS")) ? atoi(e) : (wr > 1 ? 10 : 11);
        if (wb < 10)
            wb = 10;
        if (wb > 13)
            wb = 13;
        /* smallest window with at most 64 windows over N columns */
        while (wb < 13 && ((long long) N + (1ll << wb) - 1) >> wb > BMLHIP_WIN_MAX_WINDOWS)
            wb++;
        const int fits = (((long long) N + (1ll << wb) - 1) >> wb) <= BMLHIP_WIN_MAX_WINDOWS;
        const long long wmin = (e = getenv("BML_HIP_WINDOW_MIN")) ? atoll(e) : 3000;
        if (fits && (sel == BML_HIP_ROW_ENGINE_WINDOW || est > wmin)) {
            engine = BMLHIP_ROW_WINDOW;
            out->wbits = wb;
            out->wrows = wr;
            waves = 8;
        }
    }
    out->engine = engine;
    out->waves = (e = getenv("BML_HIP_WAVES")) ? atoi(e) : waves;
    out->group = (e = getenv("BML_HIP_GROUP")) ? atoi(e) : g;
    out->table = (e = getenv("BML_HIP_TABLE")) ? atoi(e) : (int) t;
    /* 2-slot buckets for the unordered engine (its tables sit at ~1/2
     * load): 2.05 against 2.24 ms with 4-slot buckets on the lattice X^2 */
    out->bucket = (e = getenv("BML_HIP_BUCKET")) ? atoi(e)
                                                 : (engine == BMLHIP_ROW_UNORDERED ? 2 : 4);
    /* contiguous rows per XCD cut the HBM fetch of the lattice X^2 5x but
     * ran 1.3x slower than the hardware's round-robin order */
    out->remap = (e = getenv("BML_HIP_XCD_REMAP")) ? atoi(e) : 0;
    /* the exact engine's work goes to the direct-index kernel wherever its
     * LDS holds a row (a shape from the environment is the hash kernels', and
     * so is a batch's work queue) */
    if (engine == BMLHIP_ROW_EXACT && !(flags & BMLH_PICK_QUEUE) && !shape_from_env())
        pick_direct(bmlh_elem_size(precision), N, span, max_a, max_b, est, touched_hint > 0,
                    touched_hint < 0 ? distinct(-touched_hint, max_a, hint_max_a, bound) : 0,
                    touched_hint > 0 && 20 * max_a > 21 * hint_max_a, flags & BMLH_PICK_SOLVE,
                    direct_waves, out);
}

void bmlh_pick_spgemm(int precision, int N, int span, int max_a, int max_b, int touched_hint,
                      int hint_max_a, int flags, bmlh_spgemm_shape *out)
{
    pick(precision, N, span, max_a, max_b, touched_hint, hint_max_a, flags, 0, out);
}

/* ---- measured shapes ------------------------------------------------------
 *
 * With autotuning on, the first product of each kind of operand (a key of
 * precision, flags, the analytic engine and the sizes, the sizes in steps of
 * 2^(1/4)) times candidate shapes around the analytic one on the operands
 * themselves and keeps the fastest, in memory and, when a cache file is
 * named, on disk (one line per key, read back at the next start).  The
 * search is coordinate-wise: for each parameter in turn (exact engine:
 * bucket, lanes per row, table size, wavefronts; unordered: wavefronts,
 * bucket, table; window: window width, rows per block) every value is
 * timed with the others at the best so far.  Each candidate runs twice and
 * the faster time counts; a candidate that fails to launch is skipped.
 * Shapes set through the environment (BML_HIP_GROUP and the like) are left
 * alone. */
typedef struct {
    char key[128];
    bmlh_spgemm_shape sh;
    double ms;
} tune_entry;

static int g_tune = -1; /* -1: not read from the environment yet */
static char g_tune_path[1024];
static tune_entry *g_tab;
static int g_ntab, g_captab, g_loaded;

static const char *const g_override_env[] = {
    "BML_HIP_GROUP", "BML_HIP_TABLE", "BML_HIP_BUCKET", "BML_HIP_WAVES", "BML_HIP_WIN_ROWS",
    "BML_HIP_WINDOW_BITS", "BML_HIP_LDS_BUDGET", "BML_HIP_XCD_REMAP"};

static void tune_env(void)
{
    if (g_tune >= 0)
        return;
    const char *e = getenv("BML_HIP_AUTOTUNE");
    g_tune = e && atoi(e) != 0;
    const char *p = getenv("BML_HIP_TUNE_CACHE");
    if (p)
        snprintf(g_tune_path, sizeof g_tune_path, "%s", p);
}

static int tune_add(const char *key, const bmlh_spgemm_shape *sh, double ms)
{
    for (int k = 0; k < g_ntab; k++)
        if (!strcmp(g_tab[k].key, key)) {
            g_tab[k].sh = *sh;
            g_tab[k].ms = ms;
            return 1;
        }
    if (g_ntab == g_captab) {
        const int cap = g_captab ? 2 * g_captab : 64;
        tune_entry *t = realloc(g_tab, sizeof(tune_entry) * (size_t) cap);
        if (!t)
            return 0;
        g_tab = t;
        g_captab = cap;
    }
    tune_entry *t = &g_tab[g_ntab++];
    snprintf(t->key, sizeof t->key, "%s", key);
    t->sh = *sh;
    t->ms = ms;
    return 1;
}

static void tune_load(void)
{
    if (g_loaded || !g_tune_path[0])
        return;
    g_loaded = 1;
    FILE *f = fopen(g_tune_path, "r");
    if (!f)
        return;
    char line[512];
    while (fgets(line, sizeof line, f)) {
        char key[128];
        bmlh_spgemm_shape sh;
        double ms;
        if (sscanf(line, "%127s %d %d %d %d %d %d %d %d %lf", key, &sh.group, &sh.table,
                   &sh.bucket, &sh.remap, &sh.waves, &sh.engine, &sh.wbits, &sh.wrows, &ms) == 10)
            tune_add(key, &sh, ms);
    }
    fclose(f);
}

static void tune_save(const char *key, const bmlh_spgemm_shape *sh, double ms)
{
    if (!g_tune_path[0])
        return;
    FILE *f = fopen(g_tune_path, "a");
    if (!f)
        return;
    fprintf(f, "%s %d %d %d %d %d %d %d %d %.6f\n", key, sh->group, sh->table, sh->bucket,
            sh->remap, sh->waves, sh->engine, sh->wbits, sh->wrows, ms);
    fclose(f);
}

void bml_hip_set_autotune(int on, const char *cache_path)
{
    tune_env();
    g_tune = on != 0;
    if (cache_path) {
        snprintf(g_tune_path, sizeof g_tune_path, "%s", cache_path);
        g_loaded = 0;
    }
}

int bml_hip_get_autotune(void)
{
    tune_env();
    return g_tune;
}

int bml_hip_autotune_entries(void)
{
    tune_env();
    tune_load();
    return g_ntab;
}

void bml_hip_autotune_clear(void)
{
    free(g_tab);
    g_tab = NULL;
    g_ntab = g_captab = 0;
    g_loaded = 1; /* the file is not read again until a path is set */
}

static int qbucket(long long x)
{
    return x <= 1 ? 0 : (int) ceil(4.0 * log2((double) x));
}

/* time one shape: the faster of two runs, < 0 if it does not launch */
static double tune_time(const bmlh_spgemm_shape *sh, bmlh_measure_fn fn, void *ctx)
{
    double best = -1.0;
    for (int r = 0; r < 2; r++) {
        double ms = 0.0;
        if (fn(sh, ctx, &ms))
            return -1.0;
        if (best < 0.0 || ms < best)
            best = ms;
    }
    return best;
}

static void try_shape(const bmlh_spgemm_shape *c, bmlh_spgemm_shape *best, double *best_ms,
                      bmlh_measure_fn fn, void *ctx)
{
    const double ms = tune_time(c, fn, ctx);
    if (ms >= 0.0 && (*best_ms < 0.0 || ms < *best_ms)) {
        *best = *c;
        *best_ms = ms;
    }
}

void bmlh_tuned_spgemm(int precision, int N, int max_a, int max_b, int touched_hint,
                       int hint_max_a, int flags, bmlh_spgemm_shape *out, bmlh_measure_fn fn,
                       void *ctx)
{
    bmlh_pick_spgemm(precision, N, N, max_a, max_b, touched_hint, hint_max_a, flags, out);
    tune_env();
    if (!g_tune || !fn || N <= 0)
        return;
    for (size_t k = 0; k < sizeof g_override_env / sizeof g_override_env[0]; k++)
        if (getenv(g_override_env[k]))
            return;
    tune_load();
    char key[128];
    snprintf(key, sizeof key, "cu%d:p%d:f%d:e%d:n%d:a%d:b%d:t%d", bmlhip_device_cus(), precision,
             flags & (BMLH_PICK_SQUARE | BMLH_PICK_EXACT), out->engine, qbucket(N), qbucket(max_a), qbucket(max_b),
             qbucket(touched_hint));
    for (int k = 0; k < g_ntab; k++)
        if (!strcmp(g_tab[k].key, key)) {
            /* a key stands for sizes up to a fifth apart.  The direct
             * kernel's index and LDS are made for one: its entries give the
             * wavefronts, the rest follows from this call's own sizes (and
             * where that many do not fit, the analytic shape stays) */
            bmlh_spgemm_shape c = g_tab[k].sh;
            if (c.engine == BMLHIP_ROW_DIRECT) {
                pick(precision, N, N, max_a, max_b, touched_hint, hint_max_a, flags, c.waves, &c);
                if (c.engine != BMLHIP_ROW_DIRECT || c.waves != g_tab[k].sh.waves)
                    return;
            }
            *out = c;
            return;
        }
    bmlh_spgemm_shape best = *out;
    double best_ms = tune_time(out, fn, ctx);
    if (best_ms < 0.0)
        return; /* the analytic shape itself fails: leave it to report */
    bmlh_spgemm_shape c;
    if (out->engine == BMLHIP_ROW_WINDOW) {
        static const int wb[] = {10, 11};
        static const int wr[] = {1, 2, 4};
        for (int k = 0; k < 2; k++) {
            c = best;
            c.wbits = wb[k];
            if (c.wbits != best.wbits)
                try_shape(&c, &best, &best_ms, fn, ctx);
        }
        for (int k = 0; k < 3; k++) {
            c = best;
            c.wrows = wr[k];
            if (c.wrows != best.wrows)
                try_shape(&c, &best, &best_ms, fn, ctx);
        }
    } else if (out->engine == BMLHIP_ROW_UNORDERED) {
        static const int wv[] = {4, 8};
        for (int k = 0; k < 2; k++) {
            c = best;
            c.waves = wv[k];
            if (c.waves != best.waves)
                try_shape(&c, &best, &best_ms, fn, ctx);
        }
        c = best;
        c.bucket = best.bucket == 2 ? 4 : 2;
        try_shape(&c, &best, &best_ms, fn, ctx);
        const int t0 = best.table;
        for (int k = 0; k < 2; k++) {
            c = best;
            c.table = (k ? t0 * 3 / 2 : t0 * 3 / 4) / 64 * 64;
            if (c.table >= 256)
                try_shape(&c, &best, &best_ms, fn, ctx);
        }
    } else if (out->engine == BMLHIP_ROW_DIRECT) {
        /* wavefronts per block, each with the LDS that its rows need (the
         * index at its head does not shrink with them); counts whose LDS
         * cannot hold a row are no candidates */
        const int w0 = best.waves;
        for (int w = w0 > 1 ? w0 / 2 : 1; w <= 2 * w0 && w <= 8; w *= 2) {
            if (w == w0)
                continue;
            pick(precision, N, N, max_a, max_b, touched_hint, hint_max_a, flags, w, &c);
            if (c.engine == BMLHIP_ROW_DIRECT && c.waves == w)
                try_shape(&c, &best, &best_ms, fn, ctx);
        }
    } else {
        static const int bk[] = {2, 4, 8};
        for (int k = 0; k < 3; k++) {
            c = best;
            c.bucket = bk[k];
            if (c.bucket != best.bucket)
                try_shape(&c, &best, &best_ms, fn, ctx);
        }
        const int g0 = best.group;
        for (int g = g0 / 2; g <= 2 * g0 && g <= 64; g *= 2) {
            if (g < 8 || g == g0)
                continue;
            c = best;
            c.group = g;
            c.waves = 1;
            try_shape(&c, &best, &best_ms, fn, ctx);
        }
        const int t0 = best.table;
        for (int k = 0; k < 2; k++) {
            c = best;
            c.table = (k ? t0 * 3 / 2 : t0 * 3 / 4) / 64 * 64;
            if (c.table >= 64)
                try_shape(&c, &best, &best_ms, fn, ctx);
        }
        if (best.group == 64) {
            static const int wv[] = {1, 2, 3, 4};
            for (int k = 0; k < 4; k++) {
                c = best;
                c.waves = wv[k];
                if (c.waves != best.waves)
                    try_shape(&c, &best, &best_ms, fn, ctx);
            }
        }
    }
    *out = best;
    if (tune_add(key, &best, best_ms))
        tune_save(key, &best, best_ms);
}

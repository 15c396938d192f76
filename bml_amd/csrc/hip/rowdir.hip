// Row products on directly indexed accumulators: the exact engine's kernel up
// to 2^14 columns and, above, for long rows and for rows that share columns
// (the line is direct_wins in bml_hip_tune.c).
//
// W wavefronts of a block form RB = W * 64/GROUP consecutive output rows, a
// group of GROUP lanes per row (wavefronts beyond W help with steps 1 to 3
// below and end: where few rows fit a CU, its SIMDs would idle meanwhile).  The columns the block's rows can touch are
// found first and numbered in column order; a row's running sums then lie in
// an LDS array with one slot per such column, and a product's slot is
//
//   idx[k / 32].base + popcount(idx[k / 32].bits below bit k % 32),
//
// one 8-byte LDS read, a mask and a bit count: no hashing, no probing, no
// compare-and-swap.
//
//   1. columns of the block's rows of A into a bitmap, listed (U rows of B);
//   2. the columns of those rows of B into idx[].bits: neighbouring rows
//      share most of them, so U is well below RB times a row's length;
//   3. a scan of the words' bit counts gives idx[].base and D, the number of
//      columns, and colof[slot] = column;
//   4. each row: its D slots are set to -0.0, the group walks row i of A in
//      jp order and adds a * B[j, :] into the slots.
//
// Order and exactness.  All columns of one row of B are distinct, so the
// lanes of a step touch distinct slots, and a wavefront's LDS accesses are
// performed in program order: every sum is formed in jp order, with plain
// reads and writes.  A slot that still holds its start value (-0.0, which no
// sum returns, see sum0) has not been touched: its column is new and gets
// the next rank in (jp, kp) order by a ballot prefix count.  Rows therefore
// come out with the sums and the column order of a sequential walk.
//
// Measured on one MI355X against the hash-table kernels (double unless said;
// the cases below the line are beside it):
// 32^3 lattice iterate squared (177 entries a row, 1.03e9 products) 4.71 ->
// 1.81 ms (1.94 without helpers); 24^3 complex double (279 a row, 1.08e9
// products) 10.5 -> 5.5 ms (6.7);
// random banded N = 4096 (31 a row) 112 -> 37 us; N = 500 137 -> 12.6 us;
// single precision A B of N = 10007 with C merged 181 -> 70 us.
//
// What bounds it.  Each step waits for one LDS round trip (the slot lookups
// of the next step and the sums of this one are read together), with the
// rows of B loaded PD - 1 steps ahead, so the time follows instructions
// issued and the wavefronts resident, which the LDS sets: a slot costs
// sizeof(T) + 2 bytes a row and 4 a block, where a hash table at 2/3 load
// costs (sizeof(T) + 6) * 3/2.
//
// When D slots for all RB rows do not fit the block's LDS, the rows are
// formed in several passes of as many as fit; rows of a block whose D does
// not fit once are handed to the global-table pass.
#include "../bmlhip_abi.h"
#include "rowprod.h"

#include <stdio.h>
#include <type_traits>

using namespace bmlhip;

namespace {

// Slots start as -0.0 (real part).  -0.0 + p is p, and every sum is followed
// by + 0.0, which changes -0.0 to +0.0 and nothing else: the first product
// gives 0.0 + p, a touched slot never holds -0.0 again (x + y is -0.0 only
// when both are), and a slot that does is untouched.  A product that C's row
// already took (fused update) is marked with a signalling NaN, which no
// arithmetic returns; marks are written and read as integer words (the types
// may alias the sums).
typedef unsigned word1 __attribute__((may_alias));
typedef unsigned word2 __attribute__((ext_vector_type(2), may_alias));
constexpr unsigned TAKEN_F = 0x7FA43C3Cu, TAKEN_D = 0x7FF43C3Cu;  // high words
__device__ __forceinline__ bool fresh(float v) { return __float_as_uint(v) == 0x80000000u; }
__device__ __forceinline__ bool fresh(double v) {
    return __double_as_longlong(v) == (long long) 0x8000000000000000ull;
}
__device__ __forceinline__ bool fresh(cf32 v) { return fresh(v.x); }
__device__ __forceinline__ bool fresh(cf64 v) { return fresh(v.x); }
// (x + p) + 0.0 in the real part; -fno-fast-math keeps the second add
__device__ __forceinline__ float sum0(float x, float p) { return (x + p) + 0.0f; }
__device__ __forceinline__ double sum0(double x, double p) { return (x + p) + 0.0; }
__device__ __forceinline__ cf32 sum0(cf32 x, cf32 p) { return {(x.x + p.x) + 0.0f, x.y + p.y}; }
__device__ __forceinline__ cf64 sum0(cf64 x, cf64 p) { return {(x.x + p.x) + 0.0, x.y + p.y}; }
__device__ __forceinline__ float start_of(float) { return -0.0f; }
__device__ __forceinline__ double start_of(double) { return -0.0; }
__device__ __forceinline__ cf32 start_of(cf32) { return {-0.0f, 0.0f}; }
__device__ __forceinline__ cf64 start_of(cf64) { return {-0.0, 0.0}; }
__device__ __forceinline__ void take(float *s) { *(word1 *) s = TAKEN_F; }
__device__ __forceinline__ void take(double *s) { *(word2 *) s = word2{0u, TAKEN_D}; }
__device__ __forceinline__ void take(cf32 *s) { *(word1 *) s = TAKEN_F; }
__device__ __forceinline__ void take(cf64 *s) { *(word2 *) s = word2{0u, TAKEN_D}; }
__device__ __forceinline__ bool is_taken(const float *s) { return *(const word1 *) s == TAKEN_F; }
__device__ __forceinline__ bool is_taken(const double *s) { return (*(const word2 *) s).y == TAKEN_D; }
__device__ __forceinline__ bool is_taken(const cf32 *s) { return *(const word1 *) s == TAKEN_F; }
__device__ __forceinline__ bool is_taken(const cf64 *s) { return (*(const word2 *) s).y == TAKEN_D; }

__device__ __forceinline__ uint64_t ballotb(bool b) { return __builtin_amdgcn_ballot_w64(b); }

__host__ __device__ __forceinline__ unsigned up16(unsigned b) { return (b + 15u) & ~15u; }

__device__ __forceinline__ unsigned slot_of(const uint2 *idx0, unsigned col) {
    const uint2 e = idx0[col >> 5];
    return e.y + __popc(__builtin_amdgcn_ubfe(e.x, 0, col));
}

// One row's epilogue when C is merged: C <- beta*C + alpha*P, the semantics
// of fused_epilogue (ellpack.hip) on direct-indexed slots.  A product slot
// whose column C's row already took is marked TAKEN.
template <typename T, int GROUP>
__device__ int dir_fused(const SpParams &p, int i, bool rowact, const uint2 *idx0, int cbase,
                         int span, bool wide, const int *colof, T *vals, const uint16_t *ord,
                         int count, uint64_t gmask, T &d2) {
    using E = Elem<T>;
    const int lane = lane_id(), gl = lane % GROUP;
    const uint64_t ltmask = (1ull << lane) - 1ull;
    const int MC = p.MC;
    const size_t rowC = (size_t) (rowact ? i : 0) * MC;
    T *Cv = (T *) p.Cv;
    const bool usec = p.beta > 0.0 || p.beta < 0.0;
    const bool usep = p.alpha > 0.0 || p.alpha < 0.0;
    auto pkeeps = [&](int col, T pv) { return col == i || E::above(pv, p.thr); };
    const int nC = rowact && usec ? p.Cn[i] : 0;
    int kept = 0;
    for (int r0 = 0; __any(r0 < nC); r0 += GROUP) {
        const int r = r0 + gl;
        const bool act = r < nC;
        int col = 0;
        T v = E::zero();
        if (act) {
            col = p.Ci[rowC + r];
            v = E::axpy(E::zero(), p.beta, Cv[rowC + r]);
            const unsigned k = (unsigned) (col - cbase);
            if (k < (unsigned) span) {
                if (idx0[(unsigned) col >> 5].x >> (k & 31) & 1u) {
                    const unsigned s = slot_of(idx0, (unsigned) col);
                    if (!fresh(vals[s])) {
                        const T pv = vals[s];
                        if (col == i) d2 = pv;
                        if (usep && pkeeps(col, pv)) {
                            v = E::axpy(v, p.alpha, pv);
                            take(&vals[s]);
                        }
                    }
                }
            }
        }
        const bool keep = act && E::above(v, p.thr);
        const uint64_t km = ballot64(keep) & gmask;
        const int pos = kept + popc64(km & ltmask);
        const uint64_t dm = ballot64(act && col == i) & gmask;
        if (dm) d2 = shfl_any(d2, __ffsll((unsigned long long) dm) - 1);
        if (keep && pos < MC) {
            p.Ci[rowC + pos] = col;
            Cv[rowC + pos] = v;
        }
        kept += popc64(km);
    }
    int keptp = 0;
    for (int r0 = 0; __any(rowact && r0 < count); r0 += GROUP) {
        const int r = r0 + gl;
        const bool act = rowact && r < count;
        int col = -1;
        bool taken = false;
        T pv = E::zero();
        if (act) {
            const unsigned q = ord[r];
            col = wide ? colof[q] : cbase + (int) q;
            const unsigned s = wide ? q : slot_of(idx0, (unsigned) col);
            pv = vals[s];
            taken = is_taken(&vals[s]);
        }
        const bool pk = act && (taken || pkeeps(col, pv));
        keptp += popc64(ballot64(pk) & gmask);
        const uint64_t dm = ballot64(act && !taken && col == i) & gmask;
        if (dm) d2 = shfl_any(pv, __ffsll((unsigned long long) dm) - 1);
        const T v = E::axpy(E::zero(), p.alpha, pv);
        const bool keep = usep && pk && !taken && E::above(v, p.thr);
        const uint64_t km = ballot64(keep) & gmask;
        const int pos = kept + popc64(km & ltmask);
        if (keep && pos < MC) {
            p.Ci[rowC + pos] = col;
            Cv[rowC + pos] = v;
        }
        kept += popc64(km);
    }
    const bool povf = p.kind == 0 ? keptp > MC : count > MC;
    return povf && kept <= MC ? MC + 1 : kept;
}

// Steps in flight: the chunks of a step and PD - 1 steps ahead of it are in
// registers.
template <int NCH>
constexpr int pipe_depth() { return NCH == 1 ? 8 : (NCH <= 3 ? 6 : 4); }

template <typename T, int GROUP, int NCH>
__global__ __launch_bounds__(512) void k_spgemm_dir(SpParams p, unsigned lds_bytes, int nwcap,
                                                    int mode, int W) {
    using E = Elem<T>;
    constexpr int RW = 64 / GROUP;  // rows per wavefront
    constexpr int PD = pipe_depth<NCH>();
    constexpr int S = NCH * GROUP;  // entries of a row of B per step
    extern __shared__ __align__(16) unsigned char smem[];
    if (p.skip && *p.skip) return;
    const int tid = threadIdx.x, T_ = blockDim.x, H = T_ >> 6;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane / GROUP, gl = lane % GROUP;
    const uint64_t gmask = GROUP == 64 ? ~0ull : (((1ull << GROUP) - 1ull) << (g * GROUP));
    const uint64_t ltmask = (1ull << lane) - 1ull;
    const int RB = W * RW;
    const T *Av = (const T *) p.Av;
    const T *Bv = (const T *) p.Bv;
    const int *Ai = p.Ai, *Bi = p.Bi, *Bn = p.Bn;
    const unsigned MB = (unsigned) p.MB;

    uint2 *idx = (uint2 *) smem;  // nwcap words
    int *part_s = (int *) (smem + up16(8u * (unsigned) nwcap));
    int &list_s = part_s[8];
    const unsigned head = up16(8u * (unsigned) nwcap) + 48u;
    unsigned char *pool = smem + head;
    const unsigned pool_bytes = lds_bytes - head;

    const int first = (p.remap ? xcd_block(blockIdx.x, gridDim.x) : (int) blockIdx.x) * RB;
    // row r of the block (-1: none, or its system is finished)
    auto row_of = [&](int r) {
        const int i = first + r;
        if (i >= p.N) return -1;
        return p.row_sys && p.sys_done[p.row_sys[i]] ? -1 : i;
    };

    // The row being formed: entries t .. t + GROUP of row i of A, one per
    // lane, and the next GROUP of them -- the coefficient, the row of B's
    // first slot and its length (0 past the end of row i).  A row of B
    // without entries gets some other row's first slot, so that a load
    // always finds a column.
    int i = -1, nA = 0, steps = 0, prods_l = 0;
    bool live = false, have = false;
    unsigned rowA = 0, some = 0, cb = 0, xb = 0;
    int cn = 0, xn = 0, xj = -1;
    T ca = E::zero(), xa = E::zero(), trx = E::zero();
    auto entries = [&](int t0, int &j, T &a) __attribute__((always_inline)) {
        const int e = t0 + gl;
        const unsigned at = e < nA ? rowA + (unsigned) e : 0u;
        j = e < nA ? Ai[at] : -1;
        a = Av[at];
    };
    auto lengths = [&](int j, T a, unsigned &rb, int &n) __attribute__((always_inline)) {
        n = j >= 0 ? Bn[j] : 0;
        rb = (unsigned) j * MB;
        const uint64_t dm = ballotb(j == i) & gmask;
        if (dm) trx = E::add(trx, shfl_any(a, __ffsll((unsigned long long) dm) - 1));
    };
    auto settle = [&](unsigned &rb, int n) __attribute__((always_inline)) {
        prods_l += n;
        const uint64_t nz = ballotb(n > 0);
        if (nz) {
            some = bcast<64>(rb, __builtin_ctzll(nz));
            have = true;
        }
        rb = n > 0 ? rb : some;
    };
    auto begin_row = [&](int row) {
        i = row;
        live = i >= 0;
        nA = live ? p.An[i] : 0;
        rowA = live ? (unsigned) i * (unsigned) p.MA : 0u;
        if constexpr (GROUP == 64) {  // wave-uniform
            nA = __builtin_amdgcn_readfirstlane(nA);
            rowA = (unsigned) __builtin_amdgcn_readfirstlane((int) rowA);
        }
        steps = nA;  // longest row of A in the wavefront
        if constexpr (GROUP < 64) {
            for (int off = GROUP; off < 64; off <<= 1) {
                const int v = __shfl_xor(steps, off, 64);
                steps = v > steps ? v : steps;
            }
        }
        steps = __builtin_amdgcn_readfirstlane(steps);
        prods_l = 0;
        trx = E::zero();
        have = false;
        some = 0;
        int j;
        entries(0, j, ca);
        entries(GROUP, xj, xa);
        lengths(j, ca, cb, cn);
        settle(cb, cn);
        if (!have) {
            // the first GROUP rows of B named are empty: look further
            for (int t0 = GROUP; t0 < steps && !have; t0 += GROUP) {
                const int e = t0 + gl;
                const int jj = e < nA ? Ai[rowA + (unsigned) e] : -1;
                const uint64_t nz = ballotb(jj >= 0 && Bn[jj >= 0 ? jj : 0] > 0);
                if (nz) {
                    some = (unsigned) bcast<64>(jj, __builtin_ctzll(nz)) * MB;
                    have = true;
                }
            }
            if (!have) steps = 0;  // no products
            cb = some;
        }
    };
    // (helpers of a single row know it too)
    const bool own = mode == BMLHIP_DIR_OWN, shared_row = own && W == 1;
    begin_row(w < W || shared_row ? row_of((shared_row ? 0 : w) * RW + g) : -1);

    // columns the rows can reach: all, or those of the systems of the
    // block's first and last row (the systems between them too)
    int cbase = 0, span = p.N;
    if (p.row_sys) {
        int lo = p.N, hi = 0;
        const int row = lane < RB ? row_of(lane) : -1;
        if (row >= 0) {
            const int sys = p.row_sys[row];
            lo = p.row_off[sys];
            hi = p.row_off[sys + 1];
        }
        for (int off = 32; off > 0; off >>= 1) {
            const int l = __shfl_xor(lo, off, 64), h = __shfl_xor(hi, off, 64);
            lo = l < lo ? l : lo;
            hi = h > hi ? h : hi;
        }
        cbase = lo & ~31;  // a column's low five bits are its bit's number
        span = hi > lo ? hi - cbase : 0;
    }
    const int nw = (span + 31) >> 5;
    bool fits = nw <= nwcap;
    int D = 0;
    const uint2 *idx0 = idx - ((unsigned) cbase >> 5);
    if (fits && mode == BMLHIP_DIR_DENSE) {
        D = span;
        for (int k = tid; k < nw; k += T_) idx[k] = make_uint2(~0u, 32u * (unsigned) k);
    } else if (fits) {
        // The columns of the rows of B named by lanes (first slot rb, n
        // entries each) into the bitmap: each group those of its own lanes,
        // or the wavefront's 64 lanes' shared by its groups.  The first
        // chunks of several rows are in flight; a bit is only set where a
        // read finds it clear (most are set).
        constexpr int Q = NCH == 1 ? 8 : (NCH == 2 ? 6 : (NCH == 3 ? 4 : 3));
        auto mark = [&](int k, bool act) __attribute__((always_inline)) {
            const unsigned kk = act ? (unsigned) k : (unsigned) cbase;
            unsigned *word = (unsigned *) &idx0[kk >> 5].x;
            const unsigned bit = 1u << (kk & 31);
            if (act && !(*word & bit)) atomicOr(word, bit);
        };
        auto mark_rows = [&](unsigned rb, int n, int count) __attribute__((always_inline)) {
            const int stride = own ? (shared_row ? H * Q : Q) : Q * RW;
            for (int t = shared_row ? w * Q : 0; t < count; t += stride) {
                int kcol[Q][NCH], nq[Q];
                unsigned rq[Q];
#pragma unroll
                for (int q = 0; q < Q; q++) {
                    int src = own ? t + q : t + q * RW + g;
                    const bool in = src < count;
                    src = (own ? g * GROUP : 0) + (in ? src : 0);
                    rq[q] = bcast<GROUP>(rb, src);
                    nq[q] = bcast<GROUP>(n, src);
                    nq[q] = in ? nq[q] : 0;
#pragma unroll
                    for (int c = 0; c < NCH; c++) {
                        const int kp = c * GROUP + gl;
                        kcol[q][c] = Bi[kp < nq[q] ? rq[q] + (unsigned) kp : 0u];
                    }
                }
#pragma unroll
                for (int q = 0; q < Q; q++) {
#pragma unroll
                    for (int c = 0; c < NCH; c++) mark(kcol[q][c], c * GROUP + gl < nq[q]);
                    for (int k0 = S; __any(k0 < nq[q]); k0 += GROUP) {
                        const int kp = k0 + gl;
                        const bool act = kp < nq[q];
                        mark(act ? Bi[rq[q] + (unsigned) kp] : cbase, act);
                    }
                }
            }
        };
        unsigned *jbits = (unsigned *) pool;
        for (int k = tid; k < nw; k += T_) {
            idx[k] = make_uint2(0u, 0u);
            if (!own) jbits[k] = 0u;
        }
        if (tid == 0) list_s = 0;
        __syncthreads();
        if (own) {
            mark_rows(cb, cn, steps < GROUP ? steps : GROUP);
            for (int t0 = GROUP; t0 < steps; t0 += GROUP) {
                const int e = t0 + gl;
                const int j = e < nA ? Ai[rowA + (unsigned) e] : -1;
                mark_rows((unsigned) (j >= 0 ? j : 0) * MB, j >= 0 ? Bn[j] : 0,
                          steps - t0 < GROUP ? steps - t0 : GROUP);
            }
        } else {
            int *jlist = (int *) (pool + up16(4u * (unsigned) nw));
            const int jcap = (int) ((pool_bytes - up16(4u * (unsigned) nw)) / 4u);
            for (int e = gl; e < nA; e += GROUP) {
                const unsigned j = (unsigned) (Ai[rowA + (unsigned) e] - cbase);
                atomicOr(&jbits[j >> 5], 1u << (j & 31));
            }
            __syncthreads();
            for (int k = tid; k < nw; k += T_) {
                unsigned b = jbits[k];
                if (b) {
                    int at = atomicAdd(&list_s, __popc(b));
                    while (b) {
                        const int q = __ffs(b) - 1;
                        b &= b - 1u;
                        if (at < jcap) jlist[at] = cbase + 32 * k + q;
                        at++;
                    }
                }
            }
            __syncthreads();
            const int U = list_s;
            fits = U <= jcap;
            if (fits) {
                const int share = (U + H - 1) / H;
                const int u1 = (w + 1) * share < U ? (w + 1) * share : U;
                for (int u0 = w * share; u0 < u1; u0 += 64) {
                    const int n = u1 - u0 < 64 ? u1 - u0 : 64;
                    const int jl = lane < n ? jlist[u0 + lane] : jlist[u0];
                    mark_rows((unsigned) jl * MB, lane < n ? Bn[jl] : 0, n);
                }
            }
        }
        __syncthreads();
        if (fits) {
            // numbers: every thread takes consecutive words
            const int per = (nw + T_ - 1) / T_;
            const int k0 = tid * per, k1 = k0 + per < nw ? k0 + per : nw;
            int n = 0;
            for (int k = k0; k < k1; k++) n += __popc(idx[k].x);
            int inc = n;
            for (int off = 1; off < 64; off <<= 1) {
                const int v = __shfl_up(inc, off, 64);
                if (lane >= off) inc += v;
            }
            if (lane == 63) part_s[w] = inc;
            __syncthreads();
            int at = inc - n;
            for (int v = 0; v < H; v++) {
                const int pv = __builtin_amdgcn_readfirstlane(part_s[v]);
                if (v < w) at += pv;
                D += pv;
            }
            for (int k = k0; k < k1; k++) {
                idx[k].y = (unsigned) at;
                at += __popc(idx[k].x);
            }
        }
    }
    // The pool from here: one spare slot per lane, and per row D sums and the
    // list of its columns in first-touch order.  The list holds 16 bits a
    // column: the column itself (from cbase), or, where the block can reach
    // 2^16 columns or more, its slot, with colof[slot] beside it.
    const bool wide = span > 65536;
    const unsigned fixed =
        (wide ? up16(4u * (unsigned) D) : 0u) + 64u * (unsigned) W * (unsigned) sizeof(T);
    const unsigned per_row = up16((unsigned) (D * (int) sizeof(T))) + up16(2u * (unsigned) D);
    int nconc = 0;
    if (fits && D <= 65535 && fixed < pool_bytes)
        nconc = per_row ? (int) ((pool_bytes - fixed) / per_row) : RB;
    if (nconc > RB) nconc = RB;
    if (nconc == 0) {
        const int r = w * RW + g;
        if (w >= W) return;
        if (gl == 0 && i >= 0) {
            const int q = atomicAdd(&p.st->table_overflow_rows, 1);
            p.ovf[q] = i;
            atomicAdd((unsigned long long *) &p.st->prof_ovf_rows[PrecOf<T>::value], 1ull);
        } else if (gl == 0 && first + r < p.N) {
            p.rowstat[first + r] = make_int4(-1, 0, 0, 0);
        }
        return;
    }
    int *colof = (int *) pool;
    T *lanes = (T *) (pool + (wide ? up16(4u * (unsigned) D) : 0u));
    unsigned char *mine = pool + fixed + (unsigned) (w * RW + g) * per_row;
    T *vals = (T *) mine;
    uint16_t *ord = (uint16_t *) (mine + up16((unsigned) (D * (int) sizeof(T))));
    T *priv = lanes + tid;
    __syncthreads();  // idx complete, the lists no longer read
    if (wide) {
      for (int k = tid; k < nw; k += T_) {
        const uint2 e = idx[k];
        unsigned b = e.x, s = e.y;
        while (b) {
            const int q = __ffs(b) - 1;
            b &= b - 1u;
            if (s < (unsigned) D) colof[s] = cbase + 32 * k + q;
            s++;
        }
      }
      __syncthreads();
    }
    if (w >= W) return;
    *priv = E::zero();

    const bool haveslots = w * RW + g < nconc;
    for (int pass = 0; pass * nconc < RB; pass++) {
        if (w * RW >= nconc) break;  // wave-uniform
        const int r = pass * nconc + w * RW + g;
        const bool mineok = haveslots && r < RB;
        // (the first pass's rows are begun, but those without slots wait)
        if (pass > 0 || ballotb(!mineok)) begin_row(mineok ? row_of(r) : -1);
        if (mineok && !live && gl == 0 && first + r < p.N)
            p.rowstat[first + r] = make_int4(-1, 0, 0, 0);
        if (!__any(live)) continue;
        if (live)
            for (int s = gl; s < D; s += GROUP) vals[s] = start_of(T{});
        int t = 0, kb = 0;  // next step to load: entry t, its columns from kb on
        int issued = 0, done = 0;
        int col[PD][NCH], rem[PD];
        T val[PD][NCH], coef[PD];
        unsigned slot[2][NCH];

        // The next step's chunks into buffer b.  Lanes past the row's end
        // repeat its last entry.  Steps past the last one are empty.
        auto fetch = [&](int b) __attribute__((always_inline)) {
            const int src = g * GROUP + (t & (GROUP - 1));
            const int nb = bcast<GROUP>(cn, src);
            coef[b] = bcast<GROUP>(ca, src);
            const unsigned rb = bcast<GROUP>(cb, src);
            const int n = nb - kb;
            rem[b] = n;
            issued += t < steps;
            const unsigned base = rb + (unsigned) (n > 0 ? kb : 0);
            const char *bi = (const char *) (Bi + base), *bv = (const char *) (Bv + base);
            const unsigned last = n > 0 ? (unsigned) (n - 1) : 0u;
#pragma unroll
            for (int c = 0; c < NCH; c++) {
                const unsigned e = (unsigned) (gl + c * GROUP);
                const unsigned oi = 4u * e < 4u * last ? 4u * e : 4u * last;
                const unsigned ov = (unsigned) sizeof(T) * e < (unsigned) sizeof(T) * last
                                        ? (unsigned) sizeof(T) * e
                                        : (unsigned) sizeof(T) * last;
                col[b][c] = *(const int *) (bi + oi);
                val[b][c] = *(const T *) (bv + ov);
            }
            kb += S;
            if (!(GROUP == 64 ? kb < nb : ballotb(kb < nb) != 0)) {
                kb = 0;
                t++;
                if ((t & (GROUP / 2 - 1)) == 0) {
                    if (t & (GROUP / 2)) {
                        lengths(xj, xa, xb, xn);
                    } else {
                        settle(xb, xn);
                        cb = xb;
                        ca = xa;
                        cn = xn;
                        entries(t + GROUP, xj, xa);
                    }
                }
            }
        };
        uint2 ent[NCH];
        // the index words of buffer b's columns
        auto look = [&](int b) __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < NCH; c++) ent[c] = idx0[(unsigned) col[b][c] >> 5];
        };
        // slots of buffer b's columns
        auto number = [&](int b, unsigned (&sl)[NCH]) __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < NCH; c++)
                sl[c] = ent[c].y + __popc(__builtin_amdgcn_ubfe(ent[c].x, 0, (unsigned) col[b][c]));
        };
        // Step b: the sums of its columns are read together with the index
        // words of the next step's.  Lanes that repeat an entry form the
        // same sum as the lane they repeat and write the same value; a group
        // without entries in this step works on its lanes' spare slots.
        int count = 0;
        auto step = [&](int b, unsigned (&cur)[NCH], unsigned (&nxt)[NCH])
                        __attribute__((always_inline)) {
            T *at[NCH];
            T v[NCH], pr[NCH];
            look((b + 1) % PD);
            const int n = GROUP == 64 ? __builtin_amdgcn_readfirstlane(rem[b]) : rem[b];
#pragma unroll
            for (int c = 0; c < NCH; c++) {
                at[c] = vals + cur[c];
                if constexpr (GROUP < 64) at[c] = n > 0 ? at[c] : priv;
                v[c] = *at[c];
            }
            const T cf = coef[b];
#pragma unroll
            for (int c = 0; c < NCH; c++) pr[c] = E::mul(cf, val[b][c]);
            fetch((b + PD - 1) % PD);
            number((b + 1) % PD, nxt);
            if (GROUP < 64 || n > 0) {
                uint64_t any = 0;
#pragma unroll
                for (int c = 0; c < NCH; c++) any |= ballotb(fresh(v[c]));
                if (any) {
                    // new columns (a lane that repeats an entry lists nothing)
#pragma unroll
                    for (int c = 0; c < NCH; c++) {
                        const uint64_t nm =
                            ballotb(fresh(v[c])) & ballotb(gl + c * GROUP < n) & gmask;
                        const unsigned pos =
                            GROUP == 64 ? __builtin_amdgcn_mbcnt_hi(
                                              (unsigned) (nm >> 32),
                                              __builtin_amdgcn_mbcnt_lo((unsigned) nm, 0u))
                                        : (unsigned) popc64(nm & ltmask);
                        if (fresh(v[c]) & (gl + c * GROUP < n))
                            ord[count + (int) pos] =
                                (uint16_t) (wide ? cur[c] : (unsigned) (col[b][c] - cbase));
                        count += popc64(nm);
                    }
                }
#pragma unroll
                for (int c = 0; c < NCH; c++) *at[c] = sum0(v[c], pr[c]);
            }
            done++;
        };
        static_assert(PD % 2 == 0, "the slot buffers alternate");
        if (steps > 0) {
#pragma unroll
            for (int b = 0; b < PD - 1; b++) fetch(b);
            look(0);
            number(0, slot[0]);
        }
        while (done < issued) {
#pragma unroll
            for (int b = 0; b < PD; b++) {
                step(b, slot[b & 1], slot[(b & 1) ^ 1]);
            }
        }

        // epilogue: thresholded compaction in first-touch order
        const int MC = p.MC;
        const size_t rowC = (size_t) (live ? i : 0) * MC;
        T *Cv = (T *) p.Cv;
        int kept = 0;
        T d2 = E::zero();
        if (p.fuse) {
            kept = dir_fused<T, GROUP>(p, i, live, idx0, cbase, span, wide, colof, vals, ord,
                                       count, gmask, d2);
        } else for (int r0 = 0; __any(live && r0 < count); r0 += GROUP) {
            const int q = r0 + gl;
            const bool act = live && q < count;
            int cc = -1;
            T v = E::zero();
            if (act) {
                const unsigned o = ord[q];
                cc = wide ? colof[o] : cbase + (int) o;
                v = vals[wide ? o : slot_of(idx0, (unsigned) cc)];
            }
            const bool isdiag = act && cc == i;
            const bool keep = isdiag || (act && E::above(v, p.thr));
            const uint64_t km = ballot64(keep) & gmask;
            const int pos = kept + popc64(km & ltmask);
            if (keep && pos < MC) {
                p.Ci[rowC + pos] = cc;
                Cv[rowC + pos] = v;
            }
            const uint64_t dm = ballot64(isdiag) & gmask;
            if (dm) d2 = shfl_any(v, __ffsll((unsigned long long) dm) - 1);
            kept += popc64(km);
        }
        for (int off = 1; off < GROUP; off <<= 1) prods_l += __shfl_xor(prods_l, off, 64);
        if (live && gl == 0) {
            p.Cn[i] = kept < MC ? kept : MC;
            p.rowstat[i] = make_int4(kept, count, prods_l, nA);
            if (p.kind == 0) {
                p.rowtr[i] = E::re(trx);
                p.rowtr[p.N + i] = E::re(d2);
            }
        }
    }
}

int fail(const char *what, hipError_t e) {
    char buf[200];
    snprintf(buf, sizeof buf, "%s: %s", what, hipGetErrorString(e));
    bmlhip_set_errmsg(buf);
    return 3;
}

// wavefronts of a kernel that a CU's registers hold, at most 16
int resident(const void *fn) {
    hipFuncAttributes at;
    if (hipFuncGetAttributes(&at, fn) != hipSuccess || at.numRegs <= 0) return 8;
    const int n = 4 * (512 / ((at.numRegs + 7) / 8 * 8));
    return n < 4 ? 4 : (n > 16 ? 16 : n);
}

template <typename T, int GROUP, int NCH>
int launch(const SpParams &p, int waves, int lds, int span, int mode, hipStream_t s) {
    const int RB = waves * (64 / GROUP);
    const void *fn = (const void *) k_spgemm_dir<T, GROUP, NCH>;
    // helpers up to what a CU holds, where the columns are found and all
    // wavefronts can take part
    int all = waves;
    if (mode == BMLHIP_DIR_LIST || (mode == BMLHIP_DIR_OWN && RB == 1)) {
        static const int most = resident(fn);
        const int blocks = 160 * 1024 / lds;
        while (all < 8 && (all + 1) * blocks <= most) all++;
    }
    if (lds > 64 * 1024)
        (void) hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    const int nblk = (p.N + RB - 1) / RB;
    if (nblk > 0) {
        bmlhip_prof_mark_begin(PrecOf<T>::value);
        hipLaunchKernelGGL((k_spgemm_dir<T, GROUP, NCH>), dim3(nblk), dim3(64 * all), lds, s,
                           p, (unsigned) lds, span / 32 + 2, mode, waves);
        bmlhip_prof_mark_end();
    }
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : fail("k_spgemm_dir", e);
}

}  // namespace

namespace bmlhip {

template <typename T>
int launch_rowdir(const SpParams &p, int group, int nch, int waves, int lds, int span, int mode,
                  hipStream_t s, bool *whole) {
    // what the kernel assumes of its LDS: the index words and, in the rest,
    // the bitmap of A's columns and at least a short list
    const long long words = span / 32 + 2;
    if (waves < 1 || waves > 8 || lds > 160 * 1024 || span < 1 ||
        lds < 12ll * words + 128 + 1024) {
        bmlhip_set_errmsg("direct row product: launch shape out of range");
        return 2;
    }
    // Every row is formed here when a row of all reachable columns fits (the
    // kernel's layout; a batch's range starts at a multiple of 32 columns) and
    // all are numbered: how many are touched depends on the data.
    const unsigned D = (unsigned) (p.row_sys ? span + 31 : p.N);
    const unsigned need = up16(8u * (unsigned) words) + 48u + 64u * (unsigned) waves * (unsigned) sizeof(T) +
                          up16(D * (unsigned) sizeof(T)) + up16(2u * D);
    *whole = mode == BMLHIP_DIR_DENSE && D <= 65535u && (D + 31u) / 32u <= (unsigned) words &&
             need <= (unsigned) lds;
    switch (group * 8 + nch) {
    case 8 * 8 + 1: return launch<T, 8, 1>(p, waves, lds, span, mode, s);
    case 16 * 8 + 1: return launch<T, 16, 1>(p, waves, lds, span, mode, s);
    case 32 * 8 + 1: return launch<T, 32, 1>(p, waves, lds, span, mode, s);
    case 64 * 8 + 1: return launch<T, 64, 1>(p, waves, lds, span, mode, s);
    case 64 * 8 + 2: return launch<T, 64, 2>(p, waves, lds, span, mode, s);
    case 64 * 8 + 3: return launch<T, 64, 3>(p, waves, lds, span, mode, s);
    case 64 * 8 + 4: return launch<T, 64, 4>(p, waves, lds, span, mode, s);
    case 64 * 8 + 5: return launch<T, 64, 5>(p, waves, lds, span, mode, s);
    default: break;
    }
    bmlhip_set_errmsg("direct row product: lanes per row and chunks per step not built");
    return 2;
}

template int launch_rowdir<float>(const SpParams &, int, int, int, int, int, int, hipStream_t, bool *);
template int launch_rowdir<double>(const SpParams &, int, int, int, int, int, int, hipStream_t, bool *);
template int launch_rowdir<cf32>(const SpParams &, int, int, int, int, int, int, hipStream_t, bool *);
template int launch_rowdir<cf64>(const SpParams &, int, int, int, int, int, int, hipStream_t, bool *);

}  // namespace bmlhip

// The end of a row operation in one launch: the sums over rows, the row
// records folded into the status block, what an SP2 iteration decides from
// them, and the results handed to the host.
#pragma once

#include "../bmlhip_abi.h"
#include "devtypes.h"

#include <limits.h>

namespace bmlhip {

// Folds the records of rows first, first + stride, ... (first = the thread's
// row) into the status block, one set of atomics per 256-thread block.
// Records are (kept, distinct, products, nnz of A's row), kept = -1 marking a
// skipped row.  `what` selects: BMLHIP_RS_OVF_KEPT / BMLHIP_RS_OVF_DIST count
// the rows whose kept / distinct count exceeds MC (and the first of them),
// BMLHIP_RS_STORED the largest and total stored row (kept capped at MC),
// BMLHIP_RS_PROF the profiling sums of precision `prof`.
__device__ __forceinline__ void reduce_rowstat(const int4 *rs, int N, int MC, int what, int prof,
                                               int first, int stride, bmlhip_status *st) {
    int ovf = 0, low = INT_MAX, mx = 0, mt = 0;
    unsigned long long tot = 0, prods = 0, rows = 0, innz = 0, dist = 0;
    for (int i = first; i < N; i += stride) {
        const int4 r = rs[i];
        if (r.x < 0) continue;
        const int stored = r.x < MC ? r.x : MC;
        if (((what & BMLHIP_RS_OVF_KEPT) && r.x > MC) || ((what & BMLHIP_RS_OVF_DIST) && r.y > MC)) {
            ovf++;
            low = i < low ? i : low;
        }
        mx = stored > mx ? stored : mx;
        mt = r.y > mt ? r.y : mt;
        tot += (unsigned long long) stored;
        prods += (unsigned long long) (unsigned) r.z;
        rows++;
        innz += (unsigned long long) r.w;
        dist += (unsigned long long) r.y;
    }
    for (int off = 32; off > 0; off >>= 1) {
        ovf += __shfl_down(ovf, off, 64);
        const int f = __shfl_down(low, off, 64);
        low = f < low ? f : low;
        const int a = __shfl_down(mx, off, 64);
        mx = a > mx ? a : mx;
        const int b = __shfl_down(mt, off, 64);
        mt = b > mt ? b : mt;
        tot += __shfl_down(tot, off, 64);
        prods += __shfl_down(prods, off, 64);
        rows += __shfl_down(rows, off, 64);
        innz += __shfl_down(innz, off, 64);
        dist += __shfl_down(dist, off, 64);
    }
    __shared__ int si[4][4];
    __shared__ unsigned long long sl[4][5];
    const int w = threadIdx.x / 64;
    if ((threadIdx.x & 63) == 0) {
        si[w][0] = ovf; si[w][1] = low; si[w][2] = mx; si[w][3] = mt;
        sl[w][0] = tot; sl[w][1] = prods; sl[w][2] = rows; sl[w][3] = innz; sl[w][4] = dist;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < 4; k++) {
            ovf += si[k][0];
            low = si[k][1] < low ? si[k][1] : low;
            mx = si[k][2] > mx ? si[k][2] : mx;
            mt = si[k][3] > mt ? si[k][3] : mt;
            tot += sl[k][0]; prods += sl[k][1]; rows += sl[k][2]; innz += sl[k][3]; dist += sl[k][4];
        }
        if (ovf) {
            atomicAdd(&st->m_overflow_rows, ovf);
            atomicMin(&st->first_m_overflow, low);
        }
        if ((what & BMLHIP_RS_STORED) && rows) {
            atomicMax(&st->max_nnz, mx);
            atomicAdd((unsigned long long *) &st->total_nnz, tot);
        }
        if ((what & BMLHIP_RS_PROF) && rows) {
            atomicMax(&st->max_touched, mt);
            atomicAdd((unsigned long long *) &st->prof_products[prof], prods);
            atomicAdd((unsigned long long *) &st->prof_rows[prof], rows);
            atomicAdd((unsigned long long *) &st->prof_in_nnz[prof], innz);
            atomicAdd((unsigned long long *) &st->prof_out_nnz[prof], tot);
            atomicAdd((unsigned long long *) &st->prof_touched[prof], dist);
            if (!(what & BMLHIP_RS_OWN_STREAM))
                atomicAdd((unsigned long long *) &st->prof_streamed[prof], prods);
        }
    }
}

inline int rowstat_blocks(int N) {
    const int b = (N + 2047) / 2048;
    return b < 1 ? 1 : (b > 240 ? 240 : b);
}

struct TailParams {
    int N, MC, what, prof;
    const int *skip;     // when set and nonzero, the launch does nothing
    const int4 *rowstat;  // NULL: no records to fold
    // sums of x[k][0 .. N) into out[k] (k < nsum), or, with nsys systems,
    // of each unfinished system's rows into out[k][system]
    int nsum;
    const double *x[2];
    double *out[2];
    int nsys;
    const int *row_off;
    int *done;
    bmlhip_status *st;
    bmlhip_sp2_tail sp2;  // what the solve does next
    bmlhip_host *host;    // pinned: where the results go
};

// Queues the launch; the status block is then as after a reset, its values
// in host->status.
int launch_tail(const TailParams &p, hipStream_t s);

}  // namespace bmlhip

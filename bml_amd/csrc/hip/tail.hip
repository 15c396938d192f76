// One launch ends a row operation.  An x2 used to end with three small
// launches (row records, tr X, tr X^2), an SP2 iteration with as many again
// for its decisions, each call with a device-to-host copy of the status
// block, and the next operation began with a launch that reset it; each cost
// 4-5 us of launch and idle GPU, more than the product itself on small
// matrices.
//
// The blocks of the launch each take one part (a sum, or a share of the row
// records).  The block that ends last sees every part's results: it takes
// the SP2 decision, writes the status block to pinned host memory (read by
// the host once the stream has drained) and resets it for the next
// operation.
#include "tail.h"

#include <math.h>
#include <stdio.h>

using namespace bmlhip;

namespace {

__device__ __forceinline__ double peek(const double *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int peek(const int *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The sum of n doubles as 1024 threads form it (thread t: x[t], x[t + 1024],
// ... in turn; then a tree), by 256 threads that stand for four each: the
// order, and so every bit, does not depend on the block size.
__device__ double sum1024(const double *x, int n, double *part) {
    const int t = threadIdx.x;
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    int k = t;
    for (; k + 3 * 1024 + 768 < n; k += 4 * 1024) {  // 16 loads in flight
        double v[4][4];
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int q = 0; q < 4; q++) v[u][q] = x[k + 1024 * u + 256 * q];
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int q = 0; q < 4; q++) s[q] += v[u][q];
    }
    for (; k < n; k += 1024)
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (k + 256 * q < n) s[q] += x[k + 256 * q];
#pragma unroll
    for (int q = 0; q < 4; q++) part[t + 256 * q] = s[q];
    __syncthreads();
    for (int w = 512; w > 0; w >>= 1) {
        for (int u = t; u < w; u += 256) part[u] += part[u + w];
        __syncthreads();
    }
    return part[0];
}

// one system's rows, by 256 threads
__device__ double sum_rows(const double *x, int r0, int r1, double *part) {
    double acc = 0.0;
    for (int k = r0 + (int) threadIdx.x; k < r1; k += 256) acc += x[k];
    part[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int) threadIdx.x < w) part[threadIdx.x] += part[threadIdx.x + w];
        __syncthreads();
    }
    return part[0];
}

__global__ __launch_bounds__(256) void k_tail(TailParams p) {
    __shared__ double part[1024];
    __shared__ int last_s;
    if (p.skip && *p.skip) return;
    const int nsb = p.nsys > 0 ? p.nsum * p.nsys : p.nsum;
    const int b = blockIdx.x, t = threadIdx.x;
    if (b < nsb) {
        if (p.nsys > 0) {
            const int k = b / p.nsys, s = b - k * p.nsys;
            if (!p.done[s]) {
                const double v = sum_rows(p.x[k], p.row_off[s], p.row_off[s + 1], part);
                if (t == 0) p.out[k][s] = v;
            }
        } else {
            const double v = sum1024(p.x[b], p.N, part);
            if (t == 0) *p.out[b] = v;
        }
    } else {
        reduce_rowstat(p.rowstat, p.N, p.MC, p.what, p.prof, (b - nsb) * 256 + t,
                       ((int) gridDim.x - nsb) * 256, p.st);
    }
    // every block's results are visible before it is counted
    __threadfence();
    __syncthreads();
    if (t == 0) last_s = atomicAdd(&p.st->tail_done, 1) == (int) gridDim.x - 1;
    __syncthreads();
    if (!last_s) return;
    __threadfence();

    bmlhip_status *st = p.st;
    const bmlhip_sp2_tail &q = p.sp2;
    switch (q.op) {
    case BMLHIP_TAIL_DECIDE:
        if (t == 0) {
            // Niklasson's trace-correcting choice (see k_sp2_decide)
            bmlhip_sp2_state *s = q.state;
            const double trx = peek(&st->scalars[0]), trx2 = peek(&st->scalars[1]);
            const int branch =
                fabs(trx2 - q.nocc) < fabs(2.0 * trx - trx2 - q.nocc) ? 0 : 1;
            s->branch = branch;
            s->ab[0] = branch ? 2.0 : 0.0;
            s->ab[1] = branch ? -1.0 : 1.0;
            s->trx = trx;
            s->trx2 = trx2;
            s->max_touched = peek(&st->max_touched);
            s->max_nnz_x2 = peek(&st->max_nnz);
            if (q.hist && s->it < q.maxit) {
                q.hist[4 * s->it + 0] = trx;
                q.hist[4 * s->it + 1] = trx2;
                q.hist[4 * s->it + 3] = (double) branch;
            }
        }
        break;
    case BMLHIP_TAIL_CHECK:
        if (t == 0) {
            bmlhip_sp2_state *s = q.state;
            const double nrm = sqrt(peek(&st->scalars[2]));
            s->norm = nrm;
            s->max_nnz = peek(&st->max_nnz);
            if (q.touched) s->max_touched = peek(&st->max_touched);
            if (q.hist && s->it < q.maxit) q.hist[4 * s->it + 2] = nrm;
            s->it++;
            if (nrm <= q.tol) s->done = 1;
            p.host->state = *s;
        }
        break;
    case BMLHIP_TAIL_DECIDE_BATCH:
        if (t == 0) q.stats[0] = peek(&st->max_touched);
        for (int s = t; s < p.nsys; s += 256) {
            if (p.done[s]) continue;
            const double trx = peek(&p.out[0][s]), trx2 = peek(&p.out[1][s]), nc = q.d_nocc[s];
            const int br = fabs(trx2 - nc) < fabs(2.0 * trx - trx2 - nc) ? 0 : 1;
            q.branch[s] = br;
            q.ab[2 * s] = br ? 2.0 : 0.0;
            q.ab[2 * s + 1] = br ? -1.0 : 1.0;
        }
        break;
    case BMLHIP_TAIL_CHECK_BATCH:
        for (int s = t; s < p.nsys; s += 256) {
            if (p.done[s]) continue;
            const double nrm = sqrt(peek(&p.out[0][s]));
            q.norm[s] = nrm;
            q.it[s] += 1;
            if (nrm <= q.tol || q.it[s] >= q.maxit) {
                p.done[s] = nrm <= q.tol ? 1 : 2;  // 1 converged, 2 iteration cap
                atomicAdd(q.alldone, 1);
            }
        }
        __syncthreads();
        if (t == 0) {
            q.stats[1] = peek(&st->max_nnz);
            p.host->stats[0] = peek(&q.stats[0]);
            p.host->stats[1] = peek(&q.stats[1]);
            p.host->alldone = peek(q.alldone);
        }
        break;
    default:
        break;
    }
    // the status block to the host, then cleared for the next operation
    // (overflow counts and profiling sums stay)
    const int words = (int) (sizeof(bmlhip_status) / sizeof(int));
    for (int k = t; k < words; k += 256) ((int *) &p.host->status)[k] = peek((const int *) st + k);
    __syncthreads();
    if (t == 0) {
        st->table_overflow_rows = 0;
        st->max_nnz = 0;
        st->max_touched = 0;
        st->cursor = 0;
        st->total_nnz = 0;
        for (int k = 0; k < 4; k++) st->scalars[k] = 0.0;
        st->tail_done = 0;
    }
}

}  // namespace

namespace bmlhip {

int launch_tail(const TailParams &p, hipStream_t s) {
    const int nsb = p.nsys > 0 ? p.nsum * p.nsys : p.nsum;
    hipLaunchKernelGGL(k_tail, dim3(nsb + (p.rowstat ? rowstat_blocks(p.N) : 0)), dim3(256), 0, s, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        char buf[200];
        snprintf(buf, sizeof buf, "k_tail: %s", hipGetErrorString(e));
        bmlhip_set_errmsg(buf);
        return 3;
    }
    bmlhip_status_published();
    return 0;
}

}  // namespace bmlhip

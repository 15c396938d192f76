// What the row-product kernels of the ELLPACK path share: their parameters,
// and the launcher of the direct-index kernel (rowdir.hip).
#pragma once

#include "../bmlhip_abi.h"
#include "devtypes.h"

namespace bmlhip {

struct SpParams {
    int N, MA, MB, MC, kind;
    const void *Av;
    const int *Ai, *An;
    const void *Bv;
    const int *Bi, *Bn;
    void *Cv;
    int *Ci, *Cn;
    double thr;
    double *rowtr;  // [2*N]: per-row tr X and tr X^2 contributions (x2)
    bmlhip_status *st;
    int *ovf;         // rows handed to the global-table pass
    const int *skip;  // when set and nonzero, the launch does nothing
    int4 *rowstat;    // [N]: (kept, distinct columns, products, nnz of A's row),
                      // kept = -1 for a skipped row; reduced by k_row_stats
    int remap;        // XCD-aware block-to-row order
    int sym;          // symmetric x2: rows form only the columns k >= i
    // batched systems: row i belongs to system row_sys[i]; rows of systems
    // with sys_done set are skipped (both NULL: one system); system s holds
    // the rows and columns row_off[s] .. row_off[s + 1]
    const int *row_sys, *sys_done, *row_off;
    // fuse: C <- beta*C + alpha*(A*B), merged in the epilogue
    int fuse;
    double alpha, beta;
    // batched work queue (NULL: one block per row): the rows to form are
    // qlist[0 .. qinfo[0]), taken with the cursor qinfo[1]
    const int *qlist;
    int *qinfo;
};

// bml_matrix_precision_t of an element type
template <typename T> struct PrecOf;
template <> struct PrecOf<float> { static constexpr int value = 1; };
template <> struct PrecOf<double> { static constexpr int value = 2; };
template <> struct PrecOf<cf32> { static constexpr int value = 3; };
template <> struct PrecOf<cf64> { static constexpr int value = 4; };

template <typename T>
__device__ __forceinline__ T shfl_any(T v, int src) {
    static_assert(sizeof(T) % 4 == 0, "element must be a multiple of 4 bytes");
    union U {
        T t;
        int w[sizeof(T) / 4];
    } u, r;
    u.t = v;
#pragma unroll
    for (int k = 0; k < (int) (sizeof(T) / 4); k++) r.w[k] = __shfl(u.w[k], src, 64);
    return r.t;
}

// Broadcast lane src's value to the caller's lanes.  With one group per
// wavefront src is wave-uniform and a scalar readlane does it.
template <int GROUP, typename T>
__device__ __forceinline__ T bcast(T v, int src) {
    if constexpr (GROUP == 64) {
        static_assert(sizeof(T) % 4 == 0, "element must be a multiple of 4 bytes");
        union U {
            T t;
            int w[sizeof(T) / 4];
        } u, r;
        u.t = v;
#pragma unroll
        for (int k = 0; k < (int) (sizeof(T) / 4); k++)
            r.w[k] = __builtin_amdgcn_readlane(u.w[k], src);
        return r.t;
    } else {
        return shfl_any(v, src);
    }
}

// Launch of the direct-index kernel for element type T: GROUP lanes per row
// (8, 16, 32 or 64), nch chunks of a row of B per step, waves wavefronts per
// block, lds bytes of LDS per block, span = columns a block's rows can reach
// (N, or for batched systems the columns of the systems a block can touch),
// mode: BMLHIP_DIR_*.  *whole: this shape leaves no row to the global-table
// pass.
template <typename T>
int launch_rowdir(const SpParams &p, int group, int nch, int waves, int lds, int span, int mode,
                  hipStream_t s, bool *whole);

}  // namespace bmlhip

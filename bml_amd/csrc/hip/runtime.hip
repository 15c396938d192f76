// Device runtime for the bml HIP backend: one device, one stream (default
// priority), a device status block, and grow-on-demand scratch buffers.
#include <hip/hip_runtime.h>
#include <limits.h>
#include <stdio.h>
#include <string.h>

#include <mutex>
#include <unordered_map>

#include "../bmlhip_abi.h"

namespace {

struct Runtime {
    int capturing = 0;
    int profiling = 0;
    int prof_n = 0;
    hipEvent_t prof_ev[2 * 4096];
    int prof_prec[4096];
    int device = -1;
    hipStream_t stream = nullptr;
    bmlhip_status *status = nullptr;
    bmlhip_host *host = nullptr;  // pinned
    bool clear = false;      // the status block's per-operation fields are reset
    bool published = false;  // host->status is the last operation's
    void *scratch[BMLHIP_SCRATCH_SLOTS] = {};
    size_t scratch_bytes[BMLHIP_SCRATCH_SLOTS] = {};
    char msg[512] = {0};
    void *noalloc_ws[64] = {};  // address of `scratch` on each device
};

Runtime g;

// Device memory of the temporaries that calls make and drop (the second
// matrix of a solve, a multiply's product): hipMalloc, hipFree and the wait
// that a free needs took 0.6 - 5 ms of a 3001-block-row bml_multiply whose
// kernels run 0.2 ms.  Freed blocks are kept, up to POOL_BLOCKS of them and
// POOL_BYTES in all, and handed out again in stream order (all work runs on
// one stream).  They go back to the device when an allocation fails, at
// bml_hip_release_temporaries and at shutdown.
constexpr size_t POOL_BYTES = (size_t) 16 << 30;
constexpr size_t POOL_BLOCKS = 64;
struct PoolBlock {
    void *p;
    size_t n;
};
std::mutex pool_lock;
PoolBlock pool_kept[POOL_BLOCKS];
size_t pool_nkept = 0, pool_kept_bytes = 0;
std::unordered_map<void *, size_t> pool_live;

// (pool_lock held)
void pool_release() {
    if (!pool_nkept) return;
    (void) hipStreamSynchronize(g.stream);
    for (size_t k = 0; k < pool_nkept; k++) (void) hipFree(pool_kept[k].p);
    pool_nkept = pool_kept_bytes = 0;
}

// Notes a block in use (pool_lock held); false when the host has no memory
// for the note: such a block is freed as any other array.  The callers are C,
// which no exception may reach.
bool pool_note(void *p, size_t n) noexcept {
    try {
        pool_live[p] = n;
        return true;
    } catch (...) {
        return false;
    }
}

// hipMalloc; when it fails, once more with the pool given back
hipError_t device_malloc(void **p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess) {
        (void) hipGetLastError();
        {
            std::lock_guard<std::mutex> hold(pool_lock);
            pool_release();
        }
        e = hipMalloc(p, bytes);
    }
    return e;
}

int fail(hipError_t e, const char *what) {
    snprintf(g.msg, sizeof g.msg, "%s: %s", what, hipGetErrorString(e));
    return 3;  // BML_HIP_ERR_DEVICE
}

}  // namespace

// Workspace of the entry points that allocate nothing (for callers that
// cannot call hipMalloc: graph capture, tight serving loops).  Each GPU the
// library runs on holds its own copy until the process ends.  In host code
// the name is only a stand-in: the device address comes from
// hipGetSymbolAddress at bmlhip_init (noalloc_ws), and only that is passed
// to kernels.
__device__ __align__(256) unsigned char scratch[BMLHIP_NOALLOC_BYTES];

// Clears the per-operation fields of the status block on the library stream
// (a kernel rather than a memset node, so a captured graph replays it
// faithfully).  The overflow fields accumulate until the host has checked
// them and asks for them to be cleared too.
__global__ void k_status_reset(bmlhip_status *st, int clear_errors) {
    if (threadIdx.x == 0) {
        if (clear_errors) {
            st->m_overflow_rows = 0;
            st->first_m_overflow = INT_MAX;
            st->tail_done = 0;
        }
        st->table_overflow_rows = 0;
        st->max_nnz = 0;
        st->max_touched = 0;
        st->cursor = 0;
        st->total_nnz = 0;
        for (int k = 0; k < 4; k++) st->scalars[k] = 0.0;
    }
}

// the status block as it is, to the host
__global__ void k_publish(const bmlhip_status *st, bmlhip_host *host) {
    const int words = (int) (sizeof(bmlhip_status) / sizeof(int));
    for (int k = threadIdx.x; k < words; k += 64)
        ((int *) &host->status)[k] = ((const int *) st)[k];
}

#define CHECK(call)                                   \
    do {                                              \
        hipError_t e_ = (call);                       \
        if (e_ != hipSuccess) return fail(e_, #call); \
    } while (0)

extern "C" {

const char *bmlhip_errmsg(void) { return g.msg; }

void bmlhip_set_errmsg(const char *m) { snprintf(g.msg, sizeof g.msg, "%s", m); }

int bmlhip_init(int device) {
    if (g.device >= 0) return 0;
    int n = 0;
    CHECK(hipGetDeviceCount(&n));
    if (device < 0 || device >= n) {
        snprintf(g.msg, sizeof g.msg, "device %d not present (%d devices)", device, n);
        return 3;
    }
    CHECK(hipSetDevice(device));
    if (device < 64 && !g.noalloc_ws[device]) {
        void *ws = nullptr;
        CHECK(hipGetSymbolAddress(&ws, HIP_SYMBOL(scratch)));
        g.noalloc_ws[device] = ws;
    }
    CHECK(hipStreamCreateWithFlags(&g.stream, hipStreamNonBlocking));
    CHECK(hipMalloc((void **) &g.status, sizeof(bmlhip_status)));
    CHECK(hipHostMalloc((void **) &g.host, sizeof(bmlhip_host), hipHostMallocDefault));
    memset(g.host, 0, sizeof(bmlhip_host));
    g.clear = g.published = false;
    hipLaunchKernelGGL(k_status_reset, dim3(1), dim3(64), 0, g.stream, g.status, 1);
    CHECK(hipGetLastError());
    CHECK(hipStreamSynchronize(g.stream));
    g.device = device;
    return 0;
}

void bmlhip_shutdown(void) {
    if (g.device < 0) return;
    (void) hipStreamSynchronize(g.stream);
    {
        std::lock_guard<std::mutex> hold(pool_lock);
        pool_release();
    }
    for (int s = 0; s < BMLHIP_SCRATCH_SLOTS; s++) {
        if (g.scratch[s]) (void) hipFree(g.scratch[s]);
        g.scratch[s] = nullptr;
        g.scratch_bytes[s] = 0;
    }
    (void) hipFree(g.status);
    (void) hipHostFree(g.host);
    g.host = nullptr;
    (void) hipStreamDestroy(g.stream);
    g.status = nullptr;
    g.stream = nullptr;
    g.device = -1;
}

void *bmlhip_stream(void) { return (void *) g.stream; }

int bmlhip_device_cus(void) {
    int n = 0;
    if (g.device < 0 ||
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, g.device) != hipSuccess)
        return 0;
    return n;
}

// A timed region on the library stream (the autotuner's measurements):
// begin records an event, end records a second one, waits for it and gives
// the milliseconds between them.
static hipEvent_t g_tev[2];

int bmlhip_time_begin(void) {
    if (!g_tev[0]) {
        CHECK(hipEventCreate(&g_tev[0]));
        CHECK(hipEventCreate(&g_tev[1]));
    }
    CHECK(hipEventRecord(g_tev[0], g.stream));
    return 0;
}

int bmlhip_time_end(double *ms) {
    float f = 0.0f;
    CHECK(hipEventRecord(g_tev[1], g.stream));
    CHECK(hipEventSynchronize(g_tev[1]));
    CHECK(hipEventElapsedTime(&f, g_tev[0], g_tev[1]));
    *ms = (double) f;
    return 0;
}

void *bmlhip_noalloc_workspace(size_t *bytes) {
    if (bytes) *bytes = BMLHIP_NOALLOC_BYTES;
    return g.device >= 0 && g.device < 64 ? g.noalloc_ws[g.device] : nullptr;
}

int bmlhip_malloc(void **p, size_t bytes) {
    *p = nullptr;
    if (bytes == 0) bytes = 256;
    hipError_t e = device_malloc(p, bytes);
    if (e != hipSuccess) {
        snprintf(g.msg, sizeof g.msg, "hipMalloc(%zu bytes): %s", bytes, hipGetErrorString(e));
        *p = nullptr;
        return 4;  // BML_HIP_ERR_ALLOC
    }
    return 0;
}

int bmlhip_temp_malloc(void **p, size_t bytes) {
    *p = nullptr;
    bytes = (bytes + 255) / 256 * 256;
    if (bytes == 0) bytes = 256;
    {
        // the smallest kept block that is not much too large
        std::lock_guard<std::mutex> hold(pool_lock);
        size_t best = pool_nkept;
        for (size_t k = 0; k < pool_nkept; k++)
            if (pool_kept[k].n >= bytes && pool_kept[k].n <= 2 * bytes + 65536 &&
                (best == pool_nkept || pool_kept[k].n < pool_kept[best].n))
                best = k;
        if (best < pool_nkept && pool_note(pool_kept[best].p, pool_kept[best].n)) {
            *p = pool_kept[best].p;
            pool_kept_bytes -= pool_kept[best].n;
            pool_kept[best] = pool_kept[--pool_nkept];
            return 0;
        }
    }
    const int rc = bmlhip_malloc(p, bytes);
    if (rc) return rc;
    std::lock_guard<std::mutex> hold(pool_lock);
    (void) pool_note(*p, bytes);
    return 0;
}

void bmlhip_temp_free(void *p) {
    if (!p) return;
    {
        std::lock_guard<std::mutex> hold(pool_lock);
        const auto it = pool_live.find(p);
        if (it != pool_live.end() && pool_nkept < POOL_BLOCKS &&
            pool_kept_bytes + it->second <= POOL_BYTES) {
            pool_kept[pool_nkept++] = {p, it->second};
            pool_kept_bytes += it->second;
            pool_live.erase(it);
            return;
        }
    }
    bmlhip_free(p);
}

void bmlhip_temp_release(void) {
    std::lock_guard<std::mutex> hold(pool_lock);
    pool_release();
}

void bmlhip_free(void *p) {
    if (!p) return;
    {
        std::lock_guard<std::mutex> hold(pool_lock);
        pool_live.erase(p);
    }
    // frees must not race kernels still reading the buffer
    (void) hipStreamSynchronize(g.stream);
    (void) hipFree(p);
}

int bmlhip_h2d(void *d, const void *s, size_t n) {
    if (!n) return 0;
    CHECK(hipMemcpyAsync(d, s, n, hipMemcpyHostToDevice, g.stream));
    CHECK(hipStreamSynchronize(g.stream));
    return 0;
}

int bmlhip_d2h(void *d, const void *s, size_t n) {
    if (!n) return 0;
    CHECK(hipMemcpyAsync(d, s, n, hipMemcpyDeviceToHost, g.stream));
    CHECK(hipStreamSynchronize(g.stream));
    return 0;
}

int bmlhip_d2d(void *d, const void *s, size_t n) {
    if (!n) return 0;
    CHECK(hipMemcpyAsync(d, s, n, hipMemcpyDeviceToDevice, g.stream));
    return 0;
}

int bmlhip_zero(void *d, size_t n) {
    if (!n) return 0;
    CHECK(hipMemsetAsync(d, 0, n, g.stream));
    return 0;
}

int bmlhip_sync(void) {
    CHECK(hipStreamSynchronize(g.stream));
    CHECK(hipGetLastError());
    return 0;
}

void *bmlhip_scratch(int slot, size_t bytes) {
    if (slot < 0 || slot >= BMLHIP_SCRATCH_SLOTS) return nullptr;
    if (bytes == 0) bytes = 256;
    if (g.scratch_bytes[slot] >= bytes) return g.scratch[slot];
    // a graph capture cannot record an allocation: the eager pass before it
    // sizes every buffer
    if (g.capturing) {
        snprintf(g.msg, sizeof g.msg, "scratch slot %d would grow during graph capture", slot);
        return nullptr;
    }
    if (g.scratch[slot]) {
        (void) hipStreamSynchronize(g.stream);
        (void) hipFree(g.scratch[slot]);
        g.scratch[slot] = nullptr;
        g.scratch_bytes[slot] = 0;
    }
    size_t want = bytes + bytes / 4;  // headroom against regrowth
    if (device_malloc(&g.scratch[slot], want) != hipSuccess) {
        snprintf(g.msg, sizeof g.msg, "scratch allocation of %zu bytes failed", want);
        g.scratch[slot] = nullptr;
        return nullptr;
    }
    g.scratch_bytes[slot] = want;
    return g.scratch[slot];
}

void *bmlhip_scratch_zeroed(int slot, size_t bytes) {
    const bool grow = slot >= 0 && slot < BMLHIP_SCRATCH_SLOTS && g.scratch_bytes[slot] < bytes;
    void *p = bmlhip_scratch(slot, bytes);
    if (p && grow && hipMemsetAsync(p, 0, g.scratch_bytes[slot], g.stream) != hipSuccess) return nullptr;
    return p;
}

bmlhip_status *bmlhip_status_dev(void) { return g.status; }

bmlhip_host *bmlhip_host_dev(void) { return g.host; }

void bmlhip_status_published(void) { g.clear = g.published = true; }

int bmlhip_status_ready(void) {
    if (!g.clear) return bmlhip_status_reset();
    // the operation that begins here fills the block: only its own k_tail
    // says that it is clear again and that host->status is current
    g.clear = g.published = false;
    return 0;
}

int bmlhip_status_reset(void) {
    g.clear = g.published = false;
    hipLaunchKernelGGL(k_status_reset, dim3(1), dim3(64), 0, g.stream, g.status, 0);
    CHECK(hipGetLastError());
    return 0;
}

int bmlhip_status_clear_errors(void) {
    g.clear = g.published = false;
    hipLaunchKernelGGL(k_status_reset, dim3(1), dim3(64), 0, g.stream, g.status, 1);
    CHECK(hipGetLastError());
    return 0;
}

__global__ void k_prof_reset(bmlhip_status *st) {
    if (threadIdx.x < 5) {
        st->prof_products[threadIdx.x] = 0;
        st->prof_rows[threadIdx.x] = 0;
        st->prof_in_nnz[threadIdx.x] = 0;
        st->prof_out_nnz[threadIdx.x] = 0;
        st->prof_ovf_rows[threadIdx.x] = 0;
        st->prof_touched[threadIdx.x] = 0;
        st->prof_streamed[threadIdx.x] = 0;
    }
}

int bmlhip_prof_begin(void) {
    g.published = false;
    hipLaunchKernelGGL(k_prof_reset, dim3(1), dim3(64), 0, g.stream, g.status);
    CHECK(hipGetLastError());
    g.profiling = 1;
    g.prof_n = 0;
    return 0;
}

void bmlhip_prof_mark_begin(int prec) {
    if (!g.profiling || g.capturing || g.prof_n >= 4096) return;
    hipEvent_t *e = &g.prof_ev[2 * g.prof_n];
    if (hipEventCreate(&e[0]) != hipSuccess || hipEventCreate(&e[1]) != hipSuccess) return;
    g.prof_prec[g.prof_n] = prec;
    (void) hipEventRecord(e[0], g.stream);
}

void bmlhip_prof_mark_end(void) {
    if (!g.profiling || g.capturing || g.prof_n >= 4096) return;
    (void) hipEventRecord(g.prof_ev[2 * g.prof_n + 1], g.stream);
    g.prof_n++;
}

int bmlhip_prof_end(int launches[5], double kernel_ms[5]) {
    CHECK(hipStreamSynchronize(g.stream));
    for (int p = 0; p < 5; p++) {
        launches[p] = 0;
        kernel_ms[p] = 0.0;
    }
    for (int k = 0; k < g.prof_n; k++) {
        float ms = 0.0f;
        const int p = g.prof_prec[k] >= 1 && g.prof_prec[k] <= 4 ? g.prof_prec[k] : 0;
        if (hipEventElapsedTime(&ms, g.prof_ev[2 * k], g.prof_ev[2 * k + 1]) == hipSuccess) {
            kernel_ms[p] += ms;
            launches[p]++;
        }
        (void) hipEventDestroy(g.prof_ev[2 * k]);
        (void) hipEventDestroy(g.prof_ev[2 * k + 1]);
    }
    g.profiling = 0;
    g.prof_n = 0;
    return 0;
}

int bmlhip_graph_begin(void) {
    CHECK(hipStreamBeginCapture(g.stream, hipStreamCaptureModeThreadLocal));
    g.capturing = 1;
    return 0;
}

int bmlhip_graph_end(void **exec) {
    hipGraph_t graph = nullptr;
    g.capturing = 0;
    CHECK(hipStreamEndCapture(g.stream, &graph));
    hipGraphExec_t ge = nullptr;
    const hipError_t e = hipGraphInstantiate(&ge, graph, nullptr, nullptr, 0);
    (void) hipGraphDestroy(graph);
    if (e != hipSuccess) return fail(e, "hipGraphInstantiate");
    *exec = (void *) ge;
    return 0;
}

int bmlhip_graph_launch(void *exec) {
    CHECK(hipGraphLaunch((hipGraphExec_t) exec, g.stream));
    return 0;
}

void bmlhip_graph_destroy(void *exec) {
    if (exec) (void) hipGraphExecDestroy((hipGraphExec_t) exec);
}

int bmlhip_status_fetch(bmlhip_status *h) {
    if (!g.published) {
        hipLaunchKernelGGL(k_publish, dim3(1), dim3(64), 0, g.stream, g.status, g.host);
        CHECK(hipGetLastError());
    }
    CHECK(hipStreamSynchronize(g.stream));
    CHECK(hipGetLastError());
    *h = g.host->status;
    return 0;
}

int bmlhip_sp2_state_fetch(bmlhip_sp2_state *st) {
    CHECK(hipStreamSynchronize(g.stream));
    *st = g.host->state;
    return 0;
}

int bmlhip_sp2_stats_fetch(int stats[2], int *alldone) {
    CHECK(hipStreamSynchronize(g.stream));
    stats[0] = g.host->stats[0];
    stats[1] = g.host->stats[1];
    *alldone = g.host->alldone;
    return 0;
}

}  // extern "C"

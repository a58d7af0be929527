// api_compat.cpp -- C-ABI: the 12 reference-named launchers, the
// cudaSpmm-shaped dispatcher, device memory / streams / timers (CUArray and
// GpuTimer replacements), and the benchmark / dry-run loops of
// SpmvSpmmProblem.
#include <hip/hip_runtime.h>
#include <rocprofiler-sdk-roctx/roctx.h>

#include <algorithm>
#include <cstring>
#include <mutex>
#include <vector>

#include "internal.hpp"

namespace dspmm {

namespace {
thread_local int g_last_hip_error = 0;
}

dspmm_status_t hip_status(hipError_t e) {
    if (e == hipSuccess) return DSPMM_STATUS_SUCCESS;
    g_last_hip_error = (int)e;
    if (e == hipErrorOutOfMemory) return DSPMM_STATUS_ALLOC_FAILED;
    return DSPMM_STATUS_HIP_ERROR;
}

namespace {

// Argument checks shared by the launchers.  Pointers may be NULL only
// where the corresponding size makes them unused.
dspmm_status_t check_common(int nr, int nc, int nnz, int nv, const int *rowPtr,
                            const int *rowIdx, const int *colIdx, const float *values,
                            const float *B, const float *C, bool coo) {
    if (nr < 0 || nc < 0 || nnz < 0 || nv < 1) return DSPMM_STATUS_INVALID_VALUE;
    if (nr > 0 && !C) return DSPMM_STATUS_INVALID_VALUE;
    if (!coo && nr > 0 && !rowPtr) return DSPMM_STATUS_INVALID_VALUE;
    if (nnz > 0 && (!colIdx || !values || !B)) return DSPMM_STATUS_INVALID_VALUE;
    if (coo && nnz > 0 && !rowIdx) return DSPMM_STATUS_INVALID_VALUE;
    return DSPMM_STATUS_SUCCESS;
}

bool is_coo(int which) {
    return which == K_SPMV_COO_SCALAR || which == K_SPMV_COO_VECTOR ||
           which == K_SPMM_COO_SCALAR_ROW || which == K_SPMM_COO_VECTOR_ROW ||
           which == K_SPMM_COO_SCALAR_COL || which == K_SPMM_COO_VECTOR_COL;
}

bool is_col(int which) {
    return which == K_SPMM_CSR_SCALAR_COL || which == K_SPMM_CSR_VECTOR_COL ||
           which == K_SPMM_COO_SCALAR_COL || which == K_SPMM_COO_VECTOR_COL;
}

// Scratch for one call, in stream order, from a pool of the device that holds
// at most kScratchPool bytes in all.
//   * On the legacy default stream, whose work is in order whoever enqueues it,
//     the calls share one block, kept between them: a call holds the lock until
//     its last launch is enqueued.
//   * On any other stream a call takes a block before its launches and gives it
//     back behind them, so that streams and threads never share one.  That
//     costs a call 18 us, mostly the marker behind its work.
// Free blocks beyond kScratchKept go back to the device at the next
// synchronisation; dspmm_release_scratch, and every allocation of the library that
// finds the memory short (device_malloc), give back the rest.
constexpr size_t kScratchCall = (size_t)256 << 20;   // the most that one call takes
constexpr size_t kScratchKept = kScratchCall;
constexpr size_t kScratchPool = 4 * kScratchCall;
constexpr int kMaxDevices = 64;

struct DevicePool {
    std::mutex lock;                 // held while the shared block's user enqueues
    hipMemPool_t pool = nullptr;
    bool tried = false;
    void *block = nullptr;           // the legacy default stream's
    size_t bytes = 0;
};
DevicePool g_pools[kMaxDevices];

DevicePool *current_pool() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
    return &g_pools[dev];
}

// p.lock is held.
bool make_pool(DevicePool &p, int dev) {
    if (p.tried) return p.pool != nullptr;
    p.tried = true;
    hipMemPoolProps props;
    std::memset(&props, 0, sizeof(props));
    props.allocType = hipMemAllocationTypePinned;
    props.location.type = hipMemLocationTypeDevice;
    props.location.id = dev;
    props.maxSize = kScratchPool;
    hipMemPool_t pool = nullptr;
    if (hipMemPoolCreate(&pool, &props) != hipSuccess) return false;
    uint64_t kept = kScratchKept;
    int wait = 0;                    // no stream is made to wait for another one's scratch
    if (hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &kept) != hipSuccess ||
        hipMemPoolSetAttribute(pool, hipMemPoolReuseAllowInternalDependencies, &wait) != hipSuccess) {
        (void)hipMemPoolDestroy(pool);
        return false;
    }
    p.pool = pool;
    return true;
}

// Gives the current device's free scratch back.  Waits for the legacy default
// stream, whose block it frees.
dspmm_status_t release_scratch() {
    DevicePool *p = current_pool();
    if (!p) return DSPMM_STATUS_SUCCESS;
    std::lock_guard<std::mutex> held(p->lock);
    if (!p->pool) return DSPMM_STATUS_SUCCESS;
    hipError_t e = hipSuccess;
    if (p->block) e = hipFreeAsync(p->block, nullptr);
    p->block = nullptr;
    p->bytes = 0;
    if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
    if (e == hipSuccess) e = hipMemPoolTrimTo(p->pool, 0);
    return hip_status(e);
}

class Scratch {
public:
    Scratch(size_t need, hipStream_t st) : st_(st) {
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        if (st && (hipStreamIsCapturing(st, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone))
            return;
        DevicePool *p = current_pool();
        if (!p) return;
        std::unique_lock<std::mutex> held(p->lock);
        if (!make_pool(*p, (int)(p - g_pools))) return;
        size_t bytes = 1 << 20;      // few sizes, so that a freed block fits the next call
        while (bytes < need) bytes *= 2;
        if (st) {
            held.unlock();
            if (hipMallocFromPoolAsync(&ptr_, bytes, p->pool, st) != hipSuccess) ptr_ = nullptr;
            return;
        }
        if (p->bytes < bytes) {
            if (p->block) (void)hipFreeAsync(p->block, nullptr);
            p->block = nullptr;
            p->bytes = 0;
            if (hipMallocFromPoolAsync(&p->block, bytes, p->pool, nullptr) != hipSuccess) {
                p->block = nullptr;
                return;
            }
            p->bytes = bytes;
        }
        ptr_ = p->block;
        held_ = std::move(held);
    }
    void *ptr() const { return ptr_; }
    // Behind the last launch that uses it.
    dspmm_status_t release() {
        if (!ptr_) return DSPMM_STATUS_SUCCESS;
        const dspmm_status_t s = st_ ? hip_status(hipFreeAsync(ptr_, st_)) : DSPMM_STATUS_SUCCESS;
        if (held_.owns_lock()) held_.unlock();
        ptr_ = nullptr;
        return s;
    }

private:
    hipStream_t st_;
    void *ptr_ = nullptr;
    std::unique_lock<std::mutex> held_;
};

// Columns at a time with which a column-major product runs on row-major copies
// (launch_compat_flipped); 0: in place.  In place every product costs a line of
// B (about 0.22 M gathers a microsecond where B is random, twice that where the
// L2s hold it), the copies cost three to four launches (10 to 13 us, and on a
// stream other than the legacy default one 18 us more for the scratch) and a
// pass over B and C.  So the line lies at a number of products, lower where B
// is too large for the L2s.  In place / copies, us: 131072 rows of 24, nv = 32
// (100 M products) 464 / 76; 16384 rows of 32, nv = 8 (4.2 M) csr_vector 15 / 12,
// coo 21 / 14; 39^3 stencil, nv = 4 (6.1 M) csr_vector 10 / 13; 5000 rows of 12 over
// 250000 columns, nv = 16 (0.96 M, B of 16 MB) csr_vector 18 / 14; 131072 rows of 6,
// nv = 4 (3.1 M) csr_scalar 17 / 16, coo 18 / 21.  Two columns share their lines less:
// power law, nv = 2 (6.4 M), coo 33 / 37.
int flip_columns(int which, int nr, int nc, int nnz, int nv, bool null_stream) {
    if (nv < 2 || nr == 0 || nnz == 0) return 0;
    const double products = 1e-6 * nnz * nv, b = 1e-6 * nc * nv;
    bool pays;
    if (which == K_SPMM_CSR_SCALAR_COL)
        pays = products >= (null_stream ? 4.1 : 6.0);
    else if (which == K_SPMM_CSR_VECTOR_COL)
        pays = null_stream ? products >= 8.0 || (products >= 5.0 && b >= 1.0) || (products >= 1.0 && b >= 4.0)
                           : products >= 14.0 || (products >= 3.4 && b >= 1.5);
    else if (nv == 2)
        pays = products >= (null_stream ? 16.0 : 24.0);
    else
        pays = null_stream ? products >= 4.1 || (products >= 2.0 && b >= 4.0)
                           : products >= 10.0 || (products >= 3.8 && b >= 3.0);
    if (!pays) return 0;
    int cols = nv;
    while (cols > 8 && compat_flipped_bytes(nr, nc, cols) > kScratchCall) cols = (cols / 2 + 7) / 8 * 8;
    return compat_flipped_bytes(nr, nc, cols) <= kScratchCall ? cols : 0;
}

// One reference-named launcher: packed operands (ld = nv row-major; ld =
// nc / nr column-major; ld = 1 for the SpMV kernels, whose nv==1 case is
// the same in both layouts).
dspmm_status_t run_named(int which, int nr, int nc, int nnz, int nv, const int *rowPtr,
                         const int *rowIdx, const int *colIdx, const float *values,
                         const float *B, float *C, dspmm_stream_t stream) {
    dspmm_status_t st = check_common(nr, nc, nnz, nv, rowPtr, rowIdx, colIdx, values, B, C,
                                     is_coo(which));
    if (st != DSPMM_STATUS_SUCCESS) return st;
    switch (which) {
    case K_SPMV_CSR_SCALAR:
    case K_SPMV_COO_SCALAR:
        if (nv != 1) return DSPMM_STATUS_NOT_SUPPORTED;
        break;
    case K_SPMV_CSR_VECTOR:
    case K_SPMV_COO_VECTOR:
        if (nv != 1 && nv != 2 && nv != 4) return DSPMM_STATUS_NOT_SUPPORTED;
        break;
    default:
        break;
    }
    const int cols = is_col(which) ? flip_columns(which, nr, nc, nnz, nv, stream == nullptr) : 0;
    if (cols) {
        const hipStream_t hs = as_hip(stream);
        Scratch mem(compat_flipped_bytes(nr, nc, cols), hs);
        if (mem.ptr()) {
            st = launch_compat_flipped(which, nr, nc, nnz, nv, rowPtr, rowIdx, colIdx, values, B, C,
                                       static_cast<float *>(mem.ptr()), cols, hs);
            const dspmm_status_t freed = mem.release();
            return st != DSPMM_STATUS_SUCCESS ? st : freed;
        }
        (void)hipGetLastError();     // no scratch (out of memory, a captured stream): without
    }
    int64_t ldb, ldc;
    if (is_col(which)) { ldb = nc; ldc = nr; }
    else { ldb = nv; ldc = nv; }
    return launch_compat(which, nr, nc, nnz, nv, ldb, ldc, rowPtr, rowIdx, colIdx, values, B, C,
                         as_hip(stream), 0);
}

// spmvspmm.h:72-197: (alg, layout, nv) -> reference kernel.
int select_kernel(SPMV_SPMM_ALG alg, DenseLayout layout, int nv) {
    if (layout == DENSE_ROW_MAJOR) {
        switch (alg) {
        case ALG_CSR_SCALAR: return nv == 1 ? K_SPMV_CSR_SCALAR : K_SPMM_CSR_SCALAR_ROW;
        case ALG_COO_SCALAR: return nv == 1 ? K_SPMV_COO_SCALAR : K_SPMM_COO_SCALAR_ROW;
        case ALG_CSR_VECTOR: return nv <= 4 ? K_SPMV_CSR_VECTOR : K_SPMM_CSR_VECTOR_ROW;
        case ALG_COO_VECTOR: return nv <= 4 ? K_SPMV_COO_VECTOR : K_SPMM_COO_VECTOR_ROW;
        }
    } else if (layout == DENSE_COL_MAJOR) {
        switch (alg) {
        case ALG_CSR_SCALAR: return nv == 1 ? K_SPMV_CSR_SCALAR : K_SPMM_CSR_SCALAR_COL;
        case ALG_COO_SCALAR: return nv == 1 ? K_SPMV_COO_SCALAR : K_SPMM_COO_SCALAR_COL;
        case ALG_CSR_VECTOR: return nv == 1 ? K_SPMV_CSR_VECTOR : K_SPMM_CSR_VECTOR_COL;
        case ALG_COO_VECTOR: return nv == 1 ? K_SPMV_COO_VECTOR : K_SPMM_COO_VECTOR_COL;
        }
    }
    return -1;
}

}  // namespace

dspmm_status_t device_malloc(void **ptr, size_t bytes) {
    hipError_t e = hipMalloc(ptr, bytes);
    if (e == hipErrorOutOfMemory && release_scratch() == DSPMM_STATUS_SUCCESS) {
        (void)hipGetLastError();
        e = hipMalloc(ptr, bytes);
    }
    return hip_status(e);
}

}  // namespace dspmm

using namespace dspmm;

extern "C" {

const char *dspmm_get_error_string(dspmm_status_t s) {
    switch (s) {
    case DSPMM_STATUS_SUCCESS: return "success";
    case DSPMM_STATUS_INVALID_VALUE: return "invalid value";
    case DSPMM_STATUS_NOT_SUPPORTED: return "not supported";
    case DSPMM_STATUS_ALLOC_FAILED: return "allocation failed";
    case DSPMM_STATUS_HIP_ERROR: return "HIP runtime error";
    case DSPMM_STATUS_WORKSPACE_TOO_SMALL: return "workspace too small";
    case DSPMM_STATUS_ADMISSION_REJECTED: return "admission rejected (HBM budget)";
    case DSPMM_STATUS_NOT_PREPARED:
        return "not prepared (call dspmm_matrix_prepare with these arguments first)";
    }
    return "unknown status";
}

int dspmm_last_hip_error(void) { return g_last_hip_error; }

const char *dspmm_version(void) { return "dspmm 0.1 (gfx950)"; }

#define DSPMM_NAMED(fn, K)                                                                   \
    dspmm_status_t fn(int nr, int nc, int nnz, int nv, const int *rowPtr, const int *rowIdx, \
                      const int *colIdx, const float *values, const float *dnInput,          \
                      float *dnOutput, dspmm_stream_t stream) {                              \
        return run_named(K, nr, nc, nnz, nv, rowPtr, rowIdx, colIdx, values, dnInput,       \
                         dnOutput, stream);                                                  \
    }

DSPMM_NAMED(spmv_csr_scalar, K_SPMV_CSR_SCALAR)
DSPMM_NAMED(spmv_coo_scalar, K_SPMV_COO_SCALAR)
DSPMM_NAMED(spmv_csr_vector, K_SPMV_CSR_VECTOR)
DSPMM_NAMED(spmv_coo_vector, K_SPMV_COO_VECTOR)
DSPMM_NAMED(spmm_csr_scalar_row, K_SPMM_CSR_SCALAR_ROW)
DSPMM_NAMED(spmm_csr_vector_row, K_SPMM_CSR_VECTOR_ROW)
DSPMM_NAMED(spmm_coo_scalar_row, K_SPMM_COO_SCALAR_ROW)
DSPMM_NAMED(spmm_coo_vector_row, K_SPMM_COO_VECTOR_ROW)
DSPMM_NAMED(spmm_csr_scalar_col, K_SPMM_CSR_SCALAR_COL)
DSPMM_NAMED(spmm_csr_vector_col, K_SPMM_CSR_VECTOR_COL)
DSPMM_NAMED(spmm_coo_scalar_col, K_SPMM_COO_SCALAR_COL)
DSPMM_NAMED(spmm_coo_vector_col, K_SPMM_COO_VECTOR_COL)
#undef DSPMM_NAMED

dspmm_status_t dspmm_spmm(SPMV_SPMM_ALG alg, DenseLayout layout, int nr, int nc, int nnz, int nv,
                          const int *rowPtr, const int *rowIdx, const int *colIdx,
                          const float *values, const float *dnInput, float *dnOutput,
                          dspmm_stream_t stream) {
    if (nv < 1) return DSPMM_STATUS_INVALID_VALUE;
    if ((nv & (nv - 1)) != 0) return DSPMM_STATUS_NOT_SUPPORTED;   // spmvspmm.h:209
    const int k = select_kernel(alg, layout, nv);
    if (k < 0) return DSPMM_STATUS_INVALID_VALUE;
    return run_named(k, nr, nc, nnz, nv, rowPtr, rowIdx, colIdx, values, dnInput, dnOutput,
                     stream);
}

// ---- memory, streams, device --------------------------------------------

dspmm_status_t dspmm_device_alloc(void **ptr, size_t bytes) {
    if (!ptr) return DSPMM_STATUS_INVALID_VALUE;
    *ptr = nullptr;
    if (bytes == 0) return DSPMM_STATUS_SUCCESS;
    return device_malloc(ptr, bytes);
}

dspmm_status_t dspmm_release_scratch(void) { return release_scratch(); }

dspmm_status_t dspmm_device_free(void *ptr) {
    if (!ptr) return DSPMM_STATUS_SUCCESS;
    return hip_status(hipFree(ptr));
}

dspmm_status_t dspmm_memcpy_h2d(void *dst, const void *src, size_t bytes) {
    if (bytes == 0) return DSPMM_STATUS_SUCCESS;
    if (!dst || !src) return DSPMM_STATUS_INVALID_VALUE;
    return hip_status(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
}

dspmm_status_t dspmm_memcpy_d2h(void *dst, const void *src, size_t bytes) {
    if (bytes == 0) return DSPMM_STATUS_SUCCESS;
    if (!dst || !src) return DSPMM_STATUS_INVALID_VALUE;
    return hip_status(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
}

dspmm_status_t dspmm_memcpy_d2d(void *dst, const void *src, size_t bytes, dspmm_stream_t stream) {
    if (bytes == 0) return DSPMM_STATUS_SUCCESS;
    if (!dst || !src) return DSPMM_STATUS_INVALID_VALUE;
    return hip_status(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, as_hip(stream)));
}

dspmm_status_t dspmm_stream_create(dspmm_stream_t *stream) {
    if (!stream) return DSPMM_STATUS_INVALID_VALUE;
    hipStream_t s = nullptr;
    dspmm_status_t st = hip_status(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    *stream = reinterpret_cast<dspmm_stream_t>(s);
    return st;
}

dspmm_status_t dspmm_stream_destroy(dspmm_stream_t stream) {
    if (!stream) return DSPMM_STATUS_SUCCESS;
    return hip_status(hipStreamDestroy(as_hip(stream)));
}

dspmm_status_t dspmm_stream_synchronize(dspmm_stream_t stream) {
    return hip_status(hipStreamSynchronize(as_hip(stream)));
}

dspmm_status_t dspmm_device_synchronize(void) { return hip_status(hipDeviceSynchronize()); }

dspmm_status_t dspmm_get_device_info(dspmm_device_info *info) {
    if (!info) return DSPMM_STATUS_INVALID_VALUE;
    std::memset(info, 0, sizeof(*info));
    int dev = 0;
    dspmm_status_t st = hip_status(hipGetDevice(&dev));
    if (st != DSPMM_STATUS_SUCCESS) return st;
    hipDeviceProp_t p;
    st = hip_status(hipGetDeviceProperties(&p, dev));
    if (st != DSPMM_STATUS_SUCCESS) return st;
    std::strncpy(info->name, p.name, sizeof(info->name) - 1);
    std::strncpy(info->arch, p.gcnArchName, sizeof(info->arch) - 1);
    info->compute_units = p.multiProcessorCount;
    info->wave_size = p.warpSize;
    info->clock_khz = p.clockRate;
    info->l2_bytes = p.l2CacheSize;
    info->lds_per_block = p.sharedMemPerBlock;
    size_t fr = 0, tot = 0;
    st = hip_status(hipMemGetInfo(&fr, &tot));
    info->total_mem = tot;
    info->free_mem = fr;
    return st;
}

// ---- event timer ----------------------------------------------------------

struct dspmm_timer_s {
    std::vector<hipEvent_t> ev;
    int used = 0;
};

dspmm_status_t dspmm_timer_create(dspmm_timer_t *t, int max_marks) {
    if (!t || max_marks < 2) return DSPMM_STATUS_INVALID_VALUE;
    auto *tm = new dspmm_timer_s;
    tm->ev.resize((size_t)max_marks, nullptr);
    for (auto &e : tm->ev) {
        dspmm_status_t st = hip_status(hipEventCreate(&e));
        if (st != DSPMM_STATUS_SUCCESS) {
            for (auto &x : tm->ev) if (x) hipEventDestroy(x);
            delete tm;
            return st;
        }
    }
    *t = tm;
    return DSPMM_STATUS_SUCCESS;
}

dspmm_status_t dspmm_timer_destroy(dspmm_timer_t t) {
    if (!t) return DSPMM_STATUS_SUCCESS;
    for (auto &e : t->ev) hipEventDestroy(e);
    delete t;
    return DSPMM_STATUS_SUCCESS;
}

dspmm_status_t dspmm_timer_reset(dspmm_timer_t t) {
    if (!t) return DSPMM_STATUS_INVALID_VALUE;
    t->used = 0;
    return DSPMM_STATUS_SUCCESS;
}

dspmm_status_t dspmm_timer_mark(dspmm_timer_t t, dspmm_stream_t stream) {
    if (!t) return DSPMM_STATUS_INVALID_VALUE;
    if (t->used >= (int)t->ev.size()) return DSPMM_STATUS_INVALID_VALUE;
    return hip_status(hipEventRecord(t->ev[(size_t)t->used++], as_hip(stream)));
}

dspmm_status_t dspmm_timer_intervals(dspmm_timer_t t, float *ms, int n) {
    if (!t || t->used < 2 || n < 0 || n > t->used - 1) return DSPMM_STATUS_INVALID_VALUE;
    dspmm_status_t st = hip_status(hipEventSynchronize(t->ev[(size_t)t->used - 1]));
    if (st != DSPMM_STATUS_SUCCESS) return st;
    for (int i = 0; i < n; i++) {
        st = hip_status(hipEventElapsedTime(&ms[i], t->ev[(size_t)i], t->ev[(size_t)i + 1]));
        if (st != DSPMM_STATUS_SUCCESS) return st;
    }
    return DSPMM_STATUS_SUCCESS;
}

// ---- SpmvSpmmProblem::benchmark / dry_run -----------------------------------

dspmm_status_t dspmm_benchmark_compat(SPMV_SPMM_ALG alg, DenseLayout layout, int nr, int nc,
                                      int nnz, int nv, const int *rowPtr, const int *rowIdx,
                                      const int *colIdx, const float *values,
                                      const float *dnInput, float *dnOutput, int warmup,
                                      int reps, float *ms_mean, float *ms_per_launch,
                                      dspmm_stream_t stream) {
    if (reps < 1 || warmup < 0) return DSPMM_STATUS_INVALID_VALUE;
    dspmm_status_t st = DSPMM_STATUS_SUCCESS;
    for (int i = 0; i < warmup && st == DSPMM_STATUS_SUCCESS; i++)
        st = dspmm_spmm(alg, layout, nr, nc, nnz, nv, rowPtr, rowIdx, colIdx, values, dnInput,
                        dnOutput, stream);
    if (st != DSPMM_STATUS_SUCCESS) return st;
    st = hip_status(hipStreamSynchronize(as_hip(stream)));
    if (st != DSPMM_STATUS_SUCCESS) return st;
    dspmm_timer_t t = nullptr;
    st = dspmm_timer_create(&t, reps + 1);
    if (st != DSPMM_STATUS_SUCCESS) return st;
    st = dspmm_timer_mark(t, stream);
    for (int i = 0; i < reps && st == DSPMM_STATUS_SUCCESS; i++) {
        st = dspmm_spmm(alg, layout, nr, nc, nnz, nv, rowPtr, rowIdx, colIdx, values, dnInput,
                        dnOutput, stream);
        if (st == DSPMM_STATUS_SUCCESS) st = dspmm_timer_mark(t, stream);
    }
    if (st == DSPMM_STATUS_SUCCESS) {
        std::vector<float> ms((size_t)reps);
        st = dspmm_timer_intervals(t, ms.data(), reps);
        if (st == DSPMM_STATUS_SUCCESS) {
            double sum = 0;
            for (float x : ms) sum += x;
            if (ms_mean) *ms_mean = (float)(sum / reps);
            if (ms_per_launch) std::copy(ms.begin(), ms.end(), ms_per_launch);
        }
    }
    dspmm_timer_destroy(t);
    return st;
}

dspmm_status_t dspmm_dry_run_compat(SPMV_SPMM_ALG alg, DenseLayout layout, int nr, int nc,
                                    int nnz, int nv, const int *rowPtr, const int *rowIdx,
                                    const int *colIdx, const float *values,
                                    const float *dnInput, float *dnOutput, int warmup,
                                    dspmm_stream_t stream) {
    if (warmup < 0) return DSPMM_STATUS_INVALID_VALUE;
    dspmm_status_t st = DSPMM_STATUS_SUCCESS;
    for (int i = 0; i < warmup && st == DSPMM_STATUS_SUCCESS; i++)
        st = dspmm_spmm(alg, layout, nr, nc, nnz, nv, rowPtr, rowIdx, colIdx, values, dnInput,
                        dnOutput, stream);
    if (st != DSPMM_STATUS_SUCCESS) return st;
    st = hip_status(hipStreamSynchronize(as_hip(stream)));
    if (st != DSPMM_STATUS_SUCCESS) return st;
    roctxProfilerResume(0);
    roctxRangePushA("dspmm_dry_run");
    st = dspmm_spmm(alg, layout, nr, nc, nnz, nv, rowPtr, rowIdx, colIdx, values, dnInput,
                    dnOutput, stream);
    dspmm_status_t st2 = hip_status(hipStreamSynchronize(as_hip(stream)));
    roctxRangePop();
    roctxProfilerPause(0);
    return st != DSPMM_STATUS_SUCCESS ? st : st2;
}

}  // extern "C"

// C-ABI entry points of libinti_amd (declared in include/inti_amd.h):
// context / stream / profiling, quadrature upload, operators, corrections.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "apply_sym.hpp"
#include "common.hpp"

namespace inti {

static thread_local std::string g_create_err;

// Partial sums of the allocation-free apply (inti_op_apply_device_noalloc):
// a static buffer that every GPU the library runs on holds from load until
// the process ends. Host code never uses this name as an address: it is a
// host-side stand-in; the device address is looked up once per context with
// hipGetSymbolAddress (Ctx::noalloc_scratch).
constexpr size_t kNoAllocBytes = size_t(64) << 20;
static __device__ __align__(256) double scratch[kNoAllocBytes / sizeof(double)];

int set_error(Ctx *ctx, int code, const std::string &msg) {
    if (ctx) ctx->err = msg;
    else g_create_err = msg;
    return code;
}

int ctx_scratch(Ctx *ctx, int slot, size_t bytes, void **ptr) {
    if (bytes == 0) bytes = 256;
    if (ctx->scratch_bytes[slot] < bytes) {
        if (ctx->scratch[slot]) {
            INTI_HIP(ctx, hipStreamSynchronize(ctx->stream));
            INTI_HIP(ctx, hipFree(ctx->scratch[slot]));
            ctx->scratch[slot] = nullptr;
            ctx->scratch_bytes[slot] = 0;
        }
        size_t want = bytes + bytes / 4;
        if (hipMalloc(&ctx->scratch[slot], want) != hipSuccess) {
            ctx->scratch[slot] = nullptr;
            return set_error(ctx, INTI_ERR_NOMEM, "scratch allocation failed");
        }
        ctx->scratch_bytes[slot] = want;
    }
    *ptr = ctx->scratch[slot];
    return INTI_OK;
}

Arena::~Arena() {
    if (!live) return;
    (void)hipStreamSynchronize(ctx->stream);
    if (own) (void)hipFree(own);
}

int Arena::commit() {
    size_t total = 0;
    for (const Cut &c : cuts) total += (c.bytes + 255) / 256 * 256;
    void *at = nullptr;
    if (total <= kArenaKeep) {
        if (int st = ctx_scratch(ctx, kScrArena, total, &at)) return st;
    } else {
        if (hipMalloc(&own, total) != hipSuccess) {
            own = nullptr;
            return set_error(ctx, INTI_ERR_NOMEM, "device allocation failed");
        }
        at = own;
    }
    live = true;
    for (const Cut &c : cuts) {
        *c.p = at;
        at = (char *)at + (c.bytes + 255) / 256 * 256;
    }
    return INTI_OK;
}

int csr_alloc(Ctx *ctx, int64_t m, int64_t n, int64_t nnz, int cplx, Csr **out) {
    Csr *c = new inti_csr();
    c->ctx = ctx; c->m = m; c->n = n; c->nnz = nnz; c->is_complex = cplx;
    if (hipMalloc(&c->rowptr, sizeof(int32_t) * (m + 1)) != hipSuccess ||
        hipMalloc(&c->colind, sizeof(int32_t) * (nnz > 0 ? nnz : 1)) != hipSuccess ||
        hipMalloc(&c->val, sizeof(double) * (cplx ? 2 : 1) * (nnz > 0 ? nnz : 1)) != hipSuccess) {
        if (c->rowptr) (void)hipFree(c->rowptr);
        if (c->colind) (void)hipFree(c->colind);
        if (c->val) (void)hipFree(c->val);
        delete static_cast<inti_csr *>(c);
        return set_error(ctx, INTI_ERR_NOMEM, "CSR allocation failed");
    }
    *out = c;
    return INTI_OK;
}

void csr_free(Csr *c) {
    if (!c) return;
    if (c->rowptr) (void)hipFree(c->rowptr);
    if (c->colind) (void)hipFree(c->colind);
    if (c->val) (void)hipFree(c->val);
    delete static_cast<inti_csr *>(c);
}

void op_free_correction(Op *op) {
    csr_free(op->corr);
    op->corr = nullptr;
    if (op->corr_tptr) (void)hipFree(op->corr_tptr);  // one allocation for the three
    op->corr_tptr = op->corr_trow = op->corr_tperm = nullptr;
}

// Transposed pattern of an attached correction for the adjoint's gather (rows
// increasing within a column), built on the GPU by the attach. A pattern equal to
// its transpose (each element's own nodes) takes one kernel, which looks up entry
// (j, i) in row j for every (i, j) and sets *flag where it is missing; any other
// is sorted: entries counted per column, the counts summed, entries dropped into
// their columns in any order, and each column sorted by its entries' positions in
// the CSR. The host's counting sort took 280 us of an attach at 12,000 nodes
// (63,480: 700); the one kernel adds 9 (10), the sort's five 35 (50).
constexpr int64_t kOwnRow = 32;  // average entries per row up to which the lookup is tried

__global__ __launch_bounds__(256) void k_own_transpose(int64_t n, const int32_t *rowptr, const int32_t *colind,
                                                       int32_t *tptr, int32_t *trow, int32_t *tperm, int *flag) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int32_t p0 = rowptr[i], p1 = rowptr[i + 1];
    tptr[i] = p0;
    if (i == n - 1) tptr[n] = p1;
    bool bad = false;
    for (int32_t p = p0; p < p1; ++p) {
        const int32_t j = colind[p], q1 = rowptr[j + 1];
        int32_t q = rowptr[j];
        while (q < q1 && colind[q] != (int32_t)i) ++q;
        bad |= q == q1 || (p > p0 && colind[p - 1] >= j);
        trow[p] = j;
        tperm[p] = q;
    }
    if (bad) *flag = 1;
}

__global__ __launch_bounds__(256) void k_col_count(int64_t nnz, const int32_t *colind, int32_t *count) {
    const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (q < nnz) atomicAdd(&count[colind[q]], 1);
}

// sums of 1024 counts each
__global__ __launch_bounds__(256) void k_col_sums(int64_t n, const int32_t *count, int32_t *sums) {
    __shared__ int32_t s_sum[4];
    const int tid = threadIdx.x;
    int32_t v = 0;
    for (int t = 0; t < 4; ++t) {
        const int64_t j = (int64_t)blockIdx.x * 1024 + t * 256 + tid;
        v += j < n ? count[j] : 0;
    }
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if ((tid & 63) == 0) s_sum[tid >> 6] = v;
    __syncthreads();
    if (tid == 0) sums[blockIdx.x] = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3];
}

// tptr = the exclusive sums of fill (counts), which becomes their copy: a block
// takes 1024 columns and adds up the sums of the blocks before it itself
__global__ __launch_bounds__(1024) void k_col_scan(int64_t n, const int32_t *sums, int32_t *fill, int32_t *tptr) {
    __shared__ int32_t s_sum[1024];
    const int tid = threadIdx.x;
    const int64_t j = (int64_t)blockIdx.x * 1024 + tid;
    int32_t before = 0;
    for (int b = tid; b < (int)blockIdx.x; b += 1024) before += sums[b];
    const int32_t cnt = j < n ? fill[j] : 0;
    s_sum[tid] = before;
    __syncthreads();
    for (int off = 512; off > 0; off >>= 1) {
        if (tid < off) s_sum[tid] += s_sum[tid + off];
        __syncthreads();
    }
    before = s_sum[0];
    __syncthreads();
    s_sum[tid] = cnt;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        const int32_t add = tid >= off ? s_sum[tid - off] : 0;
        __syncthreads();
        s_sum[tid] += add;
        __syncthreads();
    }
    const int32_t end = before + s_sum[tid];
    if (j < n) {
        fill[j] = end - cnt;
        tptr[j] = end - cnt;
    }
    if (j == n - 1) tptr[n] = end;
}

__global__ __launch_bounds__(256) void k_col_fill(int64_t m, const int32_t *rowptr, const int32_t *colind, int32_t *fill,
                                                  int32_t *trow, int32_t *tperm) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= m) return;
    for (int32_t q = rowptr[i]; q < rowptr[i + 1]; ++q) {
        const int32_t p = atomicAdd(&fill[colind[q]], 1);
        trow[p] = (int32_t)i;
        tperm[p] = q;
    }
}

// a thread per column: insertion for the usual few entries (nearly in order
// already), heap sort for long columns
__global__ __launch_bounds__(256) void k_col_sort(int64_t n, const int32_t *tptr, int32_t *trow, int32_t *tperm) {
    const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (j >= n) return;
    const int32_t len = tptr[j + 1] - tptr[j];
    int32_t *key = tperm + tptr[j], *row = trow + tptr[j];
    if (len <= 48) {
        for (int32_t a = 1; a < len; ++a) {
            const int32_t k = key[a], r = row[a];
            int32_t b = a;
            for (; b > 0 && key[b - 1] > k; --b) {
                key[b] = key[b - 1];
                row[b] = row[b - 1];
            }
            key[b] = k;
            row[b] = r;
        }
        return;
    }
    for (int32_t start = len / 2, end = len; end > 1;) {
        int32_t k, r;
        if (start > 0) {  // make the heap
            --start;
            k = key[start];
            r = row[start];
        } else {  // its largest to the end
            --end;
            k = key[end];
            r = row[end];
            key[end] = key[0];
            row[end] = row[0];
        }
        int32_t hole = start;
        for (int32_t child = 2 * hole + 1; child < end; child = 2 * hole + 1) {
            if (child + 1 < end && key[child + 1] > key[child]) ++child;
            if (key[child] <= k) break;
            key[hole] = key[child];
            row[hole] = row[child];
            hole = child;
        }
        key[hole] = k;
        row[hole] = r;
    }
}

// The pattern of op->corr transposed: enqueued on ctx->stream; with `own` the
// lookup, whose *ctx->flag the caller reads after its wait, else the sort
static int transpose_pattern(Op *op, bool own) {
    Ctx *ctx = op->ctx;
    const Csr *c = op->corr;
    const int64_t m = c->m, n = c->n, nnz = c->nnz, nb = (n + 1023) / 1024;
    const size_t ib = sizeof(int32_t), most = std::max<size_t>((size_t)nnz, 1);
    if (!op->corr_tptr && hipMalloc((void **)&op->corr_tptr, ib * ((size_t)(n + 1) + 2 * most)) != hipSuccess) {
        op->corr_tptr = nullptr;
        return set_error(ctx, INTI_ERR_NOMEM, "attach: transposed pattern allocation failed");
    }
    op->corr_trow = op->corr_tptr + n + 1;
    op->corr_tperm = op->corr_trow + most;
    if (n == 0) return INTI_OK;  // no column to read
    hipStream_t s = ctx->stream;
    if (own) {
        *ctx->flag = 0;
        hipLaunchKernelGGL(k_own_transpose, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, c->rowptr, c->colind,
                           op->corr_tptr, op->corr_trow, op->corr_tperm, ctx->flag);
        INTI_HIP(ctx, hipGetLastError());
        return INTI_OK;
    }
    void *scr = nullptr;
    if (int st = ctx_scratch(ctx, kScrArena, ib * (size_t)(n + nb), &scr)) return st;
    int32_t *fill = (int32_t *)scr, *sums = fill + n;
    INTI_HIP(ctx, hipMemsetAsync(fill, 0, ib * (size_t)n, s));
    if (nnz > 0)
        hipLaunchKernelGGL(k_col_count, dim3((unsigned)((nnz + 255) / 256)), dim3(256), 0, s, nnz, c->colind, fill);
    hipLaunchKernelGGL(k_col_sums, dim3((unsigned)nb), dim3(256), 0, s, n, fill, sums);
    hipLaunchKernelGGL(k_col_scan, dim3((unsigned)nb), dim3(1024), 0, s, n, sums, fill, op->corr_tptr);
    if (nnz > 0) {
        hipLaunchKernelGGL(k_col_fill, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, s, m, c->rowptr, c->colind,
                           fill, op->corr_trow, op->corr_tperm);
        hipLaunchKernelGGL(k_col_sort, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, op->corr_tptr, op->corr_trow,
                           op->corr_tperm);
    }
    INTI_HIP(ctx, hipGetLastError());
    return INTI_OK;
}

// ------------------------------------------------------- coincident nodes
// A quadrature's nodes are "distinct" if every two of them are farther apart
// than 2e-14 (twice the coincidence tolerance, so that rounding differences
// between this test and the kernels' own distances cannot matter).
// Coordinates of 1e5 and beyond (and NaN) count as not distinct, which only
// keeps the mask of the pair kernels. Only operators on one quadrature ask
// (quad_distinct): point sets that are targets alone never pay for it.
//
// The bounding boxes of tiles of 256 nodes, then every pair of tiles whose
// boxes touch: consecutive nodes are neighbours on the surface, so nearly all
// pairs of tiles are dismissed by their boxes; nodes in random order cost
// n^2 / 2 distances (63,480 nodes: 0.5 ms). It replaced a sort and search of
// cells of 4e-14 on the host, 0.28 us per node and per upload (11 ms for a
// plotting grid of 40,401 points).
constexpr double kDistinctTol2 = 4.0e-28;
constexpr double kDistinctBox = 4.0e-14;  // boxes farther apart than this are dismissed
constexpr double kDistinctMax = 1.0e5;

template <int DIM>
__global__ __launch_bounds__(kSymBS) void k_tile_boxes(int64_t n, const double *c, double *box, int *flag) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    __shared__ double s_lo[kSymBS / 64][DIM], s_hi[kSymBS / 64][DIM];
    const int64_t i = (int64_t)blockIdx.x * kSymBS + tid;
    const int64_t ic = i < n ? i : n - 1;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        double lo = c[d * n + ic], hi = lo;
        if (!(fabs(lo) < kDistinctMax)) *flag = 1;
        for (int o = 32; o > 0; o >>= 1) {
            lo = fmin(lo, __shfl_xor(lo, o));
            hi = fmax(hi, __shfl_xor(hi, o));
        }
        if (lane == 0) { s_lo[wave][d] = lo; s_hi[wave][d] = hi; }
    }
    __syncthreads();
    if (tid < DIM) {
        double lo = s_lo[0][tid], hi = s_hi[0][tid];
        for (int w = 1; w < kSymBS / 64; ++w) {
            lo = fmin(lo, s_lo[w][tid]);
            hi = fmax(hi, s_hi[w][tid]);
        }
        box[(int64_t)blockIdx.x * 2 * DIM + tid] = lo;
        box[(int64_t)blockIdx.x * 2 * DIM + DIM + tid] = hi;
    }
}

// pairs of tiles [first, first + gridDim.x) of the row-major upper triangle
template <int DIM>
__global__ __launch_bounds__(kSymBS) void k_close_pairs(int64_t n, int64_t T, int64_t first, const double *c,
                                                        const double *box, int *flag) {
    __shared__ double s_y[DIM][kSymBS];
    int64_t a, b;
    sym_item(first + blockIdx.x, T, a, b);
    const double *ba = box + a * 2 * DIM, *bb = box + b * 2 * DIM;
#pragma unroll
    for (int d = 0; d < DIM; ++d)
        if (ba[d] > bb[DIM + d] + kDistinctBox || bb[d] > ba[DIM + d] + kDistinctBox) return;  // the whole block
    const int tid = threadIdx.x;
    const int64_t i = a * kSymBS + tid, j0 = b * kSymBS;
    const int64_t ic = i < n ? i : n - 1, jc = j0 + tid < n ? j0 + tid : n - 1;
    double x[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        x[d] = c[d * n + ic];
        s_y[d][tid] = c[d * n + jc];
    }
    __syncthreads();
    if (i >= n) return;
    const int cnt = (int)(n - j0 < kSymBS ? n - j0 : kSymBS);
    bool close = false;
    for (int q = 0; q < cnt; ++q) {
        double d2 = 0.0;
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            const double t = x[d] - s_y[d][q];
            d2 = __builtin_fma(t, t, d2);
        }
        close |= d2 <= kDistinctTol2 && j0 + q != i;
    }
    if (close) *flag = 1;
}

// Creating an operator must not disturb captures: with the thread's capture
// mode relaxed, the allocation, the copies and the wait below are allowed while
// other streams are being captured (in the global mode hipMalloc is refused
// then and ends their capture). The quadrature's device is made current.
struct OutsideCaptures {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    int device = 0;
    bool moved = false;
    hipError_t err;
    explicit OutsideCaptures(int dev) {
        err = hipThreadExchangeStreamCaptureMode(&mode);
        if (err == hipSuccess) err = hipGetDevice(&device);
        if (err == hipSuccess && device != dev) {
            err = hipSetDevice(dev);
            moved = err == hipSuccess;
        }
    }
    ~OutsideCaptures() {
        if (moved) (void)hipSetDevice(device);
        (void)hipThreadExchangeStreamCaptureMode(&mode);
    }
};

// Decides q->distinct once, on the stream of the quadrature's context (locked
// by the caller). While that stream is being captured nothing is launched and
// the question stays open: the mask is kept, and the next operator asks again.
static int quad_distinct(const Quad *q) {
    Ctx *ctx = q->ctx;
    if (q->distinct_known) return INTI_OK;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    INTI_HIP(ctx, hipStreamIsCapturing(ctx->stream, &cap));
    if (cap != hipStreamCaptureStatusNone) return INTI_OK;
    OutsideCaptures outside(ctx->device);
    INTI_HIP(ctx, outside.err);
    const int64_t n = q->n, T = (n + kSymBS - 1) / kSymBS;
    int flag = 0;
    if (n > 0) {
        struct Buf {
            void *p = nullptr;
            ~Buf() { if (p) (void)hipFree(p); }
        } buf;
        const size_t nbox = 2 * (size_t)q->dim * (size_t)T;
        if (hipMalloc(&buf.p, sizeof(double) * nbox + sizeof(int)) != hipSuccess)
            return set_error(ctx, INTI_ERR_NOMEM, "op_create: allocation failed");
        double *box = (double *)buf.p;
        int *dflag = (int *)(box + nbox);
        hipStream_t s = ctx->stream;
        INTI_HIP(ctx, hipMemcpyAsync(dflag, &flag, sizeof(int), hipMemcpyHostToDevice, s));
        // a launch holds fewer than 2^32 threads (1,483,008 nodes need more)
        const int64_t pairs = T * (T + 1) / 2, most = (int64_t(1) << 32) / kSymBS - 1;
        if (q->dim == 2) hipLaunchKernelGGL(k_tile_boxes<2>, dim3((unsigned)T), dim3(kSymBS), 0, s, n, q->coords, box, dflag);
        else hipLaunchKernelGGL(k_tile_boxes<3>, dim3((unsigned)T), dim3(kSymBS), 0, s, n, q->coords, box, dflag);
        for (int64_t f = 0; f < pairs; f += most) {
            const dim3 g((unsigned)std::min(most, pairs - f));
            if (q->dim == 2) hipLaunchKernelGGL(k_close_pairs<2>, g, dim3(kSymBS), 0, s, n, T, f, q->coords, box, dflag);
            else hipLaunchKernelGGL(k_close_pairs<3>, g, dim3(kSymBS), 0, s, n, T, f, q->coords, box, dflag);
        }
        const hipError_t launched = hipGetLastError();
        // the flag's copy and the buffer end before either leaves scope
        const hipError_t copied = hipMemcpyAsync(&flag, dflag, sizeof(int), hipMemcpyDeviceToHost, s);
        const hipError_t done = hipStreamSynchronize(s);
        INTI_HIP(ctx, launched);
        INTI_HIP(ctx, copied);
        INTI_HIP(ctx, done);
    }
    q->distinct = flag == 0;
    q->distinct_known = true;
    return INTI_OK;
}

int bdim_build(Op *opS, Op *opD, int deriv, int nq, int64_t ne, const int64_t *qtags,
               const int64_t *near_ptr, const int64_t *near_idx, const double *mu,
               const double *params, Csr **outS, Csr **outD, double *diag_out);
int bdim_build_types(Op *opS, Op *opD, int deriv, int ntypes, const int *nq, const int64_t *ne,
                     const int64_t *qtags, const int64_t *near_ptr, const int64_t *near_idx, const double *mu,
                     const double *params, Csr **outS, Csr **outD, double *diag_out);
int lsq_build_types(Ctx *ctx, int cplx, int nrows, int ntypes, const int *ncols, const int64_t *ne, const double *A,
                    const int64_t *cols, int64_t m, int64_t n, const int64_t *near_ptr, const int64_t *near_idx,
                    const double *rhs, Csr **out, double *diag_out);
int lsq_build(Ctx *ctx, int cplx, int nrows, int ncols, int64_t ne, const double *A, const int64_t *cols,
              int64_t m, int64_t n, const int64_t *near_ptr, const int64_t *near_idx, const double *rhs,
              Csr **out, double *diag_out);

}  // namespace inti

using namespace inti;

#define LOCK(ctx) std::lock_guard<std::mutex> lock_((ctx)->mu)
#define REQUIRE(ctx, cond, msg) \
    do { if (!(cond)) return set_error((ctx), INTI_ERR_ARG, (msg)); } while (0)

extern "C" {

int inti_version(void) { return 100; }

int inti_ctx_create(int device, inti_ctx **out) {
    if (!out) return set_error(nullptr, INTI_ERR_ARG, "out is null");
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count == 0)
        return set_error(nullptr, INTI_ERR_HIP, "no HIP device available");
    if (device < 0 || device >= count) return set_error(nullptr, INTI_ERR_ARG, "device out of range");
    if (hipSetDevice(device) != hipSuccess) return set_error(nullptr, INTI_ERR_HIP, "hipSetDevice failed");
    inti_ctx *c = new inti_ctx();
    c->device = device;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) == hipSuccess) c->num_cu = prop.multiProcessorCount;
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreate(&c->ev0) != hipSuccess || hipEventCreate(&c->ev1) != hipSuccess ||
        hipHostMalloc((void **)&c->flag, sizeof(int), hipHostMallocMapped) != hipSuccess) {
        delete c;
        return set_error(nullptr, INTI_ERR_HIP, "stream/event creation failed");
    }
    // this device's copy of the static partial-sum buffer (the device is
    // current here)
    void *sp = nullptr;
    const hipError_t se = hipGetSymbolAddress(&sp, HIP_SYMBOL(scratch));
    if (se != hipSuccess || sp == nullptr) {
        (void)hipHostFree(c->flag);
        (void)hipEventDestroy(c->ev0);
        (void)hipEventDestroy(c->ev1);
        (void)hipStreamDestroy(c->stream);
        delete c;
        return set_error(nullptr, INTI_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(se));
    }
    c->noalloc_scratch = (double *)sp;
    *out = c;
    return INTI_OK;
}

int inti_ctx_destroy(inti_ctx *ctx) {
    if (!ctx) return INTI_ERR_ARG;
    (void)hipSetDevice(ctx->device);
    (void)hipStreamSynchronize(ctx->stream);
    for (int s = 0; s < Ctx::kSlots; ++s)
        if (ctx->scratch[s]) (void)hipFree(ctx->scratch[s]);
    (void)hipHostFree(ctx->flag);
    (void)hipEventDestroy(ctx->ev0);
    (void)hipEventDestroy(ctx->ev1);
    (void)hipStreamDestroy(ctx->stream);
    delete ctx;
    return INTI_OK;
}

const char *inti_last_error(const inti_ctx *ctx) {
    return ctx ? ctx->err.c_str() : g_create_err.c_str();
}

int inti_microbench(inti_ctx *ctx, int op, double *rate) {
    if (!ctx) return INTI_ERR_ARG;
    REQUIRE(ctx, rate != nullptr, "microbench: rate is null");
    LOCK(ctx);
    return microbench(ctx, op, rate);
}

int inti_ctx_synchronize(inti_ctx *ctx) {
    if (!ctx) return INTI_ERR_ARG;
    INTI_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return INTI_OK;
}

int inti_ctx_stream(inti_ctx *ctx, void **stream) {
    if (!ctx || !stream) return INTI_ERR_ARG;
    *stream = (void *)ctx->stream;
    return INTI_OK;
}

int inti_ctx_set_profiling(inti_ctx *ctx, int on) {
    if (!ctx) return INTI_ERR_ARG;
    ctx->profiling = on ? 1 : 0;
    return INTI_OK;
}

int inti_ctx_last_kernel_ms(inti_ctx *ctx, double *ms) {
    if (!ctx || !ms) return INTI_ERR_ARG;
    LOCK(ctx);
    INTI_HIP(ctx, hipEventSynchronize(ctx->ev1));
    float t = 0.f;
    INTI_HIP(ctx, hipEventElapsedTime(&t, ctx->ev0, ctx->ev1));
    *ms = t;
    return INTI_OK;
}

int inti_device_alloc(inti_ctx *ctx, size_t bytes, void **dptr) {
    if (!ctx || !dptr) return INTI_ERR_ARG;
    if (hipMalloc(dptr, bytes ? bytes : 1) != hipSuccess)
        return set_error(ctx, INTI_ERR_NOMEM, "device allocation failed");
    return INTI_OK;
}

int inti_device_free(inti_ctx *ctx, void *dptr) {
    if (!ctx) return INTI_ERR_ARG;
    LOCK(ctx);
    INTI_HIP(ctx, hipStreamSynchronize(ctx->stream));
    INTI_HIP(ctx, hipFree(dptr));
    return INTI_OK;
}

int inti_memcpy_h2d(inti_ctx *ctx, void *dst, const void *src, size_t bytes) {
    if (!ctx || (!dst && bytes) || (!src && bytes)) return INTI_ERR_ARG;
    LOCK(ctx);
    INTI_HIP(ctx, hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, ctx->stream));
    INTI_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return INTI_OK;
}

int inti_memcpy_d2h(inti_ctx *ctx, void *dst, const void *src, size_t bytes) {
    if (!ctx || (!dst && bytes) || (!src && bytes)) return INTI_ERR_ARG;
    LOCK(ctx);
    INTI_HIP(ctx, hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
    INTI_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return INTI_OK;
}

__global__ __launch_bounds__(256) void k_copy16(const double2 *__restrict__ src,
                                                 double2 *__restrict__ dst, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
        dst[i] = src[i];
}

int inti_device_copy(inti_ctx *ctx, void *dst, const void *src, size_t bytes) {
    if (!ctx) return INTI_ERR_ARG;
    REQUIRE(ctx, bytes % 16 == 0, "device_copy: bytes must be a multiple of 16");
    REQUIRE(ctx, bytes == 0 || (dst && src), "device_copy: null pointer");
    LOCK(ctx);
    const int64_t n = (int64_t)(bytes / 16);
    if (n == 0) return INTI_OK;
    int64_t blocks = (n + 255) / 256;
    if (blocks > 8 * 1024) blocks = 8 * 1024;
    hipLaunchKernelGGL(k_copy16, dim3((unsigned)blocks), dim3(256), 0, ctx->stream,
                       (const double2 *)src, (double2 *)dst, n);
    INTI_HIP(ctx, hipGetLastError());
    INTI_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return INTI_OK;
}

// ------------------------------------------------------------- quadrature
int inti_quad_upload(inti_ctx *ctx, int dim, int64_t n, const double *coords,
                     const double *normals, const double *weights, inti_quad **out) {
    if (!ctx) return INTI_ERR_ARG;
    REQUIRE(ctx, out != nullptr, "quad_upload: out is null");
    REQUIRE(ctx, dim == 2 || dim == 3, "quad_upload: dim must be 2 or 3");
    REQUIRE(ctx, n >= 0, "quad_upload: negative size");
    REQUIRE(ctx, n == 0 || (coords && weights), "quad_upload: coords and weights are required");
    LOCK(ctx);
    inti_quad *q = new inti_quad();
    q->ctx = ctx; q->dim = dim; q->n = n;
    const size_t cb = sizeof(double) * dim * (n > 0 ? n : 1);
    if (hipMalloc(&q->coords, cb) != hipSuccess ||
        hipMalloc(&q->weights, sizeof(double) * (n > 0 ? n : 1)) != hipSuccess ||
        (normals && hipMalloc(&q->normals, cb) != hipSuccess)) {
        if (q->coords) (void)hipFree(q->coords);
        if (q->weights) (void)hipFree(q->weights);
        if (q->normals) (void)hipFree(q->normals);
        delete q;
        return set_error(ctx, INTI_ERR_NOMEM, "quad_upload: allocation failed");
    }
    if (n > 0) {
        INTI_HIP(ctx, hipMemcpyAsync(q->coords, coords, sizeof(double) * dim * n, hipMemcpyHostToDevice, ctx->stream));
        INTI_HIP(ctx, hipMemcpyAsync(q->weights, weights, sizeof(double) * n, hipMemcpyHostToDevice, ctx->stream));
        if (normals)
            INTI_HIP(ctx, hipMemcpyAsync(q->normals, normals, sizeof(double) * dim * n, hipMemcpyHostToDevice, ctx->stream));
        for (int d = 0; d < dim; ++d) {
            double lo = coords[(int64_t)d * n], hi = lo;
            for (int64_t i = 1; i < n; ++i) {
                lo = std::min(lo, coords[(int64_t)d * n + i]);
                hi = std::max(hi, coords[(int64_t)d * n + i]);
            }
            q->lo[d] = lo; q->hi[d] = hi;
        }
        INTI_HIP(ctx, hipStreamSynchronize(ctx->stream));
    }
    *out = q;
    return INTI_OK;
}

int inti_quad_destroy(inti_quad *q) {
    if (!q) return INTI_ERR_ARG;
    Ctx *ctx = q->ctx;
    {
        LOCK(ctx);
        (void)hipStreamSynchronize(ctx->stream);
        if (q->coords) (void)hipFree(q->coords);
        if (q->weights) (void)hipFree(q->weights);
        if (q->normals) (void)hipFree(q->normals);
    }
    delete q;
    return INTI_OK;
}

// --------------------------------------------------------------- operator
int inti_op_create(inti_ctx *ctx, int pde, int kind, int dim, double k, const double *coefs,
                   const inti_quad *trg, const inti_quad *src, int precision, inti_op **out) {
    if (!ctx) return INTI_ERR_ARG;
    REQUIRE(ctx, out && trg && src, "op_create: null argument");
    REQUIRE(ctx, pde == INTI_LAPLACE || pde == INTI_HELMHOLTZ, "op_create: unknown pde");
    REQUIRE(ctx, kind >= INTI_SL && kind <= INTI_FF_COMB, "op_create: unknown kernel kind");
    const bool farfield = kind >= INTI_FF_SL;
    if (farfield && pde != INTI_HELMHOLTZ)
        return set_error(ctx, INTI_ERR_UNSUPPORTED, "op_create: far-field kinds are Helmholtz only");
    REQUIRE(ctx, dim == 2 || dim == 3, "op_create: dim must be 2 or 3");
    REQUIRE(ctx, precision == INTI_FP64 || precision == INTI_MIXED, "op_create: unknown precision");
    // IntegralOperator(k, X, Y) requires equal dimensions (src/nystrom.jl:79-85)
    if (trg->dim != dim || src->dim != dim)
        return set_error(ctx, INTI_ERR_SIZE, "op_create: quadrature dimension differs from the operator's");
    const bool needs_src_n = kind != INTI_SL && kind != INTI_ADL && kind != INTI_FF_SL;
    const bool needs_trg_n = kind == INTI_ADL || kind == INTI_HS || kind == INTI_COMB_AH;
    if (needs_src_n && !src->normals)
        return set_error(ctx, INTI_ERR_ARG, "op_create: this kernel needs source normals");
    if (needs_trg_n && !trg->normals)
        return set_error(ctx, INTI_ERR_ARG, "op_create: this kernel needs target normals");
    if (pde == INTI_HELMHOLTZ) REQUIRE(ctx, k > 0.0 && std::isfinite(k), "op_create: Helmholtz needs a real k > 0");
    const bool comb = kind == INTI_COMB_SD || kind == INTI_COMB_AH || kind == INTI_FF_COMB;
    if (comb) {
        REQUIRE(ctx, coefs != nullptr, "op_create: combined kinds need coefs");
        if (pde == INTI_LAPLACE && (coefs[1] != 0.0 || coefs[3] != 0.0))
            return set_error(ctx, INTI_ERR_UNSUPPORTED, "op_create: Laplace combinations take real coefficients");
    }
    if (trg == src && !farfield) {  // the symmetric sums ask whether the nodes are distinct
        LOCK(src->ctx);
        if (int st = quad_distinct(src)) return st;
    }
    inti_op *op = new inti_op();
    op->ctx = ctx; op->pde = pde; op->kind = kind; op->dim = dim; op->k = k;
    op->precision = precision; op->trg = trg; op->src = src;
    if (comb) std::memcpy(op->coefs, coefs, sizeof(double) * 4);
    *out = op;
    return INTI_OK;
}

int inti_op_destroy(inti_op *op) {
    if (!op) return INTI_ERR_ARG;
    {
        LOCK(op->ctx);
        (void)hipStreamSynchronize(op->ctx->stream);
        op_free_correction(op);
    }
    delete op;
    return INTI_OK;
}

int inti_op_set_identity(inti_op *op, double re, double im) {
    if (!op) return INTI_ERR_ARG;
    if (op->trg->n != op->src->n)
        return set_error(op->ctx, INTI_ERR_SIZE, "op_set_identity: operator is not square");
    if (op->pde == INTI_LAPLACE && im != 0.0)
        return set_error(op->ctx, INTI_ERR_UNSUPPORTED, "op_set_identity: Laplace takes a real coefficient");
    op->cid[0] = re; op->cid[1] = im;
    return INTI_OK;
}

int inti_op_set_wavenumber_imag(inti_op *op, double kimag) {
    if (!op) return INTI_ERR_ARG;
    Ctx *ctx = op->ctx;
    REQUIRE(ctx, std::isfinite(kimag), "op_set_wavenumber_imag: kimag must be finite");
    if (kimag != 0.0) {
        if (op->pde != INTI_HELMHOLTZ || op->dim != 3)
            return set_error(ctx, INTI_ERR_UNSUPPORTED, "op_set_wavenumber_imag: complex wavenumbers are 3D Helmholtz only");
        if (op->kind >= INTI_FF_SL)
            return set_error(ctx, INTI_ERR_UNSUPPORTED, "op_set_wavenumber_imag: no far-field kernels for complex wavenumbers");
        if (op->precision != INTI_FP64)
            return set_error(ctx, INTI_ERR_UNSUPPORTED, "op_set_wavenumber_imag: complex wavenumbers run in FP64");
    }
    LOCK(ctx);
    op->kimag = kimag;
    return INTI_OK;
}

int inti_op_set_launch(inti_op *op, int block, int tpt, int split) {
    if (!op) return INTI_ERR_ARG;
    if (block != 256 || tpt != 1 || split < 0)
        return set_error(op->ctx, INTI_ERR_UNSUPPORTED, "op_set_launch: block 256, tpt 1, split >= 0");
    op->block = block; op->tpt = tpt; op->split = split;
    return INTI_OK;
}

int inti_op_set_symmetric(inti_op *op, int mode, int group) {
    if (!op) return INTI_ERR_ARG;
    if (mode < 0 || mode > 2) return set_error(op->ctx, INTI_ERR_ARG, "op_set_symmetric: mode 0, 1 or 2");
    if (group != 0 && group != 1 && group != 2 && group != 4)
        return set_error(op->ctx, INTI_ERR_ARG, "op_set_symmetric: group 0, 1, 2 or 4");
    op->sym = mode;
    op->sym_group = group;
    return INTI_OK;
}

static int apply_device_locked(inti_op *op, int nrhs, const double *x, int64_t ldx, double *y,
                               int64_t ldy, const double *alpha, const double *beta) {
    DirectLaunch L;
    L.op = op; L.nrhs = nrhs; L.x = x; L.ldx = ldx; L.y = y; L.ldy = ldy;
    L.alpha[0] = alpha ? alpha[0] : 1.0; L.alpha[1] = alpha ? alpha[1] : 0.0;
    L.beta[0] = beta ? beta[0] : 0.0; L.beta[1] = beta ? beta[1] : 0.0;
    if (op->pde == INTI_LAPLACE && (L.alpha[1] != 0.0 || L.beta[1] != 0.0))
        return set_error(op->ctx, INTI_ERR_UNSUPPORTED, "apply: Laplace operators take real alpha/beta");
    return launch_apply(L);
}

int inti_op_apply_device(inti_op *op, int nrhs, const double *x, int64_t ldx, double *y,
                         int64_t ldy, const double *alpha, const double *beta) {
    if (!op) return INTI_ERR_ARG;
    Ctx *ctx = op->ctx;
    REQUIRE(ctx, nrhs >= 0, "apply: nrhs < 0");
    REQUIRE(ctx, nrhs == 0 || (x && y), "apply: null operand");
    REQUIRE(ctx, ldx >= op->src->n && ldy >= op->trg->n, "apply: leading dimension too small");
    LOCK(ctx);
    return apply_device_locked(op, nrhs, x, ldx, y, ldy, alpha, beta);
}

int inti_op_apply_device_noalloc(inti_op *op, int nrhs, const double *x, int64_t ldx, double *y,
                                 int64_t ldy, const double *alpha, const double *beta) {
    if (!op) return INTI_ERR_ARG;
    Ctx *ctx = op->ctx;
    REQUIRE(ctx, nrhs >= 0, "apply_noalloc: nrhs < 0");
    REQUIRE(ctx, nrhs == 0 || (x && y), "apply_noalloc: null operand");
    REQUIRE(ctx, ldx >= op->src->n && ldy >= op->trg->n, "apply_noalloc: leading dimension too small");
    if (!ctx->noalloc_scratch) return set_error(ctx, INTI_ERR_HIP, "apply_noalloc: no scratch address");
    LOCK(ctx);
    DirectLaunch L;
    L.op = op; L.nrhs = nrhs; L.x = x; L.ldx = ldx; L.y = y; L.ldy = ldy;
    L.alpha[0] = alpha ? alpha[0] : 1.0; L.alpha[1] = alpha ? alpha[1] : 0.0;
    L.beta[0] = beta ? beta[0] : 0.0; L.beta[1] = beta ? beta[1] : 0.0;
    if (op->pde == INTI_LAPLACE && (L.alpha[1] != 0.0 || L.beta[1] != 0.0))
        return set_error(ctx, INTI_ERR_UNSUPPORTED, "apply_noalloc: Laplace operators take real alpha/beta");
    // every partial slot the reduction reads is written by the sum of the
    // same call (each block writes its own chunk's partial of every row of
    // its tile): nothing needs clearing between calls
    L.part = ctx->noalloc_scratch;
    L.part_bytes = kNoAllocBytes;
    return launch_apply(L);
}

int inti_op_apply(inti_op *op, int nrhs, const double *x, double *y, const double *alpha,
                  const double *beta) {
    if (!op) return INTI_ERR_ARG;
    Ctx *ctx = op->ctx;
    REQUIRE(ctx, nrhs >= 0, "apply: nrhs < 0");
    REQUIRE(ctx, nrhs == 0 || (x && y), "apply: null operand");
    if (nrhs == 0) return INTI_OK;
    LOCK(ctx);
    const int cw = op_is_complex(op) ? 2 : 1;
    const int64_t m = op->trg->n, n = op->src->n;
    void *dx = nullptr, *dy = nullptr;
    int st = ctx_scratch(ctx, kScrX, sizeof(double) * cw * n * nrhs, &dx);
    if (st) return st;
    st = ctx_scratch(ctx, kScrY, sizeof(double) * cw * m * nrhs, &dy);
    if (st) return st;
    INTI_HIP(ctx, hipMemcpyAsync(dx, x, sizeof(double) * cw * n * nrhs, hipMemcpyHostToDevice, ctx->stream));
    const bool beta_nz = beta && (beta[0] != 0.0 || beta[1] != 0.0);
    if (beta_nz)
        INTI_HIP(ctx, hipMemcpyAsync(dy, y, sizeof(double) * cw * m * nrhs, hipMemcpyHostToDevice, ctx->stream));
    st = apply_device_locked(op, nrhs, (const double *)dx, n, (double *)dy, m, alpha, beta);
    if (st) return st;
    INTI_HIP(ctx, hipMemcpyAsync(y, dy, sizeof(double) * cw * m * nrhs, hipMemcpyDeviceToHost, ctx->stream));
    INTI_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return INTI_OK;
}

int inti_op_assemble_dense(inti_op *op, double *out) {
    if (!op) return INTI_ERR_ARG;
    Ctx *ctx = op->ctx;
    REQUIRE(ctx, out != nullptr, "assemble: out is null");
    LOCK(ctx);
    const int cw = op_is_complex(op) ? 2 : 1;
    const size_t bytes = sizeof(double) * cw * (size_t)op->trg->n * op->src->n;
    if (bytes == 0) return INTI_OK;
    void *d = nullptr;
    if (hipMalloc(&d, bytes) != hipSuccess) return set_error(ctx, INTI_ERR_NOMEM, "assemble: allocation failed");
    int st = launch_assemble(op, (double *)d);
    if (st == INTI_OK) {
        if (hipMemcpyAsync(out, d, bytes, hipMemcpyDeviceToHost, ctx->stream) != hipSuccess ||
            hipStreamSynchronize(ctx->stream) != hipSuccess)
            st = set_error(ctx, INTI_ERR_HIP, "assemble: copy back failed");
    }
    (void)hipFree(d);
    return st;
}

int inti_op_assemble_dense_device(inti_op *op, double *out, int64_t ldout) {
    if (!op) return INTI_ERR_ARG;
    Ctx *ctx = op->ctx;
    REQUIRE(ctx, out != nullptr, "assemble_device: out is null");
    REQUIRE(ctx, ldout == op->trg->n, "assemble_device: the leading dimension must equal the number of targets");
    LOCK(ctx);
    return launch_assemble(op, out);
}

// A[i + lda j] += coef * csr(i, j): the axpy!(true, dS, Smat) of src/api.jl:171-173
__global__ void k_dense_add_csr(int64_t m, const int32_t *rowptr, const int32_t *colind, const double *val,
                                int cplx, double cr, double ci, double *A, int64_t lda) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= m) return;
    for (int32_t q = rowptr[i]; q < rowptr[i + 1]; ++q) {
        const int64_t o = i + lda * (int64_t)colind[q];
        if (cplx) {
            const double vr = val[2 * q], vi = val[2 * q + 1];
            A[2 * o] += cr * vr - ci * vi;
            A[2 * o + 1] += cr * vi + ci * vr;
        } else {
            A[o] += cr * val[q];
        }
    }
}

int inti_dense_add_csr(inti_ctx *ctx, const inti_csr *csr, double coef_re, double coef_im, double *A,
                       int64_t lda) {
    if (!ctx) return INTI_ERR_ARG;
    REQUIRE(ctx, csr && A, "dense_add_csr: null argument");
    REQUIRE(ctx, lda >= csr->m, "dense_add_csr: leading dimension below the row count");
    LOCK(ctx);
    if (csr->m > 0)
        hipLaunchKernelGGL(k_dense_add_csr, dim3((unsigned)((csr->m + 255) / 256)), dim3(256), 0, ctx->stream, csr->m,
                           csr->rowptr, csr->colind, csr->val, csr->is_complex, coef_re, coef_im, A, lda);
    INTI_HIP(ctx, hipGetLastError());
    return INTI_OK;
}

int inti_dense_gemm(inti_ctx *ctx, int is_complex, int64_t m, int64_t n, int nrhs, const double *A, int64_t lda,
                    const double *X, int64_t ldx, double *Y, int64_t ldy, const double *alpha, const double *beta) {
    if (!ctx) return INTI_ERR_ARG;
    REQUIRE(ctx, A && X && Y && alpha && beta, "dense_gemm: null argument");
    REQUIRE(ctx, m >= 0 && n >= 0 && nrhs >= 0, "dense_gemm: negative size");
    REQUIRE(ctx, lda >= m && ldx >= n && ldy >= m, "dense_gemm: leading dimension too small");
    LOCK(ctx);
    return dense_gemm(ctx, is_complex ? 1 : 0, m, n, nrhs, A, lda, X, ldx, Y, ldy, alpha, beta);
}

int inti_op_adjoint(inti_op *op, const double *ubar, const double *sigma, double *sigma_bar,
                    double *src_xyz_bar, double *src_normal_bar, double *src_weight_bar,
                    double *trg_xyz_bar, const double *dcoefs, double *k_bar) {
    if (!op) return INTI_ERR_ARG;
    Ctx *ctx = op->ctx;
    REQUIRE(ctx, ubar != nullptr && sigma != nullptr, "adjoint: ubar and sigma are required");
    if (op->kimag != 0.0)
        return set_error(ctx, INTI_ERR_UNSUPPORTED, "adjoint: complex wavenumbers have no pullback");
    LOCK(ctx);
    return op_adjoint(op, ubar, sigma, sigma_bar, src_xyz_bar, src_normal_bar, src_weight_bar, trg_xyz_bar,
                      dcoefs, k_bar);
}

// *flag = 1 where two index arrays differ
__global__ __launch_bounds__(256) void k_differ(int64_t n, const int32_t *a, const int32_t *b, int *flag) {
    const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (q < n && a[q] != b[q]) *flag = 1;
}

// merged correction: c_new = c_old + coef * csr (same pattern), or a copy
__global__ void k_axpy_vals(int64_t nnz, int cplx, const double *src, double cr, double ci,
                            double *dst, int accumulate) {
    const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (q >= nnz) return;
    if (cplx) {
        const double vr = src[2 * q], vi = src[2 * q + 1];
        double yr = cr * vr - ci * vi, yi = cr * vi + ci * vr;
        if (accumulate) { yr += dst[2 * q]; yi += dst[2 * q + 1]; }
        dst[2 * q] = yr; dst[2 * q + 1] = yi;
    } else {
        double yr = cr * src[q];
        if (accumulate) yr += dst[q];
        dst[q] = yr;
    }
}

int inti_op_attach_correction(inti_op *op, const inti_csr *csr, double coef_re, double coef_im) {
    if (!op) return INTI_ERR_ARG;
    Ctx *ctx = op->ctx;
    REQUIRE(ctx, csr != nullptr, "attach: csr is null");
    if (csr->m != op->trg->n || csr->n != op->src->n)
        return set_error(ctx, INTI_ERR_SIZE, "attach: correction shape differs from the operator's");
    if (csr->is_complex != (op_is_complex(op) ? 1 : 0))
        return set_error(ctx, INTI_ERR_ARG, "attach: correction value type differs from the operator's");
    if (!csr->is_complex && coef_im != 0.0)
        return set_error(ctx, INTI_ERR_UNSUPPORTED, "attach: real correction takes a real coefficient");
    LOCK(ctx);
    const int cplx = csr->is_complex;
    int accumulate = 0;
    bool own = false;
    if (op->corr) {
        // same pattern required for an in-place merge
        bool same = op->corr->nnz == csr->nnz;
        if (same && csr->nnz > 0) {
            *ctx->flag = 0;
            hipLaunchKernelGGL(k_differ, dim3((unsigned)((csr->m + 256) / 256)), dim3(256), 0, ctx->stream, csr->m + 1,
                               op->corr->rowptr, csr->rowptr, ctx->flag);
            hipLaunchKernelGGL(k_differ, dim3((unsigned)((csr->nnz + 255) / 256)), dim3(256), 0, ctx->stream, csr->nnz,
                               op->corr->colind, csr->colind, ctx->flag);
            INTI_HIP(ctx, hipGetLastError());
            INTI_HIP(ctx, hipStreamSynchronize(ctx->stream));
            same = *ctx->flag == 0;
        }
        if (!same)
            return set_error(ctx, INTI_ERR_UNSUPPORTED, "attach: corrections with different patterns cannot be merged");
        accumulate = 1;
    } else {
        Csr *c = nullptr;
        int st = csr_alloc(ctx, csr->m, csr->n, csr->nnz, cplx, &c);
        if (st) return st;
        op->corr = c;
        INTI_HIP(ctx, hipMemcpyAsync(c->rowptr, csr->rowptr, sizeof(int32_t) * (csr->m + 1), hipMemcpyDeviceToDevice, ctx->stream));
        if (csr->nnz > 0)
            INTI_HIP(ctx, hipMemcpyAsync(c->colind, csr->colind, sizeof(int32_t) * csr->nnz, hipMemcpyDeviceToDevice, ctx->stream));
        own = csr->m == csr->n && csr->nnz <= kOwnRow * csr->m;
        st = transpose_pattern(op, own);
        if (st) {
            (void)hipStreamSynchronize(ctx->stream);
            op_free_correction(op);
            return st;
        }
    }
    if (csr->nnz > 0) {
        hipLaunchKernelGGL(k_axpy_vals, dim3((unsigned)((csr->nnz + 255) / 256)), dim3(256), 0, ctx->stream,
                           csr->nnz, cplx, csr->val, coef_re, coef_im, op->corr->val, accumulate);
        INTI_HIP(ctx, hipGetLastError());
    }
    INTI_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (own && *ctx->flag) {
        if (int st = transpose_pattern(op, false)) {
            (void)hipStreamSynchronize(ctx->stream);
            op_free_correction(op);
            return st;
        }
    }
    return INTI_OK;
}

int inti_op_detach_correction(inti_op *op) {
    if (!op) return INTI_ERR_ARG;
    LOCK(op->ctx);
    (void)hipStreamSynchronize(op->ctx->stream);
    op_free_correction(op);
    return INTI_OK;
}

// ---------------------------------------------------------- DIM correction
int inti_bdim_build(inti_op *opS, inti_op *opD, int derivative, int nq, int64_t ne,
                    const int64_t *qtags, const int64_t *near_ptr, const int64_t *near_idx,
                    const double *mu, const double *params, inti_csr **dS, inti_csr **dD,
                    double *diag) {
    if (!opS) return INTI_ERR_ARG;
    Ctx *ctx = opS->ctx;
    REQUIRE(ctx, opD && qtags && mu && dS && dD, "bdim: null argument");
    REQUIRE(ctx, opD->ctx == ctx, "bdim: operators on different contexts");
    REQUIRE(ctx, opS->trg == opD->trg && opS->src == opD->src, "bdim: S and D must share target and source");
    REQUIRE(ctx, opS->pde == opD->pde && opS->dim == opD->dim && opS->k == opD->k && opS->kimag == opD->kimag,
            "bdim: S and D must be the same PDE");
    const int kS = derivative ? INTI_ADL : INTI_SL, kD = derivative ? INTI_HS : INTI_DL;
    REQUIRE(ctx, opS->kind == kS && opD->kind == kD,
            "bdim: expects (SL, DL) operators, or (ADL, HS) with derivative = 1");
    REQUIRE(ctx, nq > 0 && ne > 0, "bdim: empty element set");
    REQUIRE(ctx, (near_ptr == nullptr) == (near_idx == nullptr), "bdim: near_ptr and near_idx go together");
    REQUIRE(ctx, params == nullptr || (params[0] > 0 && params[1] > 0), "bdim: bad parameters");
    LOCK(ctx);
    Csr *s = nullptr, *d = nullptr;
    int st = bdim_build(opS, opD, derivative, nq, ne, qtags, near_ptr, near_idx, mu, params, &s, &d, diag);
    if (st) return st;
    *dS = static_cast<inti_csr *>(s);
    *dD = static_cast<inti_csr *>(d);
    return INTI_OK;
}

int inti_bdim_build_types(inti_op *opS, inti_op *opD, int derivative, int ntypes, const int *nq,
                          const int64_t *ne, const int64_t *qtags, const int64_t *near_ptr,
                          const int64_t *near_idx, const double *mu, const double *params, inti_csr **dS,
                          inti_csr **dD, double *diag) {
    if (!opS) return INTI_ERR_ARG;
    Ctx *ctx = opS->ctx;
    REQUIRE(ctx, opD && nq && ne && qtags && mu && dS && dD, "bdim: null argument");
    REQUIRE(ctx, opD->ctx == ctx, "bdim: operators on different contexts");
    REQUIRE(ctx, opS->trg == opD->trg && opS->src == opD->src, "bdim: S and D must share target and source");
    REQUIRE(ctx, opS->pde == opD->pde && opS->dim == opD->dim && opS->k == opD->k && opS->kimag == opD->kimag,
            "bdim: S and D must be the same PDE");
    const int kS = derivative ? INTI_ADL : INTI_SL, kD = derivative ? INTI_HS : INTI_DL;
    REQUIRE(ctx, opS->kind == kS && opD->kind == kD,
            "bdim: expects (SL, DL) operators, or (ADL, HS) with derivative = 1");
    REQUIRE(ctx, ntypes > 0, "bdim: no element type");
    int64_t total = 0;
    for (int t = 0; t < ntypes; ++t) {
        REQUIRE(ctx, nq[t] > 0 && ne[t] >= 0, "bdim: bad element type sizes");
        total += ne[t];
    }
    REQUIRE(ctx, total > 0, "bdim: empty element set");
    REQUIRE(ctx, (near_ptr == nullptr) == (near_idx == nullptr), "bdim: near_ptr and near_idx go together");
    REQUIRE(ctx, params == nullptr || (params[0] > 0 && params[1] > 0), "bdim: bad parameters");
    LOCK(ctx);
    Csr *s = nullptr, *d = nullptr;
    int st = bdim_build_types(opS, opD, derivative, ntypes, nq, ne, qtags, near_ptr, near_idx, mu, params, &s,
                              &d, diag);
    if (st) return st;
    *dS = static_cast<inti_csr *>(s);
    *dD = static_cast<inti_csr *>(d);
    return INTI_OK;
}

int inti_lsq_build(inti_ctx *ctx, int is_complex, int nrows, int ncols, int64_t ne, const double *A,
                   const int64_t *cols, int64_t m, int64_t n, const int64_t *near_ptr,
                   const int64_t *near_idx, const double *rhs, inti_csr **out, double *diag) {
    if (!ctx) return INTI_ERR_ARG;
    REQUIRE(ctx, A && cols && rhs && out, "lsq: null argument");
    REQUIRE(ctx, ne > 0 && m > 0 && n > 0, "lsq: empty problem");
    REQUIRE(ctx, (near_ptr == nullptr) == (near_idx == nullptr), "lsq: near_ptr and near_idx go together");
    LOCK(ctx);
    Csr *c = nullptr;
    int st = lsq_build(ctx, is_complex ? 1 : 0, nrows, ncols, ne, A, cols, m, n, near_ptr, near_idx, rhs, &c, diag);
    if (st) return st;
    *out = static_cast<inti_csr *>(c);
    return INTI_OK;
}

int inti_lsq_build_types(inti_ctx *ctx, int is_complex, int nrows, int ntypes, const int *ncols, const int64_t *ne,
                         const double *A, const int64_t *cols, int64_t m, int64_t n, const int64_t *near_ptr,
                         const int64_t *near_idx, const double *rhs, inti_csr **out, double *diag) {
    if (!ctx) return INTI_ERR_ARG;
    REQUIRE(ctx, ncols && ne && A && cols && rhs && out, "lsq: null argument");
    REQUIRE(ctx, ntypes > 0 && m > 0 && n > 0, "lsq: empty problem");
    int64_t total = 0;
    for (int t = 0; t < ntypes; ++t) {
        REQUIRE(ctx, ne[t] >= 0, "lsq: negative element count");
        total += ne[t];
    }
    REQUIRE(ctx, total > 0, "lsq: empty problem");
    REQUIRE(ctx, (near_ptr == nullptr) == (near_idx == nullptr), "lsq: near_ptr and near_idx go together");
    LOCK(ctx);
    Csr *c = nullptr;
    int st = lsq_build_types(ctx, is_complex ? 1 : 0, nrows, ntypes, ncols, ne, A, cols, m, n, near_ptr, near_idx,
                             rhs, &c, diag);
    if (st) return st;
    *out = static_cast<inti_csr *>(c);
    return INTI_OK;
}

// ----------------------------------------------------------------- solvers
// host pointers: stage b and x on the device for the solve, in the context's
// staging buffers (the solvers themselves use none of them)
struct Staged {
    void *b = nullptr, *x = nullptr;
};

static int stage_in(Ctx *ctx, Staged &S, size_t bytes, const double *b, const double *x) {
    if (int st = ctx_scratch(ctx, kScrX, bytes, &S.b)) return st;
    if (int st = ctx_scratch(ctx, kScrY, bytes, &S.x)) return st;
    INTI_HIP(ctx, hipMemcpyAsync(S.b, b, bytes, hipMemcpyHostToDevice, ctx->stream));
    INTI_HIP(ctx, hipMemcpyAsync(S.x, x, bytes, hipMemcpyHostToDevice, ctx->stream));
    return INTI_OK;
}

int inti_gmres_prec(inti_op *op, inti_op *prec, int on_device, const double *b, double *x, int restart,
                    int maxiter, double rtol, double atol, int use_graph, int *iters, double *relres) {
    if (!op) return INTI_ERR_ARG;
    Ctx *ctx = op->ctx;
    REQUIRE(ctx, b && x, "gmres: null vector");
    REQUIRE(ctx, rtol >= 0 && atol >= 0, "gmres: negative tolerance");
    LOCK(ctx);
    if (on_device) return gmres_solve(op, prec, b, x, restart, maxiter, rtol, atol, use_graph, iters, relres);
    const size_t bytes = sizeof(double) * (op_is_complex(op) ? 2 : 1) * op->src->n;
    Staged S;
    int st = stage_in(ctx, S, bytes, b, x);
    if (st) return st;
    st = gmres_solve(op, prec, (const double *)S.b, (double *)S.x, restart, maxiter, rtol, atol, use_graph, iters,
                     relres);
    if (st) return st;
    INTI_HIP(ctx, hipMemcpyAsync(x, S.x, bytes, hipMemcpyDeviceToHost, ctx->stream));
    INTI_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return INTI_OK;
}

int inti_gmres(inti_op *op, int on_device, const double *b, double *x, int restart, int maxiter,
               double rtol, double atol, int use_graph, int *iters, double *relres) {
    return inti_gmres_prec(op, nullptr, on_device, b, x, restart, maxiter, rtol, atol, use_graph, iters, relres);
}

int inti_refine_solve_prec(inti_op *op_hi, inti_op *op_lo, inti_op *prec, int on_device, const double *b,
                           double *x, int restart, int maxiter_inner, double inner_rtol, int max_outer,
                           double rtol, int use_graph, int *outer, int *inner_total, double *relres) {
    if (!op_hi || !op_lo) return INTI_ERR_ARG;
    Ctx *ctx = op_hi->ctx;
    REQUIRE(ctx, op_lo->ctx == ctx, "refine: operators on different contexts");
    REQUIRE(ctx, b && x, "refine: null vector");
    REQUIRE(ctx, restart >= 1 && maxiter_inner >= 1 && max_outer >= 0, "refine: bad iteration limits");
    LOCK(ctx);
    if (on_device)
        return refine_solve(op_hi, op_lo, prec, b, x, restart, maxiter_inner, inner_rtol, max_outer, rtol, use_graph,
                            outer, inner_total, relres);
    const size_t bytes = sizeof(double) * (op_is_complex(op_hi) ? 2 : 1) * op_hi->src->n;
    Staged S;
    int st = stage_in(ctx, S, bytes, b, x);
    if (st) return st;
    st = refine_solve(op_hi, op_lo, prec, (const double *)S.b, (double *)S.x, restart, maxiter_inner, inner_rtol,
                      max_outer, rtol, use_graph, outer, inner_total, relres);
    if (st) return st;
    INTI_HIP(ctx, hipMemcpyAsync(x, S.x, bytes, hipMemcpyDeviceToHost, ctx->stream));
    INTI_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return INTI_OK;
}

int inti_refine_solve(inti_op *op_hi, inti_op *op_lo, int on_device, const double *b, double *x,
                      int restart, int maxiter_inner, double inner_rtol, int max_outer, double rtol,
                      int use_graph, int *outer, int *inner_total, double *relres) {
    return inti_refine_solve_prec(op_hi, op_lo, nullptr, on_device, b, x, restart, maxiter_inner, inner_rtol,
                                  max_outer, rtol, use_graph, outer, inner_total, relres);
}

// --------------------------------------------------------------------- CSR
int inti_csr_info(const inti_csr *csr, int64_t *m, int64_t *n, int64_t *nnz, int *is_complex) {
    if (!csr) return INTI_ERR_ARG;
    if (m) *m = csr->m;
    if (n) *n = csr->n;
    if (nnz) *nnz = csr->nnz;
    if (is_complex) *is_complex = csr->is_complex;
    return INTI_OK;
}

int inti_csr_export(const inti_csr *csr, int64_t *rowptr, int64_t *colind, double *val) {
    if (!csr) return INTI_ERR_ARG;
    Ctx *ctx = csr->ctx;
    LOCK(ctx);
    std::vector<int32_t> rp(csr->m + 1), ci(csr->nnz);
    INTI_HIP(ctx, hipStreamSynchronize(ctx->stream));
    INTI_HIP(ctx, hipMemcpy(rp.data(), csr->rowptr, sizeof(int32_t) * (csr->m + 1), hipMemcpyDeviceToHost));
    if (csr->nnz > 0) {
        INTI_HIP(ctx, hipMemcpy(ci.data(), csr->colind, sizeof(int32_t) * csr->nnz, hipMemcpyDeviceToHost));
        if (val)
            INTI_HIP(ctx, hipMemcpy(val, csr->val, sizeof(double) * (csr->is_complex ? 2 : 1) * csr->nnz,
                                    hipMemcpyDeviceToHost));
    }
    if (rowptr) for (int64_t i = 0; i <= csr->m; ++i) rowptr[i] = rp[i];
    if (colind) for (int64_t p = 0; p < csr->nnz; ++p) colind[p] = ci[p];
    return INTI_OK;
}

int inti_csr_destroy(inti_csr *csr) {
    if (!csr) return INTI_ERR_ARG;
    Ctx *ctx = csr->ctx;
    {
        LOCK(ctx);
        (void)hipStreamSynchronize(ctx->stream);
    }
    csr_free(csr);
    return INTI_OK;
}

}  // extern "C"

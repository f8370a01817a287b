// Restarted GMRES on a (corrected) operator, device resident, and mixed
// precision iterative refinement around it.
//
// The user-side solve of Inti.jl's examples is IterativeSolvers.gmres on
// L = I/2 + D - i k S (docs/src/examples/helmholtz_scattering.jl:230,494-495;
// docs/src/examples/poisson.jl:167-168). Here one Arnoldi step is a fixed
// sequence of kernels that read the current column index k from a device
// state block: apply the operator to V[:,k], two passes of classical
// Gram-Schmidt, normalisation, and the Givens update of the Hessenberg column
// and of the residual estimate. The same sequence therefore serves every step
// and is captured once in a hipGraph and replayed; the host only looks at the
// residual estimates every few steps. No memset is recorded in the graph:
// clearing is done by kernels.
//
// For small systems a step is bound by its number of dependent kernels, so
// the vector work is four of them (k_gdots, k_gorth twice, k_gnext): each
// k_gorth block adds up the dot products itself (all blocks redundantly, in
// the same order), updates its rows and forms the next pass's partial dots or
// norm while the rows are in LDS. (Ten kernels before, each with its own
// sweep: GMRES on 4,320 complex nodes 2.58 -> 1.97 ms.)
// The redundant sums grow with the columns as the sweeps over the basis do, and
// stay below them also at 16,384 nodes, the most blocks per row (256 blocks of 64
// rows): 500 / 2,000 / 5,000 steps of one basis take 0.26 / 1.36 / 6.8 s, with
// the ten kernels 0.39 / 2.93 / 16.5 s.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <complex>
#include <vector>

#include "common.hpp"

namespace inti {

struct GState {
    int k;      // Arnoldi column of the current step (set by k_gdots)
    int knext;  // column of the next step (set by k_gnext)
};

template <bool CPLX>
struct Sc;
template <>
struct Sc<true> {
    using T = double2;
    __device__ static T zero() { return make_double2(0.0, 0.0); }
    __device__ static T conjmul(T a, T b) { return make_double2(a.x * b.x + a.y * b.y, a.x * b.y - a.y * b.x); }
    __device__ static T mul(T a, T b) { return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
    __device__ static T add(T a, T b) { return make_double2(a.x + b.x, a.y + b.y); }
    __device__ static T sub(T a, T b) { return make_double2(a.x - b.x, a.y - b.y); }
    __device__ static T scale(T a, double s) { return make_double2(a.x * s, a.y * s); }
    __device__ static double abs2(T a) { return a.x * a.x + a.y * a.y; }
    __device__ static T shfl(T v, int off) { return make_double2(__shfl_xor(v.x, off), __shfl_xor(v.y, off)); }
};
template <>
struct Sc<false> {
    using T = double;
    __device__ static T zero() { return 0.0; }
    __device__ static T conjmul(T a, T b) { return a * b; }
    __device__ static T mul(T a, T b) { return a * b; }
    __device__ static T add(T a, T b) { return a + b; }
    __device__ static T sub(T a, T b) { return a - b; }
    __device__ static T scale(T a, double s) { return a * s; }
    __device__ static double abs2(T a) { return a * a; }
    __device__ static T shfl(T v, int off) { return __shfl_xor(v, off); }
};

constexpr int kGB = 256;     // threads per block of the vector kernels
constexpr int kGRows = 4096; // rows per block of the norm kernel
constexpr int kGWaves = kGB / 64;
constexpr int kOrthRows = 1024;  // most rows of one Gram-Schmidt block
constexpr int kOrthCols = 256;   // Hessenberg entries held in LDS at a time

template <bool CPLX>
__device__ typename Sc<CPLX>::T block_sum(typename Sc<CPLX>::T v) {
    using S = Sc<CPLX>;
    __shared__ typename S::T red[kGB / 64];
    for (int off = 32; off > 0; off >>= 1) v = S::add(v, S::shfl(v, off));
    const int w = threadIdx.x / 64, l = threadIdx.x % 64;
    if (l == 0) red[w] = v;
    __syncthreads();
    typename S::T s = S::zero();
    if (threadIdx.x == 0)
        for (int q = 0; q < kGB / 64; ++q) s = S::add(s, red[q]);
    return s;  // valid in thread 0
}

// sum over the 64 lanes of a wave, valid in lane 63, in a fixed order: rows of
// 16 by shifts, then the rows one after another (cross-lane moves of the
// VALU, no LDS crossbar)
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, true);
    return v + __hiloint2double(hi, lo);
}
__device__ __forceinline__ double wave_sum(double v) {
    v = dpp_add<0x111, 0xf>(v);  // row_shr:1
    v = dpp_add<0x112, 0xf>(v);  // row_shr:2
    v = dpp_add<0x114, 0xf>(v);  // row_shr:4
    v = dpp_add<0x118, 0xf>(v);  // row_shr:8
    v = dpp_add<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
    v = dpp_add<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
    return v;
}
__device__ __forceinline__ double2 wave_sum(double2 v) { return make_double2(wave_sum(v.x), wave_sum(v.y)); }

// Gram-Schmidt work of one block: rows [r0, r0 + rows) of V and w
template <bool CPLX>
struct GArgs {
    using T = typename Sc<CPLX>::T;
    const T *V;
    int64_t ldv, n;
    int rows, nb, ldp;  // rows per block, blocks, leading dimension of the partials
    GState *st;
    T *w;
    T *pa, *pb;      // partial dots of the first and second pass: [block][column]
    double *npart;   // partial |w|^2 per block
    T *H;
    int ldh;
};

// partial[j] = sum over the block's rows of conj(V[i, j]) w_i, j <= k: a wave
// takes every fourth column, four of them at a time
template <bool CPLX>
__device__ __forceinline__ void orth_dots(const GArgs<CPLX> &a, int64_t r0, int cnt, int k,
                                          const typename Sc<CPLX>::T *s_w, typename Sc<CPLX>::T *partial) {
    using S = Sc<CPLX>;
    constexpr int C = 4;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int j0 = wave; j0 <= k; j0 += C * kGWaves) {
        typename S::T acc[C];
#pragma unroll
        for (int c = 0; c < C; ++c) acc[c] = S::zero();
        for (int i = lane; i < cnt; i += 64) {
            const typename S::T wi = s_w[i];
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const int j = j0 + c * kGWaves <= k ? j0 + c * kGWaves : k;
                acc[c] = S::add(acc[c], S::conjmul(a.V[r0 + i + a.ldv * j], wi));
            }
        }
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const typename S::T v = wave_sum(acc[c]);
            if (lane == 63 && j0 + c * kGWaves <= k) partial[j0 + c * kGWaves] = v;
        }
    }
}

// pa[b][j] = the block's share of V[:, j]^H w, j <= k; sets the step's column
template <bool CPLX>
__global__ __launch_bounds__(kGB) void k_gdots(GArgs<CPLX> a) {
    __shared__ typename Sc<CPLX>::T s_w[kOrthRows];
    const int64_t r0 = (int64_t)blockIdx.x * a.rows;
    const int cnt = (int)(a.n - r0 < a.rows ? a.n - r0 : a.rows);
    for (int i = threadIdx.x; i < cnt; i += kGB) s_w[i] = a.w[r0 + i];
    __syncthreads();
    const int k = a.st->knext;
    if (blockIdx.x == 0 && threadIdx.x == 0) a.st->k = k;
    orth_dots<CPLX>(a, r0, cnt, k, s_w, a.pa + (int64_t)blockIdx.x * a.ldp);
}

// h = the sums of the pass's partial dots, w -= V[:, 0..k] h for the block's
// rows; then the second pass's partial dots (LAST = false) or the partial
// norm. Block 0 keeps the Hessenberg column.
template <bool CPLX, bool LAST>
__global__ __launch_bounds__(kGB) void k_gorth(GArgs<CPLX> a) {
    using S = Sc<CPLX>;
    using T = typename S::T;
    __shared__ T s_w[kOrthRows];
    __shared__ T s_h[kOrthCols];
    __shared__ T s_g[kGWaves][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t r0 = (int64_t)blockIdx.x * a.rows;
    const int cnt = (int)(a.n - r0 < a.rows ? a.n - r0 : a.rows);
    const int k = a.st->k;
    const T *partial = LAST ? a.pb : a.pa;
    for (int i = tid; i < cnt; i += kGB) s_w[i] = a.w[r0 + i];
    for (int c0 = 0; c0 <= k; c0 += kOrthCols) {
        const int nc = k + 1 - c0 < kOrthCols ? k + 1 - c0 : kOrthCols;
        // h: a wave adds every fourth block's partials of 64 columns, the four
        // sums are added in wave order
        for (int q = 0; q < nc; q += 64) {
            T s = S::zero();
            if (q + lane < nc) {
                const T *p = partial + c0 + q + lane;
#pragma unroll 8
                for (int b = wave; b < a.nb; b += kGWaves) s = S::add(s, p[(int64_t)b * a.ldp]);
            }
            s_g[wave][lane] = s;
            __syncthreads();
            if (wave == 0 && q + lane < nc) {
#pragma unroll
                for (int g = 1; g < kGWaves; ++g) s = S::add(s, s_g[g][lane]);
                s_h[q + lane] = s;
                if (blockIdx.x == 0) {
                    T *h = a.H + c0 + q + lane + (int64_t)a.ldh * k;
                    *h = LAST ? S::add(*h, s) : s;
                }
            }
            __syncthreads();
        }
        // 64 rows at a time, a wave takes every fourth column
        for (int i0 = 0; i0 < cnt; i0 += 64) {
            T s = S::zero();
            if (i0 + lane < cnt) {
                const T *v = a.V + r0 + i0 + lane + a.ldv * c0;
#pragma unroll 4
                for (int j = wave; j < nc; j += kGWaves) s = S::add(s, S::mul(v[a.ldv * j], s_h[j]));
            }
            s_g[wave][lane] = s;
            __syncthreads();
            if (wave == 0 && i0 + lane < cnt) {
#pragma unroll
                for (int g = 1; g < kGWaves; ++g) s = S::add(s, s_g[g][lane]);
                s_w[i0 + lane] = S::sub(s_w[i0 + lane], s);
            }
            __syncthreads();
        }
    }
    for (int i = tid; i < cnt; i += kGB) a.w[r0 + i] = s_w[i];
    if constexpr (LAST) {
        double q = 0.0;
        for (int i = tid; i < cnt; i += kGB) q += S::abs2(s_w[i]);
        q = block_sum<false>(q);
        if (tid == 0) a.npart[blockIdx.x] = q;
    } else {
        orth_dots<CPLX>(a, r0, cnt, k, s_w, a.pb + (int64_t)blockIdx.x * a.ldp);
    }
}

// partial[b] = sum over block b of |w|^2
template <bool CPLX>
__global__ __launch_bounds__(kGB) void k_gnorm(const typename Sc<CPLX>::T *w, int64_t n,
                                               double *partial) {
    using S = Sc<CPLX>;
    const int64_t r0 = (int64_t)blockIdx.x * kGRows;
    const int64_t r1 = r0 + kGRows < n ? r0 + kGRows : n;
    double acc = 0.0;
    for (int64_t i = r0 + threadIdx.x; i < r1; i += kGB) acc += S::abs2(w[i]);
    acc = block_sum<false>(acc);
    if (threadIdx.x == 0) partial[blockIdx.x] = acc;
}

// Givens rotation of (a, b), b real and >= 0: c, s with
// [c s; -conj(s) c] [a; b] = [r; 0]
__device__ __forceinline__ void givens(double2 a, double b, double &c, double2 &s, double2 &r) {
    const double an = hypot(a.x, a.y);
    if (an == 0.0) {
        c = 0.0;
        s = make_double2(1.0, 0.0);
        r = make_double2(b, 0.0);
    } else {
        const double t = hypot(an, b);
        c = an / t;
        s = make_double2(a.x / an * b / t, a.y / an * b / t);
        r = make_double2(a.x / an * t, a.y / an * t);
    }
}
__device__ __forceinline__ void givens(double a, double b, double &c, double &s, double &r) {
    c = 1.0;
    s = 0.0;
    r = a;
    if (b != 0.0) {
        const double t = hypot(a, b);
        c = a / t;
        s = b / t;
        r = t;
    }
}
// [a; b] <- [c a + s b; -conj(s) a + c b]
__device__ __forceinline__ void rotate(double c, double2 s, double2 &a, double2 &b) {
    const double2 a0 = a, b0 = b;
    a = make_double2(c * a0.x + s.x * b0.x - s.y * b0.y, c * a0.y + s.x * b0.y + s.y * b0.x);
    b = make_double2(-(s.x * a0.x + s.y * a0.y) + c * b0.x, -(s.x * a0.y - s.y * a0.x) + c * b0.y);
}
__device__ __forceinline__ void rotate(double c, double s, double &a, double &b) {
    const double a0 = a, b0 = b;
    a = c * a0 + s * b0;
    b = -s * a0 + c * b0;
}
__device__ __forceinline__ double g_abs(double2 v) { return hypot(v.x, v.y); }
__device__ __forceinline__ double g_abs(double v) { return fabs(v); }

template <bool CPLX>
struct GNextArgs {
    using T = typename Sc<CPLX>::T;
    T *V, *vk;
    int64_t ldv, n;
    GState *st;
    const T *w;
    const double *npart;
    int nb;
    T *H;
    int ldh;
    double *cs;
    T *sn, *g;
    double *res;
};

// The norm of w (added by every block in the same order); V[:, k+1] = vk =
// w / ||w||. The last block takes no rows: it applies the earlier rotations
// to Hessenberg column k (staged in LDS, kOrthCols entries at a time), makes
// the new one, the residual estimate, and moves to column k + 1.
template <bool CPLX>
__global__ __launch_bounds__(kGB) void k_gnext(GNextArgs<CPLX> a) {
    using S = Sc<CPLX>;
    using T = typename S::T;
    __shared__ double s_nrm;
    __shared__ T s_h[kOrthCols + 1], s_sn[kOrthCols];
    __shared__ double s_cs[kOrthCols];
    const int tid = threadIdx.x;
    double q = 0.0;
    for (int b = tid; b < a.nb; b += kGB) q += a.npart[b];
    q = block_sum<false>(q);
    if (tid == 0) s_nrm = sqrt(q);
    __syncthreads();
    const double nrm = s_nrm;
    const int k = a.st->k;
    if (blockIdx.x + 1 < gridDim.x) {
        const double inv = nrm > 0.0 ? 1.0 / nrm : 0.0;
        const int64_t i = (int64_t)blockIdx.x * kGB + tid;
        if (i < a.n) {
            const T v = S::scale(a.w[i], inv);
            a.V[i + a.ldv * (k + 1)] = v;
            a.vk[i] = v;
        }
        return;
    }
    T *h = a.H + (int64_t)a.ldh * k;
    // entries 0 .. k rotated by the earlier pairs (i, i + 1), i < k
    T carry = S::zero();  // entry c0, already rotated by the pair before it
    for (int c0 = 0; c0 < k; c0 += kOrthCols) {
        const int nc = k - c0 < kOrthCols ? k - c0 : kOrthCols;
        for (int i = tid; i <= nc; i += kGB) {
            s_h[i] = h[c0 + i];
            if (i < nc) {
                s_cs[i] = a.cs[c0 + i];
                s_sn[i] = a.sn[c0 + i];
            }
        }
        __syncthreads();
        if (tid == 0) {
            T x = c0 ? carry : s_h[0];
            for (int i = 0; i < nc; ++i) {
                T y = s_h[i + 1];
                rotate(s_cs[i], s_sn[i], x, y);
                s_h[i] = x;
                x = y;
            }
            carry = x;
        }
        __syncthreads();
        for (int i = tid; i < nc; i += kGB) h[c0 + i] = s_h[i];
        __syncthreads();
    }
    if (tid == 0) {
        const T x = k ? carry : h[0];
        double c;
        T s, r;
        givens(x, nrm, c, s, r);
        h[k] = r;
        h[k + 1] = S::zero();
        a.cs[k] = c;
        a.sn[k] = s;
        T g0 = a.g[k], g1 = S::zero();
        rotate(c, s, g0, g1);
        a.g[k] = g0;
        a.g[k + 1] = g1;
        a.res[k] = g_abs(g1);
        a.st->knext = k + 1;
    }
}

// x += V[:, 0..kk-1] y
template <bool CPLX>
__global__ __launch_bounds__(kGB) void k_gxupdate(const typename Sc<CPLX>::T *V, int64_t ldv, int kk,
                                                  const typename Sc<CPLX>::T *y,
                                                  typename Sc<CPLX>::T *x, int64_t n) {
    using S = Sc<CPLX>;
    const int64_t i = (int64_t)blockIdx.x * kGB + threadIdx.x;
    if (i >= n) return;
    typename S::T s = x[i];
    for (int j = 0; j < kk; ++j) s = S::add(s, S::mul(V[i + ldv * j], y[j]));
    x[i] = s;
}

// generic vector helpers: y = a x + b y (real scalars), fill
template <bool CPLX>
__global__ __launch_bounds__(kGB) void k_gaxpby(int64_t n, double a, const typename Sc<CPLX>::T *x,
                                                double b, typename Sc<CPLX>::T *y) {
    using S = Sc<CPLX>;
    const int64_t i = (int64_t)blockIdx.x * kGB + threadIdx.x;
    if (i >= n) return;
    // b == 0 does not read y (fresh workspace may hold any bit pattern)
    y[i] = b == 0.0 ? S::scale(x[i], a) : S::add(S::scale(x[i], a), S::scale(y[i], b));
}

template <typename T>
__global__ __launch_bounds__(kGB) void k_gfill(int64_t n, T *p, T v) {
    const int64_t i = (int64_t)blockIdx.x * kGB + threadIdx.x;
    if (i < n) p[i] = v;
}

// ----------------------------------------------------------------- host side
struct GmresWork {
    int m;
    int64_t n;
    int cplx;
    void *slab = nullptr;  // one allocation, cut into the buffers below
    void *V = nullptr, *w = nullptr, *vk = nullptr, *r = nullptr, *t = nullptr;  // t: P v (preconditioned)
    void *pa = nullptr, *pb = nullptr, *H = nullptr, *sn = nullptr, *g = nullptr, *y = nullptr;
    double *cs = nullptr, *res = nullptr, *npart = nullptr;
    GState *st = nullptr;
    int nb = 1;             // blocks of the norm kernel
    int orows = 64, onb = 1;  // rows per block and blocks of the Gram-Schmidt kernels
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    hipStream_t stream = nullptr;
    // Teardown order: drain the stream (an error return may leave launches
    // queued), destroy the executable graph and the graph whose kernel nodes
    // hold pointers into the buffers, and only then release the buffers.
    ~GmresWork() {
        if (stream) (void)hipStreamSynchronize(stream);
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
        if (slab) (void)hipFree(slab);
    }
};

// Rows of a Gram-Schmidt block: whole 64-row groups in at most 256 blocks (one
// per CU; every block adds up all blocks' partial dots), at most kOrthRows.
static int gwork_alloc(Ctx *ctx, GmresWork &W, int m, int64_t n, int cplx) {
    W.m = m; W.n = n; W.cplx = cplx;
    W.stream = ctx->stream;
    const size_t es = cplx ? 16 : 8;
    W.nb = (int)std::max<int64_t>(1, (n + kGRows - 1) / kGRows);
    const int64_t groups = std::max<int64_t>(1, (n + 63) / 64);
    W.orows = (int)std::min<int64_t>(kOrthRows, 64 * ((groups + 255) / 256));
    W.onb = (int)std::max<int64_t>(1, (n + W.orows - 1) / W.orows);
    const size_t part = es * (size_t)W.onb * (m + 1);
    struct { void **p; size_t bytes; } cut[] = {
        {&W.V, es * (size_t)n * (m + 1)}, {&W.w, es * n}, {&W.vk, es * n}, {&W.r, es * n}, {&W.t, es * n},
        {&W.pa, part}, {&W.pb, part}, {&W.H, es * (size_t)(m + 1) * m}, {&W.sn, es * m}, {&W.g, es * (m + 1)},
        {&W.y, es * (m + 1)}, {(void **)&W.cs, sizeof(double) * m}, {(void **)&W.res, sizeof(double) * m},
        {(void **)&W.npart, sizeof(double) * std::max(W.nb, W.onb)}, {(void **)&W.st, sizeof(GState)}};
    size_t total = 0;
    for (auto &c : cut) total += (c.bytes + 255) / 256 * 256;
    if (hipMalloc(&W.slab, total) != hipSuccess) {
        W.slab = nullptr;
        return set_error(ctx, INTI_ERR_NOMEM, "gmres: workspace allocation failed");
    }
    char *at = (char *)W.slab;
    for (auto &c : cut) {
        *c.p = at;
        at += (c.bytes + 255) / 256 * 256;
    }
    return INTI_OK;
}

// y = alpha A x + beta y (real alpha, beta) on the context's stream
static int apply_vec(Op *op, const void *x, void *y, int64_t n, double alpha, double beta) {
    DirectLaunch L;
    L.op = op; L.nrhs = 1; L.x = (const double *)x; L.ldx = n; L.y = (double *)y; L.ldy = n;
    L.alpha[0] = alpha; L.alpha[1] = 0.0; L.beta[0] = beta; L.beta[1] = 0.0;
    return launch_apply(L);
}

// one Arnoldi step on the stream (also what the graph records); with a
// right preconditioner P the step applies A P
template <bool CPLX>
static int arnoldi_step(Op *op, Op *prec, GmresWork &W, hipStream_t s) {
    using T = typename Sc<CPLX>::T;
    const int64_t n = W.n;
    int rc = prec ? apply_vec(prec, W.vk, W.t, n, 1.0, 0.0) : INTI_OK;
    if (rc) return rc;
    rc = apply_vec(op, prec ? W.t : W.vk, W.w, n, 1.0, 0.0);
    if (rc) return rc;
    GArgs<CPLX> a;
    a.V = (const T *)W.V; a.ldv = n; a.n = n;
    a.rows = W.orows; a.nb = W.onb; a.ldp = W.m + 1;
    a.st = W.st; a.w = (T *)W.w; a.pa = (T *)W.pa; a.pb = (T *)W.pb;
    a.npart = W.npart; a.H = (T *)W.H; a.ldh = W.m + 1;
    hipLaunchKernelGGL(k_gdots<CPLX>, dim3((unsigned)W.onb), dim3(kGB), 0, s, a);
    hipLaunchKernelGGL((k_gorth<CPLX, false>), dim3((unsigned)W.onb), dim3(kGB), 0, s, a);
    hipLaunchKernelGGL((k_gorth<CPLX, true>), dim3((unsigned)W.onb), dim3(kGB), 0, s, a);
    GNextArgs<CPLX> b;
    b.V = (T *)W.V; b.vk = (T *)W.vk; b.ldv = n; b.n = n;
    b.st = W.st; b.w = (const T *)W.w; b.npart = W.npart; b.nb = W.onb;
    b.H = (T *)W.H; b.ldh = W.m + 1; b.cs = W.cs; b.sn = (T *)W.sn; b.g = (T *)W.g; b.res = W.res;
    hipLaunchKernelGGL(k_gnext<CPLX>, dim3((unsigned)((n + kGB - 1) / kGB + 1)), dim3(kGB), 0, s, b);
    return hipGetLastError() == hipSuccess ? INTI_OK
                                           : set_error(op->ctx, INTI_ERR_HIP, "gmres: kernel launch failed");
}

// r = b - A x (device vectors), returns ||r||
template <bool CPLX>
static int residual(Op *op, GmresWork &W, const double *b, const double *x, double *r, double &nrm) {
    using T = typename Sc<CPLX>::T;
    Ctx *ctx = op->ctx;
    hipStream_t s = ctx->stream;
    const int64_t n = W.n;
    const dim3 gv((unsigned)((n + kGB - 1) / kGB));
    INTI_HIP(ctx, hipMemcpyAsync(r, b, (CPLX ? 16 : 8) * n, hipMemcpyDeviceToDevice, s));
    DirectLaunch L;
    L.op = op; L.nrhs = 1; L.x = x; L.ldx = n; L.y = r; L.ldy = n;
    L.alpha[0] = -1.0; L.alpha[1] = 0.0; L.beta[0] = 1.0; L.beta[1] = 0.0;
    int rc = launch_apply(L);
    if (rc) return rc;
    hipLaunchKernelGGL(k_gnorm<CPLX>, dim3((unsigned)W.nb), dim3(kGB), 0, s, (const T *)r, n, W.npart);
    std::vector<double> np(W.nb);
    INTI_HIP(ctx, hipMemcpyAsync(np.data(), W.npart, sizeof(double) * W.nb, hipMemcpyDeviceToHost, s));
    INTI_HIP(ctx, hipStreamSynchronize(s));
    double t = 0.0;
    for (double v : np) t += v;
    nrm = std::sqrt(t);
    (void)gv;
    return INTI_OK;
}

// GMRES(m) solving A x = b to ||b - A x|| <= tol_abs; x in/out (device).
// prec (or null): a right preconditioner P, GMRES on A P y = b - A x0 with
// x = x0 + P y (the residual it minimises is the true one).
template <bool CPLX>
static int gmres_core(Op *op, Op *prec, GmresWork &W, const double *b, double *x, int maxiter, double tol_abs,
                      int use_graph, int check_every, int *iters, double *resnorm) {
    using T = typename Sc<CPLX>::T;
    using cd = std::complex<double>;
    Ctx *ctx = op->ctx;
    hipStream_t s = ctx->stream;
    const int64_t n = W.n;
    const int m = W.m;
    const dim3 gv((unsigned)((n + kGB - 1) / kGB));
    const size_t es = CPLX ? 16 : 8;
    int it = 0;
    double rn = 0.0;
    int rc = residual<CPLX>(op, W, b, x, (double *)W.r, rn);
    if (rc) return rc;
    const int saved_prof = ctx->profiling;
    ctx->profiling = 0;  // no event records inside the solver (or its graph)
    // INTI_GMRES_LOG=N: a progress line on stderr every N Arnoldi steps
    const char *log_env = std::getenv("INTI_GMRES_LOG");
    const int log_every = log_env ? std::max(0, std::atoi(log_env)) : 0;
    while (rn > tol_abs && it < maxiter) {
        // V[:,0] = vk = r / rn; g = (rn, 0, ...); k = 0
        hipLaunchKernelGGL(k_gaxpby<CPLX>, gv, dim3(kGB), 0, s, n, 1.0 / rn, (const T *)W.r, 0.0, (T *)W.V);
        hipLaunchKernelGGL(k_gaxpby<CPLX>, gv, dim3(kGB), 0, s, n, 1.0 / rn, (const T *)W.r, 0.0, (T *)W.vk);
        hipLaunchKernelGGL(k_gfill<double>, dim3((unsigned)(((m + 1) * (CPLX ? 2 : 1) + kGB - 1) / kGB)),
                           dim3(kGB), 0, s, (int64_t)(m + 1) * (CPLX ? 2 : 1), (double *)W.g, 0.0);
        hipLaunchKernelGGL(k_gfill<double>, dim3(1), dim3(kGB), 0, s, (int64_t)1, (double *)W.g, rn);
        hipLaunchKernelGGL(k_gfill<int>, dim3(1), dim3(kGB), 0, s, (int64_t)2, (int *)W.st, 0);
        INTI_HIP(ctx, hipGetLastError());
        int k = 0, kk = 0;
        std::vector<double> res(m);
        while (k < m && it + k < maxiter) {
            const int steps = std::min({check_every, m - k, maxiter - it - k});
            for (int q = 0; q < steps; ++q) {
                if (use_graph) {
                    if (!W.exec) {
                        // the apply's scratch must exist before capture: no
                        // allocation may happen while the stream records
                        rc = apply_reserve(op, 1);
                        if (!rc && prec) rc = apply_reserve(prec, 1);
                        if (rc) { ctx->profiling = saved_prof; return rc; }
                        INTI_HIP(ctx, hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
                        rc = arnoldi_step<CPLX>(op, prec, W, s);
                        hipGraph_t gph = nullptr;
                        hipError_t e = hipStreamEndCapture(s, &gph);
                        if (rc) { if (gph) (void)hipGraphDestroy(gph); ctx->profiling = saved_prof; return rc; }
                        if (e != hipSuccess) { ctx->profiling = saved_prof; return set_error(ctx, INTI_ERR_HIP, "gmres: graph capture failed"); }
                        W.graph = gph;
                        INTI_HIP(ctx, hipGraphInstantiate(&W.exec, W.graph, nullptr, nullptr, 0));
                    }
                    INTI_HIP(ctx, hipGraphLaunch(W.exec, s));
                } else {
                    rc = arnoldi_step<CPLX>(op, prec, W, s);
                    if (rc) { ctx->profiling = saved_prof; return rc; }
                }
            }
            k += steps;
            INTI_HIP(ctx, hipMemcpyAsync(res.data(), W.res, sizeof(double) * k, hipMemcpyDeviceToHost, s));
            INTI_HIP(ctx, hipStreamSynchronize(s));
            kk = k;
            if (log_every > 0 && (it + k) / log_every != (it + k - steps) / log_every)
                std::fprintf(stderr, "gmres: step %d, residual estimate %.3e (target %.3e)\n", it + k, res[k - 1],
                             tol_abs);
            for (int q = k - steps; q < k; ++q)
                if (res[q] <= tol_abs) { kk = q + 1; break; }
            if (kk < k || res[k - 1] <= tol_abs) break;
        }
        // solve the kk x kk triangular system H y = g on the host
        std::vector<double> Hh((size_t)(m + 1) * m * (CPLX ? 2 : 1)), gh((m + 1) * (CPLX ? 2 : 1));
        INTI_HIP(ctx, hipMemcpyAsync(Hh.data(), W.H, es * (size_t)(m + 1) * m, hipMemcpyDeviceToHost, s));
        INTI_HIP(ctx, hipMemcpyAsync(gh.data(), W.g, es * (m + 1), hipMemcpyDeviceToHost, s));
        INTI_HIP(ctx, hipStreamSynchronize(s));
        std::vector<cd> y(kk);
        auto Hv = [&](int i, int j) {
            const size_t o = (size_t)i + (size_t)(m + 1) * j;
            return CPLX ? cd(Hh[2 * o], Hh[2 * o + 1]) : cd(Hh[o], 0.0);
        };
        for (int i = kk - 1; i >= 0; --i) {
            cd t = CPLX ? cd(gh[2 * i], gh[2 * i + 1]) : cd(gh[i], 0.0);
            for (int j = i + 1; j < kk; ++j) t -= Hv(i, j) * y[j];
            y[i] = t / Hv(i, i);
        }
        std::vector<double> yd(kk * (CPLX ? 2 : 1));
        for (int i = 0; i < kk; ++i) {
            if (CPLX) { yd[2 * i] = y[i].real(); yd[2 * i + 1] = y[i].imag(); }
            else yd[i] = y[i].real();
        }
        INTI_HIP(ctx, hipMemcpyAsync(W.y, yd.data(), es * kk, hipMemcpyHostToDevice, s));
        if (prec) {
            // x += P (V y): V y into t, then the preconditioner's apply adds onto x
            hipLaunchKernelGGL(k_gfill<double>, dim3((unsigned)((n * (CPLX ? 2 : 1) + kGB - 1) / kGB)), dim3(kGB),
                               0, s, n * (CPLX ? 2 : 1), (double *)W.t, 0.0);
            hipLaunchKernelGGL(k_gxupdate<CPLX>, gv, dim3(kGB), 0, s, (const T *)W.V, n, kk, (const T *)W.y,
                               (T *)W.t, n);
            INTI_HIP(ctx, hipGetLastError());
            rc = apply_vec(prec, W.t, x, n, 1.0, 1.0);
            if (rc) { ctx->profiling = saved_prof; return rc; }
        } else {
            hipLaunchKernelGGL(k_gxupdate<CPLX>, gv, dim3(kGB), 0, s, (const T *)W.V, n, kk, (const T *)W.y,
                               (T *)x, n);
        }
        INTI_HIP(ctx, hipGetLastError());
        it += kk;
        rc = residual<CPLX>(op, W, b, x, (double *)W.r, rn);
        if (rc) { ctx->profiling = saved_prof; return rc; }
    }
    ctx->profiling = saved_prof;
    if (iters) *iters = it;
    if (resnorm) *resnorm = rn;
    return INTI_OK;
}

static double dev_norm(Ctx *ctx, GmresWork &W, const double *v, bool cplx) {
    if (cplx)
        hipLaunchKernelGGL(k_gnorm<true>, dim3((unsigned)W.nb), dim3(kGB), 0, ctx->stream, (const double2 *)v, W.n, W.npart);
    else
        hipLaunchKernelGGL(k_gnorm<false>, dim3((unsigned)W.nb), dim3(kGB), 0, ctx->stream, v, W.n, W.npart);
    std::vector<double> np(W.nb);
    (void)hipMemcpyAsync(np.data(), W.npart, sizeof(double) * W.nb, hipMemcpyDeviceToHost, ctx->stream);
    (void)hipStreamSynchronize(ctx->stream);
    double t = 0.0;
    for (double x : np) t += x;
    return std::sqrt(t);
}

static int check_prec(Op *op, Op *prec) {
    if (!prec) return INTI_OK;
    if (prec->ctx != op->ctx) return set_error(op->ctx, INTI_ERR_ARG, "gmres: preconditioner on another context");
    if (prec->trg->n != op->src->n || prec->src->n != op->src->n)
        return set_error(op->ctx, INTI_ERR_SIZE, "gmres: preconditioner must be square of the operator's size");
    if (op_is_complex(prec) != op_is_complex(op))
        return set_error(op->ctx, INTI_ERR_ARG, "gmres: preconditioner and operator value types differ");
    return INTI_OK;
}

int gmres_solve(Op *op, Op *prec, const double *b, double *x, int restart, int maxiter, double rtol, double atol,
                int use_graph, int *iters, double *relres) {
    Ctx *ctx = op->ctx;
    const int64_t n = op->src->n;
    if (op->trg->n != n) return set_error(ctx, INTI_ERR_SIZE, "gmres: operator is not square");
    if (int rc = check_prec(op, prec)) return rc;
    if (restart < 1 || maxiter < 0) return set_error(ctx, INTI_ERR_ARG, "gmres: restart >= 1, maxiter >= 0");
    const bool cplx = op_is_complex(op);
    GmresWork W;
    int rc = gwork_alloc(ctx, W, restart, n, cplx);
    if (rc) return rc;
    const double bn = dev_norm(ctx, W, b, cplx);
    const double tol = std::max(rtol * bn, atol);
    double rn = 0.0;
    rc = cplx ? gmres_core<true>(op, prec, W, b, x, maxiter, tol, use_graph, 8, iters, &rn)
              : gmres_core<false>(op, prec, W, b, x, maxiter, tol, use_graph, 8, iters, &rn);
    if (rc) return rc;
    if (relres) *relres = bn > 0 ? rn / bn : rn;
    return INTI_OK;
}

int refine_solve(Op *op_hi, Op *op_lo, Op *prec, const double *b, double *x, int restart, int maxiter_inner,
                 double inner_rtol, int max_outer, double rtol, int use_graph, int *outer,
                 int *inner_total, double *relres) {
    Ctx *ctx = op_hi->ctx;
    const int64_t n = op_hi->src->n;
    if (op_lo->src != op_hi->src || op_lo->trg != op_hi->trg)
        return set_error(ctx, INTI_ERR_ARG, "refine: operators must share target and source");
    if (int rc = check_prec(op_hi, prec)) return rc;
    if (op_hi->trg->n != n) return set_error(ctx, INTI_ERR_SIZE, "refine: operator is not square");
    const bool cplx = op_is_complex(op_hi);
    if (cplx != op_is_complex(op_lo)) return set_error(ctx, INTI_ERR_ARG, "refine: value types differ");
    GmresWork W;
    int rc = gwork_alloc(ctx, W, restart, n, cplx);
    if (rc) return rc;
    const size_t es = cplx ? 16 : 8;
    void *r = nullptr, *d = nullptr;
    if (hipMalloc(&r, es * n) != hipSuccess || hipMalloc(&d, es * n) != hipSuccess) {
        if (r) (void)hipFree(r);
        return set_error(ctx, INTI_ERR_NOMEM, "refine: allocation failed");
    }
    struct Free { void *a, *b; ~Free() { (void)hipFree(a); (void)hipFree(b); } } fr{r, d};
    const double bn = dev_norm(ctx, W, b, cplx);
    double rn = 0.0;
    rc = cplx ? residual<true>(op_hi, W, b, x, (double *)r, rn) : residual<false>(op_hi, W, b, x, (double *)r, rn);
    if (rc) return rc;
    int o = 0, tot = 0;
    const dim3 gv((unsigned)((n + kGB - 1) / kGB));
    while (rn > rtol * bn && o < max_outer) {
        // d = 0; solve A_lo d = r to inner_rtol; x += d; r = b - A_hi x
        hipLaunchKernelGGL(k_gfill<double>, dim3((unsigned)((n * (cplx ? 2 : 1) + kGB - 1) / kGB)), dim3(kGB), 0,
                           ctx->stream, n * (cplx ? 2 : 1), (double *)d, 0.0);
        int it = 0;
        double irn = 0.0;
        const double itol = inner_rtol * rn;
        rc = cplx ? gmres_core<true>(op_lo, prec, W, (const double *)r, (double *)d, maxiter_inner, itol, use_graph, 8,
                                     &it, &irn)
                  : gmres_core<false>(op_lo, prec, W, (const double *)r, (double *)d, maxiter_inner, itol, use_graph, 8,
                                      &it, &irn);
        if (rc) return rc;
        tot += it;
        if (cplx)
            hipLaunchKernelGGL(k_gaxpby<true>, gv, dim3(kGB), 0, ctx->stream, n, 1.0, (const double2 *)d, 1.0, (double2 *)x);
        else
            hipLaunchKernelGGL(k_gaxpby<false>, gv, dim3(kGB), 0, ctx->stream, n, 1.0, (const double *)d, 1.0, x);
        rc = cplx ? residual<true>(op_hi, W, b, x, (double *)r, rn) : residual<false>(op_hi, W, b, x, (double *)r, rn);
        if (rc) return rc;
        ++o;
    }
    if (outer) *outer = o;
    if (inner_total) *inner_total = tot;
    if (relres) *relres = bn > 0 ? rn / bn : rn;
    return INTI_OK;
}

}  // namespace inti

// Direct-sum driver: operator parameters (post factors), the choice of
// source chunks, the multi-right-hand-side dispatch of k_apply
// (apply_kernel.hpp), and the epilogue pass (split reduction + post factor +
// fused CSR correction + identity + alpha/beta).
#include <complex>

#include "apply_kernel.hpp"
#include "apply_sym.hpp"

namespace inti {

// y_i = alpha * (post * sum_c part[c][i] + (dA x)_i + cid x_i) + beta * y_i,
// one right-hand side per blockIdx.y
// A chain of `split` loads per row and one thread per row leave the chip idle
// where rows are few: NS = 4 gives a block 64 rows, whose partials its four
// waves share in contiguous quarters, added in wave order (see launch_apply).
template <bool CPLX, int NS>
__global__ __launch_bounds__(256) void k_reduce(ReduceArgs a) {
    constexpr int ROWS = 256 / NS;
    __shared__ double2 s_w[NS][ROWS];
    const int row = threadIdx.x % ROWS, q = threadIdx.x / ROWS;
    const int64_t i = (int64_t)blockIdx.x * ROWS + row;
    if (NS == 1 && i >= a.m) return;
    const int64_t ic = i < a.m ? i : a.m - 1;
    const int r = blockIdx.y;
    const double *x = a.x + (CPLX ? 2 : 1) * (int64_t)r * a.ldx;
    double *y = a.y + (CPLX ? 2 : 1) * (int64_t)r * a.ldy;
    const int64_t pbase = (int64_t)r * a.split * a.m;
    const int per = (a.split + NS - 1) / NS, c0 = q * per, c1 = c0 + per < a.split ? c0 + per : a.split;
    double sr = 0.0, si = 0.0;
    // many partials per row (one per tile group of the symmetric sum): the
    // unrolled loop keeps several loads in flight per thread (the order of
    // the additions is unchanged)
    if constexpr (CPLX) {
        const double2 *pp = reinterpret_cast<const double2 *>(a.part) + pbase;
#pragma unroll 8
        for (int c = c0; c < c1; ++c) {
            double2 v = pp[(int64_t)c * a.m + ic];
            sr += v.x; si += v.y;
        }
    } else {
#pragma unroll 8
        for (int c = c0; c < c1; ++c) sr += a.part[pbase + (int64_t)c * a.m + ic];
    }
    if constexpr (NS > 1) {
        s_w[q][row] = make_double2(sr, si);
        __syncthreads();
        if (q || i >= a.m) return;
#pragma unroll
        for (int w = 1; w < NS; ++w) {
            sr += s_w[w][row].x;
            si += s_w[w][row].y;
        }
    }
    reduce_epilogue<CPLX>(a, i, x, y, sr, si);
}

// Long correction rows (a stencil of many elements per target: hundreds of
// entries per row): W lanes share a row, so the value and index loads of a
// wave are contiguous, and y_i += alpha (dA x)_i after k_reduce (which then
// skips the rows). The W partial sums of a row combine by a fixed butterfly,
// so the result does not depend on the launch. One row per W lanes, 256
// threads per block, one right-hand side per blockIdx.y.
struct CsrAddArgs {
    int64_t m;
    int64_t ldx, ldy;
    const int32_t *rowptr;
    const int32_t *colind;
    const double *cval;
    const double *x;
    double *y;
    double ar, ai;
};

template <bool CPLX, int W>
__global__ __launch_bounds__(256) void k_csr_add(CsrAddArgs a) {
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) / W;
    const int lane = threadIdx.x % W;
    if (i >= a.m) return;  // whole groups of W lanes leave together
    const int r = blockIdx.y;
    const double *x = a.x + (CPLX ? 2 : 1) * (int64_t)r * a.ldx;
    double *y = a.y + (CPLX ? 2 : 1) * (int64_t)r * a.ldy;
    const int32_t p0 = a.rowptr[i], p1 = a.rowptr[i + 1];
    double sr = 0.0, si = 0.0;
    if constexpr (CPLX) {
        const double2 *v = reinterpret_cast<const double2 *>(a.cval);
        const double2 *xv = reinterpret_cast<const double2 *>(x);
#pragma unroll 4
        for (int32_t p = p0 + lane; p < p1; p += W) {
            const double2 c = v[p], xx = xv[a.colind[p]];
            sr = fma(c.x, xx.x, fma(-c.y, xx.y, sr));
            si = fma(c.x, xx.y, fma(c.y, xx.x, si));
        }
    } else {
#pragma unroll 4
        for (int32_t p = p0 + lane; p < p1; p += W) sr = fma(a.cval[p], x[a.colind[p]], sr);
    }
#pragma unroll
    for (int o = W / 2; o > 0; o /= 2) {
        sr += __shfl_xor(sr, o, W);
        if constexpr (CPLX) si += __shfl_xor(si, o, W);
    }
    if (lane == 0) {
        if constexpr (CPLX) {
            y[2 * i] += a.ar * sr - a.ai * si;
            y[2 * i + 1] += a.ar * si + a.ai * sr;
        } else {
            y[i] += a.ar * sr;
        }
    }
}

// lanes per row of the correction: the fused per-thread walk of k_reduce
// for short rows (the element's own nodes: a few entries), a group of 16 or
// 64 lanes for long ones; 0 = fused
static int csr_lanes(const Csr *c) {
    if (!c || c->m == 0) return 0;
    const int64_t avg = c->nnz / c->m;
    return avg >= 96 ? 64 : avg >= 16 ? 16 : 0;
}

// ------------------------------------------------------------- dispatch
static ApplyFn pick_apply(int pde, int dim, int kind, int mixed, int nr) {
    if (pde == INTI_LAPLACE && dim == 2) return apply_pick_lap2(kind, mixed, nr);
    if (pde == INTI_LAPLACE && dim == 3) return apply_pick_lap3(kind, mixed, nr);
    if (pde == INTI_HELMHOLTZ && dim == 2) return apply_pick_helm2(kind, mixed, nr);
    if (pde == INTI_HELMHOLTZ && dim == 3) return apply_pick_helm3(kind, mixed, nr);
    if (pde == kHelmCK && dim == 3 && !mixed) return apply_pick_helm3c(kind, nr);
    return nullptr;
}

static RowFn pick_row(int pde, int dim, int kind, int mixed, int nr) {
    if (pde == INTI_LAPLACE && dim == 2) return row_pick_lap2(kind, mixed, nr);
    if (pde == INTI_LAPLACE && dim == 3) return row_pick_lap3(kind, mixed, nr);
    if (pde == INTI_HELMHOLTZ && dim == 2) return row_pick_helm2(kind, mixed, nr);
    if (pde == INTI_HELMHOLTZ && dim == 3) return row_pick_helm3(kind, mixed, nr);
    if (pde == kHelmCK && dim == 3 && !mixed) return row_pick_helm3c(kind, nr);
    return nullptr;
}

static SymFn pick_sym(int pde, int dim, int kind, int mixed, const SymPlan &P) {
    if (pde == INTI_LAPLACE && dim == 2) return sym_pick_lap2(kind, mixed, P.tile, P.G);
    if (pde == INTI_LAPLACE && dim == 3) return sym_pick_lap3(kind, mixed, P.tile, P.G);
    if (pde == INTI_HELMHOLTZ && dim == 2) return sym_pick_helm2(kind, mixed, P.tile, P.G);
    if (pde == INTI_HELMHOLTZ && dim == 3) return sym_pick_helm3(kind, mixed, P.tile, P.G);
    return nullptr;
}

bool op_is_complex(const Op *op) { return op->pde == INTI_HELMHOLTZ; }
int op_kernel_pde(const Op *op) { return op->pde == INTI_HELMHOLTZ && op->kimag != 0.0 ? kHelmCK : op->pde; }

// partial sums of the symmetric evaluation are capped: beyond this the
// plain direct sum runs
constexpr size_t kSymMaxBytes = size_t(4) << 30;

// Partial sums of the small-tile plans (n^2 / tile of them): the gain of the
// small tiles is not worth more memory than this.
constexpr size_t kSymSmallBytes = size_t(512) << 20;

// Tiles of 256 nodes keep the partial sums few, but a sum of n nodes is then
// only T (T + 1) / 2 blocks, and with a few waves per SIMD the chip waits on
// its dependency chains and on the last round of blocks. Smaller sums are
// therefore cut into one-wave blocks of 64 nodes (one target per lane, below
// 12 waves per CU of 128-node blocks, about 10,000 nodes) or 128 nodes (two
// targets per lane, below 72 tile pairs of 256 nodes per CU, about 49,000).
// The 2D Helmholtz pairs take 64 wherever the partial sums allow (in mixed
// precision up to 24 tile pairs per CU, about 28,000 nodes): their Hankel
// evaluation branches on the argument, and one wave without barriers waits
// for no other wave's branch. Measured, us per apply with 256 / 128 /
// 64-node tiles (before: one direction below 8,200 nodes):
//   3D Helmholtz CF FP64   4,320: 101 / 57 / 44 (one direction 83)
//                         12,000: 253 / 213 / 206    24,000: 837 / 734 / 750
//                         40,000: 2001 / 1926 / 2084 63,480: 4826 / 4894 / 5320
//   3D Laplace SL FP64     4,320: 55 / 22 / 19 (29)  8,500: 58 / 42 / 41
//                         24,000: 214 / 188 / 216    63,480: 1125 / 1171 / 1463
//   2D Helmholtz CF FP64   6,006: 333 / - / 179 (328)  30,720: 2592 / - / 2583
//   2D Helmholtz CF mixed  6,006: 123 / - / 82 (146)   40,000: 1989 / - / 2019
// Where the 256-node tile pairs nearly fill their last round (4 blocks per CU) the
// smaller tiles of the cheap pairs gain nothing and cost their staging: there
// 3D Laplace but for SL, from about 15,400 nodes, keeps 256 nodes, and so do mixed
// 2D Laplace DL (29,000), mixed Laplace SL and 2D (38,000) and, in the two rounds
// that end at 16,128 nodes, 2D Laplace but for the logarithms and mixed 3D
// Helmholtz SL and CF. With 256 / 128 at full rounds: 16,125 nodes, 2D Laplace DL
// mixed 0.88x, HS 0.90x; 3D Laplace HS FP64 0.92x, mixed 3D Helmholtz SL 0.93x;
// 28,000: mixed 3D Laplace DL 268 / 289 us, FP64 346 / 381; 46,077: mixed 2D
// Laplace DL 0.94x; with rounds 0.8 - 0.9 full (21,245, 26,877 nodes) 128 nodes
// are up to 9 % faster.
// Sums of 256 nodes or fewer run in one direction (k_apply_row). An explicit
// group has tiles of 256. Beyond kSymMaxBytes of partial sums the groups of
// 2 and 4 tiles halve and quarter them.
static bool full_rounds(const Op *op, int kind, int64_t blocks) {
    const int64_t cu = op->ctx->num_cu, round = 4 * cu, rounds = (blocks + round - 1) / round;
    if ((double)blocks < 0.93 * (double)(rounds * round)) return false;
    const bool mixed = op->precision == INTI_MIXED, two = rounds == 2, sl = kind == INTI_SL;
    const bool dl = kind == INTI_DL || kind == INTI_ADL;
    if (op->pde == INTI_HELMHOLTZ) return two && mixed && (sl || kind == INTI_COMB_SD);
    if (op->dim == 3) return sl ? mixed && blocks >= 44 * cu : rounds >= 2;
    if (mixed && blocks >= (dl ? 26 : 44) * cu) return true;
    return two && !sl && (mixed || kind != INTI_COMB_SD);
}

bool plan_sym(const Op *op, int kind, SymPlan &P) {
    if (op->sym == 0 || op->trg != op->src || kind >= INTI_FF_SL || op->kimag != 0.0) return false;
    const int64_t n = op->src->n;
    auto tiles = [n](int tile) { return (n + tile - 1) / tile; };
    if (tiles(kSymBS) < 2) return false;
    // a source split asked for (inti_op_set_launch) is the one-direction sum's,
    // and a group asked for is one of 256-node tiles: automatic mode takes those
    // two where the tile pairs give every CU two blocks. Below, one direction is
    // faster than such groups (4,320 nodes with groups of 1 / 4: 3D Helmholtz CF
    // 101 / 1,522 us against 85, mixed 3D Laplace SL 41 / 519 against 24)
    if (op->sym == 1 && (op->split > 0 || op->sym_group > 0) &&
        tiles(kSymBS) * (tiles(kSymBS) + 1) / 2 < 2LL * op->ctx->num_cu)
        return false;
    const size_t es = sizeof(double) * (op_is_complex(op) ? 2 : 1);
    if (op->sym_group == 0) {
        const int64_t t128 = tiles(128), t256 = tiles(kSymBS), cu = op->ctx->num_cu;
        const bool helm2 = op->pde == INTI_HELMHOLTZ && op->dim == 2;
        int tile = kSymBS;
        const bool mixed = op->precision == INTI_MIXED;
        if (helm2 ? !mixed || t256 * (t256 + 1) / 2 < 24 * cu : t128 * (t128 + 1) / 2 < 12 * cu) tile = 64;
        else if (helm2) tile = kSymBS;
        else if (t256 * (t256 + 1) / 2 < 72 * cu) tile = full_rounds(op, kind, t256 * (t256 + 1) / 2) ? kSymBS : 128;
        if (tile < kSymBS && (size_t)tiles(tile) * (size_t)n * es <= kSymSmallBytes) {
            P = SymPlan{tile, 1, tiles(tile), tiles(tile)};
            return true;
        }
    }
    for (int g : {1, 2, 4}) {
        if (op->sym_group && g != op->sym_group) continue;
        const int64_t T = tiles(kSymBS), S = (T + g - 1) / g;
        if ((size_t)S * (size_t)n * es <= kSymMaxBytes) {
            P = SymPlan{kSymBS, g, T, S};
            return true;
        }
    }
    return false;
}

// Whether nr right-hand sides of m targets and n sources take the one-launch
// sum (k_apply_row). Four targets per block and 64 threads per target keep
// every thread's source chain short; it reads each source's data once per 16
// threads instead of staging it, so it pays where launches, barriers and an
// idle chip cost more than the loads: few pairs. Against the symmetric sum it
// is faster up to about 1,800 nodes (3D Helmholtz CF 1,280: 15 / 20 us, 3,000:
// 41 / 33; 3D Laplace SL 1,280: 8 / 11, 3,000: 23 / 15) and, for 2D Helmholtz,
// up to 3,400 (CF 3,000: 73 / 102; 4,320: 145 / 125).
//
// Against the one-direction sum its time follows the blocks of the fullest CU x
// the chain of a thread, `work`, at about 0.2 us per unit in 3D Laplace and 0.4
// in FP64 2D Helmholtz, while the other sum takes 20 - 120 us whatever the size
// until it fills the chip. So the lines stand at a number of units per kind of
// pair. One column, m x n (units): times the row form is faster,
//   Laplace DL, CF         2,040^2 (64): 1.3 - 1.5, 5,000 x 1,000 (80): 1.1 - 1.25,
//                          2,300^2 (108): 0.83 - 1.0
//   Laplace SL, HS         2,300^2: 1.04 - 1.2, 300 x 8,192 (128): 0.8 - 1.0; FP64
//                          logarithms 5,000 x 2,500 (200): 1.3 - 1.6
//   3D Helmholtz FP64      3,300^2 (208): 1.02 - 1.3, 3,900^2 (244): DL, HS 0.9, SL, CF
//                          1.0 - 1.1
//   3D Helmholtz mixed     2,300^2: 1.08 - 1.15, 2,700^2 (129): 0.96 - 1.04; SL, HS
//                          3,000^2 (141): 1.2, 3,300^2: 0.85 - 0.9
//   2D far fields          (no Hankel function) FP64 3,900^2: 1.07 - 1.3, 40,000 x
//                          6,000 (3,760): 0.6 - 0.7; mixed SL 3,600^2 (228): 1.16, CF
//                          10,000 x 1,000 (160): 1.14, 3,300^2: 0.9, 40,000 x 6,000: 0.3
//   2D Helmholtz FP64      a wave of 4 targets x 16 neighbouring sources takes the
//                          same side of the Hankel functions' branch more often than
//                          one of 64 targets: 40,401 x 2,500 (1,600): 1.06 - 1.13,
//                          20,000^2 (6,260): 1.08 - 1.13, 30,720^2 (14,400): 0.90 - 1.03
//   2D Helmholtz mixed     40,401 x 1,000 (640): 1.01 - 1.26, 6,500^2 (714): 0.93 (DL),
//                          9,000^2: 0.74 - 1.04; 1,024 x 50,000: 0.5 - 0.66
// With 64 sources or fewer a part of each wave idles, but both sums then grow
// with m alone: 160,000 x 64: Laplace 0.8 - 1.05, 3D Helmholtz 1.1 - 2.4; 1,000,000
// x 3: 1.0 - 3, mixed far fields 0.78 - 1.1.
// Four right-hand sides reuse each pair value, so the staged kernel overtakes
// earlier: 2,048 nodes in 3D Helmholtz (2,040: 1.3 - 1.4x faster, 2,300: 0.8 -
// 1.05x), 1,800 for Laplace (3D SL 1,280: 12 / 18, 2,000: 18 / 18) and 3,700 in
// 2D Helmholtz (CF FP64 1,280: 26 / 140, 3,200: 106 / 156, mixed 3,200: 62 / 72,
// 4,320: 104 / 90); long chains (300 x 4,096 Laplace: 0.8 - 1.1x, 300 x 8,192 3D
// Helmholtz 0.6x, mixed 2D Helmholtz 0.8x) and many targets of few sources
// (40,000 x 64 Laplace 0.8 - 1.1x, with FP64 logarithms 1.45x, 200,000 x 4: 82 /
// 38, 80,000 x 3 mixed 2D Helmholtz 0.9x) are slower. 16 go to the matrix-core kernel
// at once.
static bool plan_row(const Op *op, int64_t m, int64_t n, bool sym, int nr) {
    if (op->split > 0 || n <= 0 || nr > 4) return false;
    const int kd = op->kind;
    const bool lap = op->pde == INTI_LAPLACE, ff = kd >= INTI_FF_SL, mixed = op->precision == INTI_MIXED;
    const bool hankel = !lap && op->dim == 2 && !ff;
    const bool log64 = lap && op->dim == 2 && !mixed && (kd == INTI_SL || kd == INTI_COMB_SD);
    const bool dl = kd == INTI_DL || kd == INTI_ADL || (kd == INTI_COMB_SD && !log64);
    const double pairs = (double)m * (double)n;
    const int64_t span = (int64_t)kRowTargets * op->ctx->num_cu, per_cu = (m + span - 1) / span;
    double lim;
    int64_t most_n, most_m;
    if (nr == 4) {
        if (hankel) lim = 3700.0, most_n = mixed ? 6144 : 8192, most_m = mixed ? 48 : 160;
        else if (lap) lim = 1800.0, most_n = log64 ? 4096 : 3072, most_m = log64 ? 80 : 20;
        else if (ff && op->dim == 2 && !mixed) lim = kd == INTI_FF_SL ? 3000.0 : 2240.0, most_n = kd == INTI_FF_SL ? 6144 : 4096, most_m = 20;
        else if (ff) lim = 2048.0, most_n = mixed ? 3072 : 4096, most_m = 20;
        else lim = 2048.0, most_n = mixed && dl ? 5120 : 4096, most_m = dl ? 40 : 20;
        return pairs <= lim * lim && n <= most_n && per_cu <= most_m;
    }
    if (sym) {
        lim = hankel ? 3400.0 : 1800.0;
        return op->sym != 2 && pairs <= lim * lim;
    }
    const double thin = ff && mixed ? 0.25 : 0.08;  // units of a chain of 16 sources or fewer
    const double chain = n > 64 ? (double)((n + 63) / 64) : n > 16 ? thin + (0.7 - thin) * (double)(n - 16) / 48.0 : thin;
    if (hankel) lim = mixed ? 700.0 : 8000.0;
    else if (lap) lim = log64 ? 200.0 : dl ? 80.0 : 109.0;
    else if (ff && op->dim == 2) lim = kd == INTI_FF_SL ? 240.0 : mixed ? 190.0 : 250.0;
    else if (mixed) lim = ff ? 109.0 : dl ? 120.0 : 160.0;
    else lim = kd == INTI_SL || kd == INTI_COMB_SD || kd == INTI_FF_SL ? 245.0 : 208.0;
    most_n = hankel && !mixed && m >= span ? INT64_MAX : 8192;
    // (a launch holds fewer than 2^32 threads, 64 per target)
    return (double)per_cu * chain <= lim && n <= most_n && m < int64_t(1) << 26;
}

KParams op_params(const Op *op, int *eff_kind) {
    using cd = std::complex<double>;
    KParams p = basic_params(op->k);
    p.kimag = op->kimag;
    int kind = op->kind;
    const cd c0(op->coefs[0], op->coefs[1]), c1(op->coefs[2], op->coefs[3]);
    cd post, ch(0.0, 0.0);
    double pr, pi;
    if (kind == INTI_COMB_SD || kind == INTI_COMB_AH || kind == INTI_FF_COMB) {
        const int ka = kind == INTI_COMB_SD ? INTI_SL : kind == INTI_COMB_AH ? INTI_ADL : INTI_FF_SL;
        const int kb = kind == INTI_COMB_SD ? INTI_DL : kind == INTI_COMB_AH ? INTI_HS : INTI_FF_DL;
        double ar, ai, br, bi;
        basic_post(op->pde, op->dim, ka, op->k, ar, ai);
        basic_post(op->pde, op->dim, kb, op->k, br, bi);
        if (c1 == cd(0.0, 0.0)) {  // only the first component remains
            kind = ka;
            post = c0 * cd(ar, ai);
        } else {
            // K = c1 postB (rawB + ch rawA), ch = c0 postA / (c1 postB); the
            // 3D/2D Helmholtz raw values of the combined kinds fold the
            // remaining constants as documented with helm3_raw / helm2_raw
            post = c1 * cd(br, bi);
            ch = c0 * cd(ar, ai) / post;
            if (op->pde == INTI_HELMHOLTZ && op->dim == 3 && kind == INTI_COMB_AH)
                ch = -ch;  // the ADL raw part inside COMB_AH carries -rdnx
            if (op->pde == INTI_HELMHOLTZ && op->dim == 2 && kind == INTI_COMB_AH)
                ch = -ch;
        }
    } else {
        basic_post(op->pde, op->dim, kind, op->k, pr, pi);
        post = cd(pr, pi);
    }
    p.postr = post.real(); p.posti = post.imag();
    p.chr = ch.real(); p.chi = ch.imag();
    if (eff_kind) *eff_kind = kind;
    return p;
}

// number of source chunks: enough workgroups to fill 256 CUs several
// times over, a multiple of the 8 XCDs when more than 8.
// Source chunks of the one-direction sum: block b works on target tile
// b / split and chunk b % split. The base split gives about 8 blocks per CU
// in whole 256-source tiles, a multiple of 8 from 8 on (all blocks of one XCD
// then share a chunk in their L2); an explicit split (inti_op_set_launch)
// replaces it. Without one, the plan then looks at splits from half to twice
// the base (multiples of 8 from 8 on) with chunks of whole LDS source tiles of
// the kernel and takes the one with the least rounds x chunk, where blocks run
// in rounds of `cap` resident blocks (occupancy x CUs): a grid just past a
// multiple of cap leaves its last round nearly empty.
// With 4 or 16 right-hand sides one or two blocks keep a CU busy, so the time
// follows the blocks of the fullest CU x chunk whatever the occupancy, and all
// splits from half to four times the base are looked at, down to one LDS tile
// (128 or 64 sources) per chunk; a shorter chunk would cost as much as a whole
// one (the inner loop runs over padding). chunk_cost, in sources, stands for a
// block's start and its partial sums; where a lone block per CU waits on its
// own chains (4 columns, and the Hankel functions) it costs as much as a second
// one beside it. Against rounds of resident blocks: 4 columns, 3D Helmholtz DL,
// 4,320 nodes 100 -> 75 us, 9,000: 280 -> 224; 16 columns, 1,700 nodes 79 -> 31,
// 4,320: 115 -> 102.
// With 16 columns the partial sums weigh more beside cheap pairs. A cost of 8 /
// 24, us: mixed 2D Helmholtz SL 10,000 nodes 366 / 289, 16,000: 772 / 692; mixed
// 3D Helmholtz SL 200,000 x 300: 201 / 165, 20,000 x 1,000: 70 / 62; 3D Laplace
// 200,000 x 300 mixed 99 / 76, FP64 118 / 106; mixed 2D far field 200,000 x 300
// (with the lone block's cost) 180, without 125. Where the pairs are dear, 24 is
// too much: FP64 2D Helmholtz SL, 6,500 nodes 8 % slower, FP64 2D Laplace SL
// 20,000 x 1,000: 60 / 73, FP64 3D Helmholtz CF 102 / 118. The mixed 2D
// Helmholtz SL and DL take 32 (6,500 nodes 152 / 147).
static int64_t chunk_cost(const Op *op, int nr) {
    if (nr != 16) return nr == 1 ? 0 : 8;
    const int kd = op->kind;
    if (op->precision == INTI_MIXED)
        return op->pde == INTI_HELMHOLTZ && op->dim == 2 && (kd == INTI_SL || kd == INTI_DL || kd == INTI_ADL) ? 32 : 24;
    return op->pde == INTI_LAPLACE && (op->dim == 3 || (kd != INTI_SL && kd != INTI_COMB_SD)) ? 24 : 8;
}
static int64_t base_split(const Op *op, int64_t m, int64_t n) {
    const int64_t ntiles = (m + kApplyBS - 1) / kApplyBS;
    const int64_t stiles = (n + kApplyBS - 1) / kApplyBS;
    int64_t s0 = op->split;
    if (s0 <= 0) {
        s0 = (8LL * op->ctx->num_cu + ntiles - 1) / ntiles;
        if (s0 >= 8) s0 = (s0 + 7) / 8 * 8;
    }
    return std::max<int64_t>(1, std::min(s0, stiles));
}

static void plan_split(const Op *op, int64_t m, int64_t n, ApplyFn fn, int nr, int &split, int64_t &chunk) {
    const int64_t ntiles = (m + kApplyBS - 1) / kApplyBS;
    const int64_t stiles = (n + kApplyBS - 1) / kApplyBS;
    const int64_t s0 = base_split(op, m, n);
    chunk = (stiles + s0 - 1) / s0 * kApplyBS;
    if (op->split <= 0 && fn && n > 0) {
        const int64_t gran = nr == 16 ? kMfmaTT : nr == 4 ? ApplyTile<4>::TT : ApplyTile<1>::TT;
        const int64_t gtiles = (n + gran - 1) / gran;
        const int64_t cus = op->ctx->num_cu, cap = nr == 1 ? (int64_t)fn(nullptr, dim3(0), nullptr) * cus : cus;
        const bool hankel = op->pde == INTI_HELMHOLTZ && op->dim == 2 && op->kind < INTI_FF_SL;
        const int64_t lone = nr == 4 || (nr == 16 && hankel) ? 1 : 0;
        const int64_t over = chunk_cost(op, nr), smax = std::min((nr == 1 ? 2 : 4) * s0, gtiles);
        auto cost_of = [&](int64_t c) { return ((ntiles * ((n + c - 1) / c) + cap - 1) / cap + lone) * (c + over); };
        int64_t best = cost_of(chunk);  // the base plan stays unless a candidate beats it
        for (int64_t s = std::max<int64_t>(1, s0 / 2); s <= smax; s += s < 8 || nr > 1 ? 1 : 8) {
            const int64_t c = (gtiles + s - 1) / s * gran, cost = cost_of(c);
            if (cost < best) {
                best = cost;
                chunk = c;
            }
        }
    }
    split = (int)((n + chunk - 1) / chunk);
    if (split < 1) split = 1;
}

// Scratch of the column blocks (16, 4, 1) of a call of nrhs columns, one column
// among them always and both the symmetric and the one-direction sums, also
// where the call takes the one-launch sum and needs none: after one eager call,
// calls of the same operator with one column, with overlapping operands or
// with set_symmetric(0) allocate nothing, as a stream capture requires.
int apply_reserve(const Op *op, int nrhs) {
    const int cw = op_is_complex(op) ? 2 : 1;
    const int64_t m = op->trg->n, n = op->src->n;
    int kind = op->kind;
    SymPlan sp;
    (void)op_params(op, &kind);
    // one column: at most twice the base split (plan_split)
    size_t bytes = sizeof(double) * cw * (size_t)m * 2 * base_split(op, m, n);
    for (int nr : {16, 4}) {
        if (nrhs < nr) continue;
        int split;
        int64_t chunk;
        plan_split(op, m, n, pick_apply(op_kernel_pde(op), op->dim, kind, op->precision == INTI_MIXED, nr), nr, split, chunk);
        bytes = std::max(bytes, sizeof(double) * cw * (size_t)m * split * nr);
    }
    if (plan_sym(op, kind, sp)) bytes = std::max(bytes, sizeof(double) * cw * (size_t)sp.S * (size_t)n);
    void *scr = nullptr;
    return ctx_scratch(op->ctx, kScrPartial, bytes, &scr);
}

int launch_apply(const DirectLaunch &L) {
    const Op *op = L.op;
    Ctx *ctx = op->ctx;
    const bool cplx = op_is_complex(op);
    const int cw = cplx ? 2 : 1;
    const int64_t m = op->trg->n, n = op->src->n;
    if (m == 0 || L.nrhs == 0) return INTI_OK;
    int kind = op->kind;
    const KParams kp = op_params(op, &kind);
    const bool given = L.part != nullptr;
    double *part = L.part;
    // the one-launch sum writes rows of y while others still read x: an apply
    // in place keeps the sums whose second kernel writes y
    const double *xend = L.x + cw * ((int64_t)(L.nrhs - 1) * L.ldx + n), *yend = L.y + cw * ((int64_t)(L.nrhs - 1) * L.ldy + m);
    const bool rows = L.x >= yend || L.y >= xend;
    if (!given) {
        int st = apply_reserve(op, L.nrhs);
        if (st) return st;
        void *scr = nullptr;
        st = ctx_scratch(ctx, kScrPartial, 0, &scr);
        if (st) return st;
        part = (double *)scr;
    }
    const int64_t ntiles = (m + kApplyBS - 1) / kApplyBS;
    SymPlan sp{};
    const bool sym = !given && plan_sym(op, kind, sp);
    for (int r0 = 0; r0 < L.nrhs;) {
        const int left = L.nrhs - r0;
        const int nr = left >= 16 ? 16 : left >= 4 ? 4 : 1;
        const double *xr = L.x + (int64_t)r0 * L.ldx * cw;
        double *yr = L.y + (int64_t)r0 * L.ldy * cw;
        ReduceArgs ra;
        ra.m = m;
        ra.ldx = L.ldx; ra.ldy = L.ldy;
        const int cl = csr_lanes(op->corr);
        ra.rowptr = op->corr && !cl ? op->corr->rowptr : nullptr;
        ra.colind = op->corr && !cl ? op->corr->colind : nullptr;
        ra.cval = op->corr && !cl ? op->corr->val : nullptr;
        ra.x = xr; ra.y = yr;
        ra.ar = L.alpha[0]; ra.ai = L.alpha[1];
        ra.br = L.beta[0]; ra.bi = L.beta[1];
        ra.beta_zero = (L.beta[0] == 0.0 && L.beta[1] == 0.0);
        ra.cr = op->cid[0]; ra.ci = op->cid[1];
        ra.pr = kp.postr; ra.pi = kp.posti;
        ra.has_id = (op->cid[0] != 0.0 || op->cid[1] != 0.0);
        RowFn rfn = rows && plan_row(op, m, n, sym, nr) ? pick_row(op_kernel_pde(op), op->dim, kind, op->precision == INTI_MIXED, nr)
                                                           : nullptr;
        ApplyFn fn = rfn || (sym && nr == 1) ? nullptr : pick_apply(op_kernel_pde(op), op->dim, kind, op->precision == INTI_MIXED, nr);
        int split = 1;
        int64_t chunk = n;
        if (fn) plan_split(op, m, n, fn, nr, split, chunk);
        if (given && n > 0) {
            // the largest split whose partials fit the caller's buffer, in
            // chunks of whole 256-source tiles
            const size_t per = sizeof(double) * cw * (size_t)m * nr;
            const int64_t cap = (int64_t)(L.part_bytes / per);
            if (cap < 1)
                return set_error(ctx, INTI_ERR_SIZE, "apply: the partial sums of this shape exceed the buffer");
            if (fn && split > cap) {
                const int64_t stiles = (n + kApplyBS - 1) / kApplyBS;
                chunk = (stiles + cap - 1) / cap * kApplyBS;
                split = (int)((n + chunk - 1) / chunk);
            }
        }
        int nsplit = split;
        if (rfn) {
            RowArgs a;
            a.s.m = m; a.s.n = n;
            a.s.tstride = m; a.s.sstride = n;
            a.s.tx = op->trg->coords; a.s.tn = op->trg->normals;
            a.s.sx = op->src->coords; a.s.sn = op->src->normals; a.s.sw = op->src->weights;
            a.s.x = xr; a.s.ldx = L.ldx; a.s.part = nullptr; a.s.split = 0; a.s.chunk = 0;
            a.s.p = kp;
            a.e = ra;
            a.tb = kRowTargets;
            if (ctx->profiling) INTI_HIP(ctx, hipEventRecord(ctx->ev0, ctx->stream));
            rfn(a, dim3((unsigned)((m + kRowTargets - 1) / kRowTargets)), ctx->stream);
            INTI_HIP(ctx, hipGetLastError());
            if (ctx->profiling) INTI_HIP(ctx, hipEventRecord(ctx->ev1, ctx->stream));
        } else if (n > 0 && nr == 1 && sym) {
            SymFn sfn = pick_sym(op->pde, op->dim, kind, op->precision == INTI_MIXED, sp);
            if (!sfn) return set_error(ctx, INTI_ERR_UNSUPPORTED, "no symmetric kernel for this operator");
            SymArgs a;
            a.n = n;
            a.xy = op->src->coords; a.nrm = op->src->normals; a.w = op->src->weights;
            a.x = xr; a.part = part;
            a.ntiles = sp.T; a.ngroups = sp.S;
            a.distinct = op->src->distinct ? 1 : 0;
            // c0 SL + c1 DL with c0 = -i k c1 (the combined field of the
            // reference's examples): ch q needs no LDS slot of its own
            a.ch_ik = kind == INTI_COMB_SD && op->pde == INTI_HELMHOLTZ && op->dim == 3 &&
                              std::fabs(kp.chr) <= 1e-15 * kp.k && std::fabs(kp.chi + kp.k) <= 1e-15 * kp.k
                          ? 1
                          : 0;
            a.p = kp;
            if (ctx->profiling) INTI_HIP(ctx, hipEventRecord(ctx->ev0, ctx->stream));
            sfn(a, sp.S * (sp.S + 1) / 2, ctx->stream);
            INTI_HIP(ctx, hipGetLastError());
            if (ctx->profiling) INTI_HIP(ctx, hipEventRecord(ctx->ev1, ctx->stream));
            nsplit = (int)sp.S;
        } else if (n > 0) {
            if (!fn) return set_error(ctx, INTI_ERR_UNSUPPORTED, "no direct-sum kernel for this operator");
            ApplyArgs a;
            a.m = m; a.n = n;
            a.tstride = m; a.sstride = n;
            a.tx = op->trg->coords; a.tn = op->trg->normals;
            a.sx = op->src->coords; a.sn = op->src->normals; a.sw = op->src->weights;
            a.x = xr; a.ldx = L.ldx; a.part = part; a.split = split; a.chunk = chunk;
            a.p = kp;
            dim3 grid((unsigned)(ntiles * split));
            if (ctx->profiling) INTI_HIP(ctx, hipEventRecord(ctx->ev0, ctx->stream));
            fn(&a, grid, ctx->stream);
            INTI_HIP(ctx, hipGetLastError());
            if (ctx->profiling) INTI_HIP(ctx, hipEventRecord(ctx->ev1, ctx->stream));
        }
        if (!rfn) {
            ra.split = n > 0 ? nsplit : 0;
            ra.part = part;
            // four waves per 64 rows from 16 partials on, while blocks of 256
            // rows would leave CUs idle (a solve of 4,320 nodes with 68 partials
            // per row: 1,975 -> 1,889 us for 26 sums; one sum of 6,006: 172 -> 168;
            // with 480 blocks, 122,880 nodes, it is bound by bandwidth and the
            // longer rows of the one-thread form are read faster: 95 / 103)
            const bool few = ra.split >= 16 && ntiles * nr < ctx->num_cu;
            dim3 rg((unsigned)(few ? (m + 63) / 64 : ntiles), (unsigned)nr);
            if (few && cplx) hipLaunchKernelGGL((k_reduce<true, 4>), rg, dim3(256), 0, ctx->stream, ra);
            else if (few) hipLaunchKernelGGL((k_reduce<false, 4>), rg, dim3(256), 0, ctx->stream, ra);
            else if (cplx) hipLaunchKernelGGL((k_reduce<true, 1>), rg, dim3(256), 0, ctx->stream, ra);
            else hipLaunchKernelGGL((k_reduce<false, 1>), rg, dim3(256), 0, ctx->stream, ra);
            INTI_HIP(ctx, hipGetLastError());
        }
        if (cl) {
            CsrAddArgs ca;
            ca.m = m; ca.ldx = L.ldx; ca.ldy = L.ldy;
            ca.rowptr = op->corr->rowptr; ca.colind = op->corr->colind; ca.cval = op->corr->val;
            ca.x = xr; ca.y = yr;
            ca.ar = L.alpha[0]; ca.ai = L.alpha[1];
            dim3 cg((unsigned)((m * cl + 255) / 256), (unsigned)nr);
            if (cplx) {
                if (cl == 64) hipLaunchKernelGGL((k_csr_add<true, 64>), cg, dim3(256), 0, ctx->stream, ca);
                else hipLaunchKernelGGL((k_csr_add<true, 16>), cg, dim3(256), 0, ctx->stream, ca);
            } else {
                if (cl == 64) hipLaunchKernelGGL((k_csr_add<false, 64>), cg, dim3(256), 0, ctx->stream, ca);
                else hipLaunchKernelGGL((k_csr_add<false, 16>), cg, dim3(256), 0, ctx->stream, ca);
            }
            INTI_HIP(ctx, hipGetLastError());
        }
        r0 += nr;
    }
    return INTI_OK;
}

}  // namespace inti

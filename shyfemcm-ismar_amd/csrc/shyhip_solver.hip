// shyhip_solver.hip -- zeta system solve on gfx950.
//
// Preconditioner: block-Jacobi ILU(0).  Rows are split into contiguous blocks
// (<= 1024 rows, one workgroup each); each diagonal block is factorised in
// LDS with level scheduling (rows of one level in parallel, workgroup
// barriers between levels).  Every factor entry (i,j) is computed as
// a_ij - sum_k l_ik u_kj over the pattern, k ascending -- the updates of
// ilu0's IKJ loop (spk_ilut.f90:1832-1950) in their order, listed once on
// the host -- so a basin of at most one block of nodes gets exactly ILU(0);
// lusol :2309-2345 applies it.  The block factors are staged in LDS by every
// kernel that applies them.
//
// Krylov method: BiCGStab in the arrangement the reference uses -- runrc with
// ipar(2)=1, which bisinit maps to LEFT preconditioning (spk_iters.f90:
// 1061-1334, 3433-3500) -- with stopping test ||M^-1 r|| <= rtol*||M^-1 r0||
// + atol and at most itermax matvecs.  Basins whose blocks can all be
// resident at once are solved in one launch (k_zeta, see there).  The others
// take two kernels per iteration: every vector update is fused into the
// SpMV/preconditioner kernel that consumes it (the update of x and r closing
// an iteration is done by the first kernel of the next, from five dot
// products of the second), and every dot product is written as per-workgroup
// partials that every workgroup of the next kernel reduces itself in the
// same fixed order -- no atomics or device-scope fences, visibility comes
// from the kernel boundary, and all workgroups (and all runs) see bitwise
// identical scalars.
// The FP32 path runs this in FP32 inside an FP64 iterative refinement whose
// control also lives on the device: inside the one launch, or every kernel
// of a refinement round returns at once when the FP64 residual test has
// passed, so the host enqueues the expected number of rounds and reads the
// flags once.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstring>

#include <algorithm>
#include <cmath>
#include <functional>

#include "shyhip_budget.h"
#include "shyhip_internal.h"

namespace shy {

// scalar slots; rho/alpha/omega are double-buffered by iteration parity so a
// kernel never overwrites a value that another workgroup of it still reads
enum { SC_TARGET = 0, SC_NORM0 = 1, SC_RHO = 2, SC_ALPHA = 4, SC_OMEGA = 6, SC_RNORM = 8, SC_RES64 = 9,
       SC_BNORM = 10 };
// partial-sum regions: [region][q][workgroup]
enum { PR_A = 0, PR_B = 1, PR_C = 2, PR_R = 3 };

template <typename V>
struct SolvArgs {
    int n, nblk, brows, mx, mxp, itermax, sweeps;
    double rtol, atol;
    const int *rowptr, *cols;
    const V *A;
    const int *brp, *bcol, *bsrc, *bdiag, *frows, *flptr, *fnlev, *brows_l, *blptr, *bnlev;
    const int *cp_ptr, *cp_a, *cp_b, *bjd;
    const int *pcol, *prp, *pdg;     // block pattern at a fixed stride per block
    const int *elp, *elr, *enlev;    // entry-level factorisation schedule
    const int4 *fdesc;               // per entry in level order: {entry, pairs begin, end, pivot}
    const int2 *fpair;               // update pairs {l_ik, u_kj} entries, relative to the block
    int edmax;
    const int *ell_col, *ell_len;    // ELL slices of the matrix rows
    const V *ell_a;
    // block factor rows slot-major ([k*n + i]: slot 0 the inverted pivot,
    // slots 1..nL the L entries, then the U entries; local columns) and per
    // row nL | cnt << 8; fs_val null: not used
    const int *fs_col, *fs_meta;
    V *fs_val;
    V *lu;                           // block factors at a fixed stride per block
    const double *aval;
    V *b, *x0, *r0, *r, *p0, *p1, *v0, *v1, *s, *t, *dx;
    double *part, *scal;
    int *ctrl;
    int nparts;      // stride of one partial-sum array
    // exchange slots of the one-launch solve, emptied by the factorisation
    // (null: not used)
    void *xch;
    unsigned long long *pslot;
    const int *send;
    int nsend;
    // two-kernel iteration with halos (null: not laid out): byte offsets of
    // the row's columns in its block's operand and of its factor columns in
    // the block's rows, two per word [k/2][n], each block's halo rows
    const unsigned *lcol, *fcol;
    const int *hcol, *hcnt;
    int hmax;
};

template <typename V>
static SolvArgs<V> solv_args(Model &M, const V *A, V *b, V *x0) {
    // zeroed first: the bytes, padding included, identify the launches
    SolvArgs<V> a;
    std::memset(&a, 0, sizeof a);
    a.n = M.nkn; a.nblk = M.sv.nblk; a.brows = M.sv.brows; a.mx = M.sv.max_blk_nnz; a.mxp = M.sv.max_blk_pairs;
    a.itermax = M.p.itermax;
    a.sweeps = M.p.tri_sweeps;
    a.rtol = M.p.rtol; a.atol = M.p.atol;
    a.rowptr = M.m.rowptr; a.cols = M.m.cols; a.A = A;
    a.brp = M.m.blk_rowptr; a.bcol = M.m.blk_cols; a.bsrc = M.m.blk_src; a.bdiag = M.m.blk_diag;
    a.frows = M.m.fwd_rows; a.flptr = M.m.fwd_lptr; a.fnlev = M.m.fwd_nlev;
    a.brows_l = M.m.bwd_rows; a.blptr = M.m.bwd_lptr; a.bnlev = M.m.bwd_nlev;
    a.cp_ptr = M.m.blk_cp_ptr; a.cp_a = M.m.blk_cp_a; a.cp_b = M.m.blk_cp_b; a.bjd = M.m.blk_jd;
    a.pcol = M.m.blk_pcol; a.prp = M.m.blk_prp; a.pdg = M.m.blk_pdg;
    a.elp = M.m.blk_elp; a.elr = M.m.blk_elr; a.enlev = M.m.blk_enlev; a.edmax = M.sv.max_elev;
    a.fdesc = (const int4 *)M.m.blk_fdesc; a.fpair = (const int2 *)M.m.blk_fpair;
    a.ell_col = M.m.ell_col; a.ell_len = M.m.ell_len; a.ell_a = (const V *)M.sv.ell_a;
    a.fs_col = M.m.fs_col; a.fs_meta = M.m.fs_meta;
    // factor rows in registers: one row per work-item and Jacobi sweeps
    a.fs_val = (M.p.tri_sweeps > 0 && M.sv.brows <= kThreads) ? (V *)M.sv.fs_val : nullptr;
    a.lu = (V *)M.sv.lu; a.aval = M.s.aval;
    a.b = b; a.x0 = x0;
    a.r0 = (V *)M.sv.r0; a.r = (V *)M.sv.r; a.p0 = (V *)M.sv.p0; a.p1 = (V *)M.sv.p1;
    a.v0 = (V *)M.sv.v0; a.v1 = (V *)M.sv.v1; a.s = (V *)M.sv.s; a.t = (V *)M.sv.t; a.dx = (V *)M.sv.dx;
    a.part = M.sv.part; a.scal = M.sv.scal; a.ctrl = M.sv.ctrl;
    a.nparts = M.sv.nparts;
    if (M.sv.zeta_t > 0) {
        a.xch = M.sv.xch;
        a.pslot = M.sv.pslot;
        a.send = M.m.z_send;
        a.nsend = M.sv.zeta_nsend;
    } else if (M.sv.zeta_hmax > 0) {
        a.lcol = M.m.z_lcol; a.fcol = M.m.z_fcol; a.hcol = M.m.z_hcol; a.hcnt = M.m.z_hcnt; a.hmax = M.sv.zeta_hmax;
    }
    return a;
}

// ---------------------------------------------------------------- reductions
// Workgroup sums: butterfly within each 64-lane wavefront (every lane ends
// with the same total), then the wavefront totals added in a fixed order.
// The same data always give the same bits.
constexpr int kWaves = kThreads / 64;
constexpr int kRegion = 8;            // partial-sum slots per region

// v from the DPP-permuted lane (CTRL: a GFX9 DPP control code whose source
// lane always lies in the same row of 16, so every lane is written)
template <int CTRL>
__device__ inline double dpp_f64(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}

__device__ inline double readlane_f64(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Sum over the 64 lanes, the same in every lane: exchanges within rows of
// 16 by DPP (lanes i^1, i^2 by quad permutes, then the mirrored halves of
// 8 and of 16 lanes, which hold equal values by then), then the four row
// sums read from lanes 0, 16, 32, 48.  Each exchange adds two values that
// the partner lane adds in the other order, so all lanes agree bitwise.
__device__ inline double wave_sum(double v) {
    v = v + dpp_f64<0xB1>(v);      // quad_perm [1,0,3,2]
    v = v + dpp_f64<0x4E>(v);      // quad_perm [2,3,0,1]
    v = v + dpp_f64<0x141>(v);     // row_half_mirror
    v = v + dpp_f64<0x140>(v);     // row_mirror
    return (readlane_f64(v, 0) + readlane_f64(v, 16)) + (readlane_f64(v, 32) + readlane_f64(v, 48));
}

template <int NQ>
__device__ inline void block_sum(double (&v)[NQ]) {
    __shared__ double red[NQ][kWaves];
    for (int q = 0; q < NQ; q++) v[q] = wave_sum(v[q]);
    if ((threadIdx.x & 63) == 0)
        for (int q = 0; q < NQ; q++) red[q][threadIdx.x >> 6] = v[q];
    __syncthreads();
    for (int q = 0; q < NQ; q++) {
        double t = red[q][0];
        for (int w = 1; w < kWaves; w++) t += red[q][w];
        v[q] = t;
    }
    __syncthreads();
}

// per-workgroup partials: part[(region*kRegion + q)*nparts + slot], slot =
// the workgroup's block (or its index)
template <int NQ>
__device__ inline void store_partials(double (&vals)[NQ], double *part, int region, int nparts, int slot) {
    block_sum<NQ>(vals);
    if (threadIdx.x == 0)
        for (int q = 0; q < NQ; q++) part[((size_t)region * kRegion + q) * nparts + slot] = vals[q];
}

// Block of a workgroup: xcd_block(w, n) gives each XCD a contiguous range of
// blocks, so the blocks a block couples to (its neighbours in node order)
// and its own factors are mostly produced on the same XCD and read from
// its L2.

// total of the partials of the previous kernel (n workgroups), computed by
// every workgroup in the same order; the result is returned to all threads
template <int NQ>
__device__ inline void sum_partials(const double *part, int region, int nparts, int n, double (&out)[NQ]) {
    for (int q = 0; q < NQ; q++) out[q] = 0.;
    for (int i = threadIdx.x; i < n; i += kThreads)
        for (int q = 0; q < NQ; q++) out[q] += part[((size_t)region * kRegion + q) * nparts + i];
    block_sum<NQ>(out);
}

// The same total with this work-item's first partials loaded early (the
// loads are issued at kernel start, the reduction done when needed); only
// the first nq of the NQ slots are read, the others are zero.
template <int NQ>
struct Partials {
    double v[NQ];
    __device__ inline void load(const double *part, int region, int nparts, int n, int nq) {
#pragma unroll
        for (int q = 0; q < NQ; q++)
            v[q] = (q < nq && (int)threadIdx.x < n) ? part[((size_t)region * kRegion + q) * nparts + threadIdx.x] : 0.;
    }
    __device__ inline void total(const double *part, int region, int nparts, int n, int nq, double (&out)[NQ]) {
#pragma unroll
        for (int q = 0; q < NQ; q++) out[q] = 0. + v[q];
        for (int i = threadIdx.x + kThreads; i < n; i += kThreads)
            for (int q = 0; q < nq; q++) out[q] += part[((size_t)region * kRegion + q) * nparts + i];
        block_sum<NQ>(out);
    }
};

__device__ inline bool breakdown(double x) {   // brkdn: zero or not finite
    if (x > 0.) return !(1. / x > 0.);
    if (x < 0.) return !(1. / x < 0.);
    return true;
}

// ---------------------------------------------------------------- block solve
// One diagonal block of the preconditioner: row starts, diagonal positions,
// local columns and factor values (diagonal stored inverted), either in
// global memory or staged in LDS.  Entry indices are relative to the arrays
// the view points at.
template <typename V>
struct BlockView {
    const int *rp, *dg, *col;
    const V *lu;
};

// LDS bytes of a kernel that stages its block: y and w (brows values each),
// the block's factor values and columns, row starts and diagonals
template <typename V>
static size_t staged_lds(int brows, int mx) {
    return (size_t)(2 * brows + mx) * sizeof(V) + (size_t)(mx + 2 * brows + 1) * sizeof(int);
}

// The block's factors, columns, row starts and diagonals at the block's
// fixed stride: load() issues the global loads into registers (up to
// kStageRegs entries per work-item; the rest are copied by store()), store()
// writes them to LDS and returns the view (visible after the caller's
// barrier).  Without STAGE the view points at global memory.
constexpr int kStageRegs = 8;

template <typename V, bool STAGE>
struct BlockStage {
    V lu[kStageRegs];
    int col[kStageRegs];
    int rp = 0, dg = 0, rpe = 0;
    __device__ inline void load(const SolvArgs<V> &a, int blk) {
        if (!STAGE) return;
        const size_t e0 = (size_t)blk * a.mx;
#pragma unroll
        for (int k = 0; k < kStageRegs; k++) {
            const int e = threadIdx.x + k * kThreads;
            if (e < a.mx) {
                lu[k] = a.lu[e0 + e];
                col[k] = a.pcol[e0 + e];
            }
        }
        const size_t r0 = (size_t)blk * (a.brows + 1);
        if ((int)threadIdx.x < a.brows) {
            rp = a.prp[r0 + threadIdx.x];
            dg = a.pdg[(size_t)blk * a.brows + threadIdx.x];
        }
        if (threadIdx.x == 0) rpe = a.prp[r0 + a.brows];
    }
    __device__ inline BlockView<V> store(const SolvArgs<V> &a, int blk, unsigned char *lds) const {
        const size_t e0 = (size_t)blk * a.mx, r0 = (size_t)blk * (a.brows + 1), d0 = (size_t)blk * a.brows;
        if (!STAGE) return BlockView<V>{a.prp + r0, a.pdg + d0, a.pcol + e0, a.lu + e0};
        V *llu = reinterpret_cast<V *>(lds);
        int *lrp = reinterpret_cast<int *>(llu + a.mx);
        int *ldg = lrp + a.brows + 1;
        int *lcol = ldg + a.brows;
#pragma unroll
        for (int k = 0; k < kStageRegs; k++) {
            const int e = threadIdx.x + k * kThreads;
            if (e < a.mx) {
                llu[e] = lu[k];
                lcol[e] = col[k];
            }
        }
        for (int e = threadIdx.x + kStageRegs * kThreads; e < a.mx; e += kThreads) {
            llu[e] = a.lu[e0 + e];
            lcol[e] = a.pcol[e0 + e];
        }
        if ((int)threadIdx.x < a.brows) {
            lrp[threadIdx.x] = rp;
            ldg[threadIdx.x] = dg;
        }
        for (int li = threadIdx.x + kThreads; li < a.brows; li += kThreads) {
            lrp[li] = a.prp[r0 + li];
            ldg[li] = a.pdg[d0 + li];
        }
        if (threadIdx.x == 0) lrp[a.brows] = rpe;
        return BlockView<V>{lrp, ldg, lcol, llu};
    }
};

// (LU)^-1 y for the local rows of block blk; y and w are LDS buffers of
// the block's rows, y holds the right-hand side (visible: the caller's
// barrier).  Returns the buffer that holds the result.
//   Exact: level-scheduled forward and backward substitution in lusol's
//   order, in place in y (rows of a level written by any work-item, a
//   barrier after each level).
//   a.sweeps = k > 0: each triangular factor applied by k Jacobi sweeps,
//   x <- y - L x from x = y, then x <- D^-1 (f - U x) from x = D^-1 f,
//   alternating between y and w (one barrier per sweep) with the
//   right-hand sides in registers; the result does not depend on the
//   order in which wavefronts run, and each work-item reads back only the
//   rows it wrote itself.
template <typename V>
__device__ inline V *block_lusol(const SolvArgs<V> &a, const BlockView<V> &B, int blk, int b0, int nb, V *y,
                                 V *w) {
    if (a.sweeps > 0) {
        constexpr int RPT = kMaxBlockRows / kThreads;   // rows per work-item
        V bl[RPT];
        V *src = y, *dst = w;
        int nr = 0;
        for (int li = threadIdx.x; li < nb; li += blockDim.x, nr++) bl[nr] = y[li];
        for (int sw = 1; sw < a.sweeps; sw++) {
            nr = 0;
            for (int li = threadIdx.x; li < nb; li += blockDim.x, nr++) {
                V acc = bl[nr];
                for (int q = B.rp[li]; q < B.dg[li]; q++) acc = acc - B.lu[q] * src[B.col[q]];
                dst[li] = acc;
            }
            __syncthreads();
            V *t = src; src = dst; dst = t;
        }
        // backward, right-hand side f = the forward result (own rows)
        nr = 0;
        for (int li = threadIdx.x; li < nb; li += blockDim.x, nr++) {
            bl[nr] = src[li];
            dst[li] = B.lu[B.dg[li]] * bl[nr];
        }
        __syncthreads();
        { V *t = src; src = dst; dst = t; }
        for (int sw = 1; sw < a.sweeps; sw++) {
            nr = 0;
            for (int li = threadIdx.x; li < nb; li += blockDim.x, nr++) {
                V acc = bl[nr];
                for (int q = B.dg[li] + 1; q < B.rp[li + 1]; q++) acc = acc - B.lu[q] * src[B.col[q]];
                dst[li] = B.lu[B.dg[li]] * acc;
            }
            __syncthreads();
            V *t = src; src = dst; dst = t;
        }
        return src;
    }
    const int stride = a.brows + 1;
    const int *lp = a.flptr + (size_t)blk * stride;
    const int nf = a.fnlev[blk];
    for (int lv = 0; lv < nf; lv++) {
        for (int t = lp[lv] + threadIdx.x; t < lp[lv + 1]; t += blockDim.x) {
            const int li = a.frows[b0 + t];
            V acc = y[li];
            for (int q = B.rp[li]; q < B.dg[li]; q++) acc = acc - B.lu[q] * y[B.col[q]];
            y[li] = acc;
        }
        __syncthreads();
    }
    const int *bp = a.blptr + (size_t)blk * stride;
    const int nbl = a.bnlev[blk];
    for (int lv = 0; lv < nbl; lv++) {
        for (int t = bp[lv] + threadIdx.x; t < bp[lv + 1]; t += blockDim.x) {
            const int li = a.brows_l[b0 + t];
            V acc = y[li];
            for (int q = B.dg[li] + 1; q < B.rp[li + 1]; q++) acc = acc - B.lu[q] * y[B.col[q]];
            y[li] = B.lu[B.dg[li]] * acc;
        }
        __syncthreads();
    }
    return y;
}

// One row of the block factors held in registers by the work-item that
// owns the row (blocks of at most one row per work-item): its inverted
// pivot (slot 0), L entries (slots 1..nl) and U entries (slots nl+1..cnt-1)
// with their local columns, loaded at kernel start from the slot-major copy,
// so that the Jacobi sweeps read only the neighbour values from LDS.  Same
// operations in the same order as block_lusol's sweeps.
constexpr int kFacWidth = kEllWidth;

template <typename V>
struct FacRow {
    V v[kFacWidth];
    int c[kFacWidth];
    int nl = 0, cnt = 0;
    __device__ __attribute__((always_inline)) void load(const SolvArgs<V> &a, int i, bool valid) {
        if (!valid) return;
        const int meta = a.fs_meta[i];
        nl = meta & 255;
        cnt = meta >> 8;
#pragma unroll
        for (int k = 0; k < kFacWidth; k++) {
            v[k] = a.fs_val[(size_t)k * a.n + i];
            c[k] = a.fs_col[(size_t)k * a.n + i];
        }
    }
    // (LU)^-1 y for this row, a.sweeps > 0 Jacobi sweeps per factor
    // alternating between y and w; returns the buffer holding the result
    __device__ __attribute__((always_inline)) V *lusol(int sweeps, bool mine, int li, V *y, V *w) const {
        V *src = y, *dst = w;
        V bl = mine ? y[li] : (V)0;
        for (int sw = 1; sw < sweeps; sw++) {
            if (mine) {
                V acc = bl;
#pragma unroll
                for (int k = 1; k < kFacWidth; k++)
                    if (k <= nl) acc = acc - v[k] * src[c[k]];
                dst[li] = acc;
            }
            __syncthreads();
            V *t = src; src = dst; dst = t;
        }
        const V dinv = v[0];
        if (mine) {
            bl = src[li];
            dst[li] = dinv * bl;
        }
        __syncthreads();
        { V *t = src; src = dst; dst = t; }
        for (int sw = 1; sw < sweeps; sw++) {
            if (mine) {
                V acc = bl;
#pragma unroll
                for (int k = 0; k < kFacWidth; k++)
                    if (k > nl && k < cnt) acc = acc - v[k] * src[c[k]];
                dst[li] = dinv * acc;
            }
            __syncthreads();
            V *t = src; src = dst; dst = t;
        }
        return src;
    }
};

// ILU(0) of each diagonal block (the pivot is stored inverted).  Row i,
// entries in column order:
//   l_ij = (a_ij - sum_{k<j} l_ik u_kj) * (1/u_jj)   (j < i)
//   u_ij =  a_ij - sum_{k<i} l_ik u_kj               (j >= i)
// with the (k ascending) update pairs of each entry.  Entries are computed
// level by level of the entry dependence graph (an entry's level is one
// more than that of every entry it reads), one work-item per entry, a
// barrier per level; each entry is the same expression in the same order
// as in a row-by-row factorisation.  Four wavefronts per block: staging
// and the wide early levels spread over 256 work-items (measured on the
// 50k-node lagoon, 256-row blocks: 56 us against 60 us with two
// wavefronts and 75 us with one).
// Per entry, in level order, one descriptor {entry, first pair, end of
// pairs, pivot entry (>= 0) / -1 (U) / -2 - row (diagonal)} and the pairs'
// two entries packed together, all relative to the block; with stage the
// descriptors and pairs are copied to LDS.
constexpr int kFactorThreads = 256;
// Warm start (sweeps > 0): the factors of the previous solve, whose matrix
// differs little, refined by synchronous sweeps over all entries at once
// (Chow and Patel, fine-grained parallel ILU, SIAM J. Sci. Comput. 37,
// 2015): every entry is recomputed from the current values of the others,
// in the same operations as above; after k sweeps every entry within
// dependence depth k is exact.  kWarmEntries bounds the entries a
// work-item keeps the matrix values of (larger blocks run cold).
constexpr int kWarmEntries = 8;

template <typename V>
__device__ inline void zeta_empty_slots(const SolvArgs<V> &a, int blk, int b0, int nb);

template <typename V>
__global__ __launch_bounds__(kFactorThreads) void k_bilu_factor(SolvArgs<V> a, int stage, int sweeps) {
    extern __shared__ double smem[];
    V *val = reinterpret_cast<V *>(smem);
    const int blk = blockIdx.x, b0 = blk * a.brows;
    const int nb = min(a.n, b0 + a.brows) - b0;
    // the one-launch solve that follows: no slot filled, no flag set
    if (a.pslot) zeta_empty_slots(a, blk, b0, nb);
    const int q0 = a.brp[b0], q1 = a.brp[b0 + nb], ne = q1 - q0;
    const int p0 = a.cp_ptr[q0], np = a.cp_ptr[q1] - p0;
    const int nl = a.enlev[blk];
    const int *elp = a.elp + (size_t)blk * (a.edmax + 1);   // level starts
    const int4 *desc = a.fdesc + (size_t)blk * a.mx;         // entries by level
    const int2 *pairs = a.fpair + p0;
    // the lists start 16-byte aligned after the values (two value buffers
    // when warm)
    const size_t vreg = (a.mx * sizeof(V) + 15) & ~(size_t)15;
    unsigned char *lfree = reinterpret_cast<unsigned char *>(smem) + vreg * (sweeps > 0 ? 2 : 1);
    if (stage) {
        int4 *l_d = reinterpret_cast<int4 *>(lfree);
        int2 *l_p = reinterpret_cast<int2 *>(l_d + a.mx);
        int *l_e = reinterpret_cast<int *>(l_p + a.mxp);
        for (int t = threadIdx.x; t < ne; t += blockDim.x) l_d[t] = desc[t];
        for (int p = threadIdx.x; p < np; p += blockDim.x) l_p[p] = pairs[p];
        for (int t = threadIdx.x; t <= nl; t += blockDim.x) l_e[t] = elp[t];
        desc = l_d; pairs = l_p; elp = l_e;
    }
    if (sweeps > 0) {
        // this work-item's entries: descriptors and matrix values in registers
        V av[kWarmEntries];
        int4 dd[kWarmEntries];
        const V *prev = a.lu + (size_t)blk * a.mx;
        V *nxt = reinterpret_cast<V *>(reinterpret_cast<unsigned char *>(smem) + vreg);
#pragma unroll
        for (int k = 0; k < kWarmEntries; k++) {
            const int t = threadIdx.x + k * blockDim.x;
            if (t < ne) {
                dd[k] = desc[t];
                av[k] = (V)a.aval[a.bsrc[q0 + dd[k].x]];
            }
        }
        for (int e = threadIdx.x; e < ne; e += blockDim.x) val[e] = prev[e];
        __syncthreads();
        V *cur = val;
        for (int sw = 0; sw < sweeps; sw++) {
#pragma unroll
            for (int k = 0; k < kWarmEntries; k++) {
                const int t = threadIdx.x + k * blockDim.x;
                if (t >= ne) break;
                const int4 d = dd[k];
                V acc = av[k];
                for (int p = d.y; p < d.z; p++) {
                    const int2 pr = pairs[p];
                    acc = acc - cur[pr.x] * cur[pr.y];
                }
                V out;
                if (d.w >= 0) out = acc * cur[d.w];
                else if (d.w == -1) out = acc;
                else {
                    if (acc == (V)0) atomicCAS(a.ctrl + CT_FACTOR, 0, 1 + b0 + (-2 - d.w));
                    out = (V)1 / acc;
                }
                nxt[d.x] = out;
            }
            __syncthreads();
            V *tmp = cur; cur = nxt; nxt = tmp;
        }
        if (cur != val) {
            for (int e = threadIdx.x; e < ne; e += blockDim.x) val[e] = cur[e];
            __syncthreads();
        }
    } else {
        for (int q = q0 + threadIdx.x; q < q1; q += blockDim.x) val[q - q0] = (V)a.aval[a.bsrc[q]];
        __syncthreads();
    }
    for (int lv = 0; lv < (sweeps > 0 ? 0 : nl); lv++) {
        for (int t = elp[lv] + threadIdx.x; t < elp[lv + 1]; t += blockDim.x) {
            const int4 d = desc[t];
            V acc = val[d.x];
            for (int p = d.y; p < d.z; p++) {
                const int2 pr = pairs[p];
                acc = acc - val[pr.x] * val[pr.y];
            }
            if (d.w >= 0) {
                val[d.x] = acc * val[d.w];
            } else if (d.w == -1) {
                val[d.x] = acc;
            } else {
                if (acc == (V)0) atomicCAS(a.ctrl + CT_FACTOR, 0, 1 + b0 + (-2 - d.w));
                val[d.x] = (V)1 / acc;
            }
        }
        __syncthreads();
    }
    for (int e = threadIdx.x; e < ne; e += blockDim.x) a.lu[(size_t)blk * a.mx + e] = val[e];
    if (a.fs_val) {
        const int *rp = a.prp + (size_t)blk * (a.brows + 1);
        for (int li = threadIdx.x; li < nb; li += blockDim.x)
            for (int e = rp[li]; e < rp[li + 1]; e++) {
                const int pos = e - rp[li], nlr = a.fs_meta[b0 + li] & 255;
                const int slot = pos < nlr ? pos + 1 : (pos == nlr ? 0 : pos);
                a.fs_val[(size_t)slot * a.n + b0 + li] = val[e];
            }
    }
}

// The operands of one matrix row -- values and NV gathered vectors at the
// row's columns, and the vectors at the row itself -- held in registers.
// The row is read from its ELL slots (padding: column i, value 0), so every
// load is issued at kernel start without waiting for the row's start; the
// entries beyond kEllWidth are read from the CSR arrays where they are used.
template <typename V, int NV>
struct RowOps {
    V a[kEllWidth];
    V x[NV][kEllWidth];
    V own[NV];
    int len = 0;
    template <typename... P>
    __device__ inline void load(const SolvArgs<V> &s, int i, bool valid, P... vec) {
        const V *vs[NV] = {vec...};
        if (!valid) return;
        len = s.ell_len[i];
        int j[kEllWidth];
#pragma unroll
        for (int k = 0; k < kEllWidth; k++) {
            const size_t slot = (size_t)k * s.n + i;
            j[k] = s.ell_col[slot];
            a[k] = s.ell_a[slot];
        }
#pragma unroll
        for (int v = 0; v < NV; v++) own[v] = vs[v][i];
#pragma unroll
        for (int k = 0; k < kEllWidth; k++)
#pragma unroll
            for (int v = 0; v < NV; v++) x[v][k] = vs[v][j[k]];
    }
    // CSR range of the entries beyond the ELL slots (empty for most rows)
    __device__ inline void tail(const SolvArgs<V> &s, int i, int &q0, int &q1) const {
        q0 = q1 = 0;
        if (len > kEllWidth) {
            q1 = s.rowptr[i + 1];
            q0 = q1 - len + kEllWidth;
        }
    }
};

// A matrix row and its factor row for blocks with halo tables, in registers.
// The product's operand is formed once per row of the block and once per row
// of its halo (the neighbour rows in other blocks, some 80 for 256 rows), in
// LDS, instead of by every row for each of its columns (4 vectors gathered at
// 10 columns: k_bicg_a on 300k rows in FP64 52 us against 31, k_bicg_b 23
// against 19; in FP32 on 285k rows 17.4 against 12.3 and 11.9 against 8.2).  Terms
// are added as in RowOps and FacRow, the padding's as zeros, and slots beyond
// those that some row of the wavefront fills are left out.
template <typename V>
struct HaloRow {
    V a[kEllWidth], f[kFacWidth];
    unsigned lc[kEllWidth / 2], fc[kFacWidth / 2];
    int nl = 0, cnt = 0, len = 0;
    bool a8, l3, l6, u3, u6;        // some row of the wavefront fills slots 8.., L or U slots 4.. and 7..
    int h[2], nh;
    __device__ __attribute__((always_inline)) void load(const SolvArgs<V> &s, int blk, int i, bool valid) {
#pragma unroll
        for (int k = 0; k < kEllWidth; k++) a[k] = f[k] = 0;
#pragma unroll
        for (int k = 0; k < kEllWidth / 2; k++) lc[k] = fc[k] = 0;
        nh = s.hcnt[blk];
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int e = threadIdx.x + k * kThreads;
            h[k] = e < s.hmax ? s.hcol[(size_t)blk * s.hmax + e] : 0;
        }
        if (valid) {
            len = s.ell_len[i];
            const int meta = s.fs_meta[i];
            nl = meta & 255;
            cnt = meta >> 8;
#pragma unroll
            for (int k = 0; k < kEllWidth; k++) {
                a[k] = s.ell_a[(size_t)k * s.n + i];
                f[k] = s.fs_val[(size_t)k * s.n + i];
            }
#pragma unroll
            for (int k = 0; k < kEllWidth / 2; k++) {
                lc[k] = s.lcol[(size_t)k * s.n + i];
                fc[k] = s.fcol[(size_t)k * s.n + i];
            }
        }
    }
    __device__ __attribute__((always_inline)) void bounds() {
        a8 = __any(len > 8);
        l3 = __any(nl > 3);
        l6 = __any(nl > 6);
        u3 = __any(cnt > 4);
        u6 = __any(cnt > 7);
    }
    __device__ static __attribute__((always_inline)) V at(const V *base, const unsigned *w, int k) {
        const unsigned o = (k & 1) ? w[k / 2] >> 16 : w[k / 2] & 0xffffu;
        return *reinterpret_cast<const V *>(reinterpret_cast<const char *>(base) + o);
    }
    __device__ __attribute__((always_inline)) V product(const V *X) const {
        V t = 0, g[kEllWidth];
#pragma unroll
        for (int k = 0; k < 8; k++) g[k] = at(X, lc, k);
#pragma unroll
        for (int k = 0; k < 8; k++) t = t + a[k] * g[k];
        if (a8)
#pragma unroll
            for (int k = 8; k < kEllWidth; k++) t = t + a[k] * at(X, lc, k);
        return t;
    }
    // t minus the terms of slots K0 .. K0+2 on the wanted side of the diagonal
    template <int K0, bool UPPER>
    __device__ __attribute__((always_inline)) V three(V t, const V *src) const {
        V g[3];
#pragma unroll
        for (int k = 0; k < 3; k++) g[k] = at(src, fc, K0 + k);
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const bool on = UPPER ? K0 + k > nl && K0 + k < cnt : K0 + k <= nl;
            t = t - (on ? f[K0 + k] : (V)0) * g[k];
        }
        return t;
    }
    // (LU)^-1 of the block applied to t (in y, visible): this row's result
    __device__ __attribute__((always_inline)) V lusol(int sweeps, bool mine, V t, V *y, V *w) const {
        V *src = y, *dst = w, cur = t;
        for (int sw = 1; sw < sweeps; sw++) {
            cur = three<1, false>(t, src);
            if (l3) cur = three<4, false>(cur, src);
            if (l6) cur = three<7, false>(cur, src);
            if (mine) dst[threadIdx.x] = cur;
            __syncthreads();
            V *x = src; src = dst; dst = x;
        }
        const V bl = cur;
        cur = f[0] * bl;
        for (int sw = 1; sw < sweeps; sw++) {
            if (mine) dst[threadIdx.x] = cur;
            __syncthreads();
            V *x = src; src = dst; dst = x;
            cur = three<1, true>(bl, src);
            if (u3) cur = three<4, true>(cur, src);
            if (u6) cur = three<7, true>(cur, src);
            cur = f[0] * cur;
        }
        return cur;
    }
};

// r0 = M^-1 (b - A x0) (x0 = 0 when zero_x0), dx = 0; (r0,r0) into both
// slots of region C
template <typename V, bool STAGE>
__global__ __launch_bounds__(kThreads) void k_bicg_init(SolvArgs<V> a, int zero_x0) {
    if (a.ctrl[CT_REFCONV]) return;
    extern __shared__ double smem[];
    V *y = reinterpret_cast<V *>(smem), *w = y + a.brows;
    const int blk = xcd_block(blockIdx.x, gridDim.x), b0 = blk * a.brows;
    const int nb = min(a.n, b0 + a.brows) - b0;
    BlockStage<V, STAGE> st;
    st.load(a, blk);
    const BlockView<V> B = st.store(a, blk, reinterpret_cast<unsigned char *>(w + a.brows));
    for (int li = threadIdx.x; li < nb; li += blockDim.x) {
        const int i = b0 + li;
        V t = 0;
        if (!zero_x0)
            for (int q = a.rowptr[i]; q < a.rowptr[i + 1]; q++) t = t + a.A[q] * a.x0[a.cols[q]];
        y[li] = a.b[i] - t;
    }
    __syncthreads();
    const V *z = block_lusol(a, B, blk, b0, nb, y, w);
    double loc[2] = {0., 0.};
    for (int li = threadIdx.x; li < nb; li += blockDim.x) {
        const int i = b0 + li;
        const V r = z[li];
        a.r0[i] = r;
        a.dx[i] = 0;
        loc[0] += (double)r * (double)r;
    }
    loc[1] = loc[0];
    store_partials<2>(loc, a.part, PR_C, a.nparts, blk);
    if (blk == 0 && threadIdx.x == 0) {
        a.ctrl[CT_STOPIT] = 0; a.ctrl[CT_CONV] = 0; a.ctrl[CT_FAIL] = 0; a.ctrl[CT_MAXIT] = 0; a.ctrl[CT_NMV] = 1;
    }
}

// Iteration it, first kernel.  For it > 0 it completes iteration it-1 from
// the partial sums of k_bicg_b: omega = (t,s)/(t,t), x += alpha p + omega s,
// r = s - omega t, with |r|^2 = (s,s) - 2 omega (t,s) + omega^2 (t,t) and
// rho = (r0,s) - omega (r0,t); then the stopping test (stopbis), beta, the
// new direction p = r + beta (p - omega v) (neighbour rows formed on the
// fly), v = M^-1 A p and the partial (r0,v).  A stop decided by this kernel
// (convergence, iteration limit) is stamped with it+1 in CT_STOPIT, so that
// its own workgroups still finish the update of x; breakdowns are found by
// every workgroup before any update.  With blocks of at most one row per
// work-item, every load that depends on no other load (control words,
// scalars, the block's factors, the row's operands, the partial sums) is
// issued before the first test.
template <typename V, int MODE>
__global__ __launch_bounds__(kThreads) void k_bicg_a(SolvArgs<V> a, int it) {
    constexpr bool STAGE = MODE == 1;      // block factors staged in LDS (0: read from global memory)
    extern __shared__ double smem[];
    V *y = reinterpret_cast<V *>(smem), *w = y + a.brows;
    const int par = it & 1, pp = par ^ 1;
    const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
    const int blk = xcd_block(blockIdx.x, gridDim.x), b0 = blk * a.brows;
    const int nb = min(a.n, b0 + a.brows) - b0;
    const V *pold = pp ? a.p1 : a.p0;     // direction of iteration it-1 (it = 0: unused)
    const V *vold = pp ? a.v1 : a.v0;
    V *pnew = par ? a.p1 : a.p0;
    V *vnew = par ? a.v1 : a.v0;
    const bool pre = a.brows <= kThreads;
    const int i = b0 + threadIdx.x;
    const bool mine = pre && (int)threadIdx.x < nb;
    const int nq = it == 0 ? 2 : 5, region = it == 0 ? PR_C : PR_B;
    // independent loads first
    const int stop = a.ctrl[CT_STOPIT], fail = a.ctrl[CT_FAIL], refconv = a.ctrl[CT_REFCONV];
    const double alpha_prev = a.scal[SC_ALPHA + pp], target_prev = a.scal[SC_TARGET], rho_prev = a.scal[SC_RHO + pp];
    constexpr bool regs = MODE == 2;       // factor rows in registers, no block staging
    constexpr bool halo = MODE == 3;       // the same with the block's halo
    BlockStage<V, STAGE> st;
    FacRow<V> fr;
    HaloRow<V> hr;
    V hs[2] = {}, ht[2] = {}, hp[2] = {}, hv[2] = {};
    if constexpr (halo) hr.load(a, blk, i, mine);
    else if constexpr (regs) fr.load(a, i, mine);
    else st.load(a, blk);
    Partials<5> ps;
    ps.load(a.part, region, a.nparts, a.nblk, nq);
    RowOps<V, 4> ro;
    V r0_i = 0, dx_i = 0;
    if constexpr (halo) {
        const V *first = it == 0 ? a.r0 : a.s;
        if (mine) {
            r0_i = a.r0[i];
            ro.own[0] = first[i];
            if (it > 0) {
                ro.own[1] = a.t[i]; ro.own[2] = pold[i]; ro.own[3] = vold[i];
                dx_i = a.dx[i];
            }
        }
#pragma unroll
        for (int k = 0; k < 2; k++)
            if ((int)threadIdx.x + k * kThreads < hr.nh) {
                hs[k] = first[hr.h[k]];
                if (it > 0) { ht[k] = a.t[hr.h[k]]; hp[k] = pold[hr.h[k]]; hv[k] = vold[hr.h[k]]; }
            }
    } else if (pre) {
        if (it == 0) ro.load(a, i, mine, a.r0, a.r0, a.r0, a.r0);
        else ro.load(a, i, mine, a.s, a.t, pold, vold);
        if (mine) {
            r0_i = a.r0[i];
            if (it > 0) dx_i = a.dx[i];
        }
    }
    if (fail || refconv || (stop != 0 && stop <= it)) return;
    const BlockView<V> B = regs || halo ? BlockView<V>{}
                                        : st.store(a, blk, reinterpret_cast<unsigned char *>(w + a.brows));
    double q[5];   // it = 0: (r0,r0) (r0,r0); else (t,t) (t,s) (s,s) (r0,s) (r0,t)
    ps.total(a.part, region, a.nparts, a.nblk, nq, q);
    double rn, rho, omega = 0., alpha = 0.;
    if (it == 0) {
        rn = sqrt(q[0]);
        rho = q[1];
    } else {
        if (breakdown(q[0])) {
            if (lead) a.ctrl[CT_FAIL] = -3;
            return;
        }
        omega = q[1] / q[0];
        if (breakdown(omega)) {
            if (lead) a.ctrl[CT_FAIL] = -3;
            return;
        }
        alpha = alpha_prev;
        rn = sqrt(fmax(0., q[2] - 2. * omega * q[1] + omega * omega * q[0]));
        rho = q[3] - omega * q[4];
        const V va = (V)alpha, vo = (V)omega;
        if (pre) {
            if (mine) {
                a.dx[i] = dx_i + (va * ro.own[2] + vo * ro.own[0]);
                a.r[i] = ro.own[0] - vo * ro.own[1];
            }
        } else {
            for (int li = threadIdx.x; li < nb; li += blockDim.x) {
                const int k = b0 + li;
                a.dx[k] = a.dx[k] + (va * pold[k] + vo * a.s[k]);
                a.r[k] = a.s[k] - vo * a.t[k];
            }
        }
        if (lead) { a.scal[SC_OMEGA + pp] = omega; a.ctrl[CT_ITS] += 1; }
    }
    double target;
    if (it == 0) {
        target = a.rtol * rn + a.atol;
        if (lead) { a.scal[SC_TARGET] = target; a.scal[SC_NORM0] = rn; }
    } else {
        target = target_prev;
    }
    if (lead) { a.scal[SC_RNORM] = rn; a.ctrl[CT_NMV] = 1 + 2 * it; }
    if (!(rn > target)) {
        if (lead) { a.ctrl[CT_STOPIT] = it + 1; a.ctrl[CT_CONV] = 1; }
        return;
    }
    if (it > 0 && a.itermax > 0 && 1 + 2 * it >= a.itermax) {
        if (lead) { a.ctrl[CT_STOPIT] = it + 1; a.ctrl[CT_MAXIT] = 1; }
        return;
    }
    double beta = 0.;
    if (it > 0) {
        if (breakdown(rho)) {
            if (lead) a.ctrl[CT_FAIL] = -3;
            return;
        }
        beta = rho * alpha / (omega * rho_prev);
    }
    if (lead) a.scal[SC_RHO + par] = rho;
    const V vb = (V)beta, vo = (V)omega;
    V z_i = 0;
    if constexpr (halo) {
        V *X = w + a.brows, p = ro.own[0];
        if (it > 0) p = (ro.own[0] - vo * ro.own[1]) + vb * (ro.own[2] - vo * ro.own[3]);
        if (mine) {
            X[threadIdx.x] = p;
            pnew[i] = p;
        }
#pragma unroll
        for (int k = 0; k < 2; k++)
            if ((int)threadIdx.x + k * kThreads < hr.nh)
                X[a.brows + threadIdx.x + k * kThreads] =
                    it == 0 ? hs[k] : (hs[k] - vo * ht[k]) + vb * (hp[k] - vo * hv[k]);
        hr.bounds();
        __syncthreads();
        const V t = hr.product(X);
        if (mine) y[threadIdx.x] = t;
        __syncthreads();
        z_i = hr.lusol(a.sweeps, mine, t, y, w);
    } else if (pre) {
        if (mine) {
            V t = 0;
            int q0, q1;
            ro.tail(a, i, q0, q1);
            if (it == 0) {
#pragma unroll
                for (int k = 0; k < kEllWidth; k++)
                    if (k < ro.len) t = t + ro.a[k] * ro.x[0][k];
                for (int q = q0; q < q1; q++) t = t + a.A[q] * a.r0[a.cols[q]];
                pnew[i] = ro.own[0];
            } else {
#pragma unroll
                for (int k = 0; k < kEllWidth; k++) {
                    if (k < ro.len) {
                        const V rj = ro.x[0][k] - vo * ro.x[1][k];
                        const V pj = rj + vb * (ro.x[2][k] - vo * ro.x[3][k]);
                        t = t + ro.a[k] * pj;
                    }
                }
                for (int q = q0; q < q1; q++) {
                    const int j = a.cols[q];
                    const V rj = a.s[j] - vo * a.t[j];
                    const V pj = rj + vb * (pold[j] - vo * vold[j]);
                    t = t + a.A[q] * pj;
                }
                const V ri = ro.own[0] - vo * ro.own[1];
                pnew[i] = ri + vb * (ro.own[2] - vo * ro.own[3]);
            }
            y[threadIdx.x] = t;
        }
    } else if (it == 0) {
        for (int li = threadIdx.x; li < nb; li += blockDim.x) {
            const int k = b0 + li;
            V t = 0;
            for (int q = a.rowptr[k]; q < a.rowptr[k + 1]; q++) t = t + a.A[q] * a.r0[a.cols[q]];
            y[li] = t;
            pnew[k] = a.r0[k];
        }
    } else {
        for (int li = threadIdx.x; li < nb; li += blockDim.x) {
            const int k = b0 + li;
            V t = 0;
            for (int q = a.rowptr[k]; q < a.rowptr[k + 1]; q++) {
                const int j = a.cols[q];
                const V rj = a.s[j] - vo * a.t[j];
                const V pj = rj + vb * (pold[j] - vo * vold[j]);
                t = t + a.A[q] * pj;
            }
            y[li] = t;
            const V ri = a.s[k] - vo * a.t[k];
            pnew[k] = ri + vb * (pold[k] - vo * vold[k]);
        }
    }
    const V *z = nullptr;
    if constexpr (!halo) {
        __syncthreads();
        z = regs ? fr.lusol(a.sweeps, mine, threadIdx.x, y, w) : block_lusol(a, B, blk, b0, nb, y, w);
    }
    double loc[1] = {0.};
    if constexpr (halo) {
        if (mine) {
            vnew[i] = z_i;
            loc[0] = (double)r0_i * (double)z_i;
        }
    } else if (pre) {
        if (mine) {
            vnew[i] = z[threadIdx.x];
            loc[0] = (double)r0_i * (double)z[threadIdx.x];
        }
    } else {
        for (int li = threadIdx.x; li < nb; li += blockDim.x) {
            const int k = b0 + li;
            vnew[k] = z[li];
            loc[0] += (double)a.r0[k] * (double)z[li];
        }
    }
    store_partials<1>(loc, a.part, PR_A, a.nparts, blk);
}

// Iteration it, second kernel: alpha = rho / (r0,v); s = r - alpha v
// (fused); t = M^-1 A s; partials (t,t) (t,s) (s,s) (r0,s) (r0,t).
// Independent loads are issued first, as in k_bicg_a.
template <typename V, int MODE>
__global__ __launch_bounds__(kThreads) void k_bicg_b(SolvArgs<V> a, int it) {
    constexpr bool STAGE = MODE == 1;      // block factors staged in LDS (0: read from global memory)
    extern __shared__ double smem[];
    V *y = reinterpret_cast<V *>(smem), *w = y + a.brows;
    const int par = it & 1;
    const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
    const V *vnew = par ? a.v1 : a.v0;
    const V *rv = it == 0 ? a.r0 : a.r;
    const int blk = xcd_block(blockIdx.x, gridDim.x), b0 = blk * a.brows;
    const int nb = min(a.n, b0 + a.brows) - b0;
    const bool pre = a.brows <= kThreads;
    const int i = b0 + threadIdx.x;
    const bool mine = pre && (int)threadIdx.x < nb;
    const int stop = a.ctrl[CT_STOPIT], fail = a.ctrl[CT_FAIL], refconv = a.ctrl[CT_REFCONV];
    const double rho = a.scal[SC_RHO + par];
    constexpr bool regs = MODE == 2, halo = MODE == 3;
    BlockStage<V, STAGE> st;
    FacRow<V> fr;
    HaloRow<V> hr;
    V hs[2] = {}, hv[2] = {};
    if constexpr (halo) hr.load(a, blk, i, mine);
    else if constexpr (regs) fr.load(a, i, mine);
    else st.load(a, blk);
    Partials<1> ps;
    ps.load(a.part, PR_A, a.nparts, a.nblk, 1);
    RowOps<V, 2> ro;
    V r0_i = 0;
    if constexpr (halo) {
        if (mine) {
            r0_i = a.r0[i];
            ro.own[0] = rv[i];
            ro.own[1] = vnew[i];
        }
#pragma unroll
        for (int k = 0; k < 2; k++)
            if ((int)threadIdx.x + k * kThreads < hr.nh) {
                hs[k] = rv[hr.h[k]];
                hv[k] = vnew[hr.h[k]];
            }
    } else if (pre) {
        ro.load(a, i, mine, rv, vnew);
        if (mine) r0_i = a.r0[i];
    }
    if (stop || fail || refconv) return;
    const BlockView<V> B = regs || halo ? BlockView<V>{}
                                        : st.store(a, blk, reinterpret_cast<unsigned char *>(w + a.brows));
    double d[1];
    ps.total(a.part, PR_A, a.nparts, a.nblk, 1, d);
    if (breakdown(d[0])) {
        if (lead) a.ctrl[CT_FAIL] = -3;
        return;
    }
    const double alpha = rho / d[0];
    if (lead) a.scal[SC_ALPHA + par] = alpha;
    const V va = (V)alpha;
    V s_i = 0, z_i = 0;
    if constexpr (halo) {
        V *X = w + a.brows;
        s_i = ro.own[0] - va * ro.own[1];
        if (mine) {
            X[threadIdx.x] = s_i;
            a.s[i] = s_i;
        }
#pragma unroll
        for (int k = 0; k < 2; k++)
            if ((int)threadIdx.x + k * kThreads < hr.nh) X[a.brows + threadIdx.x + k * kThreads] = hs[k] - va * hv[k];
        hr.bounds();
        __syncthreads();
        const V t = hr.product(X);
        if (mine) y[threadIdx.x] = t;
        __syncthreads();
        z_i = hr.lusol(a.sweeps, mine, t, y, w);
    } else if (pre) {
        if (mine) {
            V t = 0;
            int q0, q1;
            ro.tail(a, i, q0, q1);
#pragma unroll
            for (int k = 0; k < kEllWidth; k++)
                if (k < ro.len) t = t + ro.a[k] * (ro.x[0][k] - va * ro.x[1][k]);
            for (int q = q0; q < q1; q++) {
                const int j = a.cols[q];
                t = t + a.A[q] * (rv[j] - va * vnew[j]);
            }
            y[threadIdx.x] = t;
            s_i = ro.own[0] - va * ro.own[1];
            a.s[i] = s_i;
        }
    } else {
        for (int li = threadIdx.x; li < nb; li += blockDim.x) {
            const int k = b0 + li;
            V t = 0;
            for (int q = a.rowptr[k]; q < a.rowptr[k + 1]; q++) {
                const int j = a.cols[q];
                const V sj = rv[j] - va * vnew[j];
                t = t + a.A[q] * sj;
            }
            y[li] = t;
            a.s[k] = rv[k] - va * vnew[k];
        }
    }
    const V *z = nullptr;
    if constexpr (!halo) {
        __syncthreads();
        z = regs ? fr.lusol(a.sweeps, mine, threadIdx.x, y, w) : block_lusol(a, B, blk, b0, nb, y, w);
        if (pre && mine) z_i = z[threadIdx.x];
    }
    double loc[5] = {0., 0., 0., 0., 0.};
    if (halo || pre) {
        if (mine) {
            const double tv = (double)z_i, sv = (double)s_i, r0 = (double)r0_i;
            a.t[i] = z_i;
            loc[0] = tv * tv;
            loc[1] = tv * sv;
            loc[2] = sv * sv;
            loc[3] = r0 * sv;
            loc[4] = r0 * tv;
        }
    } else {
        for (int li = threadIdx.x; li < nb; li += blockDim.x) {
            const int k = b0 + li;
            const double tv = (double)z[li], sv = (double)a.s[k], r0 = (double)a.r0[k];
            a.t[k] = z[li];
            loc[0] += tv * tv;
            loc[1] += tv * sv;
            loc[2] += sv * sv;
            loc[3] += r0 * sv;
            loc[4] += r0 * tv;
        }
    }
    store_partials<5>(loc, a.part, PR_B, a.nparts, blk);
}

// x = x0 + dx (tidycg) into the FP64 solution; with add, x += dx unless the
// refinement has converged
template <typename V>
__global__ void k_bicg_finish(const V *x0, const V *dx, double *x, int n, int add, const int *ctrl) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || (add && ctrl[CT_REFCONV]) || (!add && !ctrl[CT_CONV])) return;
    if (add) x[i] = x[i] + (double)dx[i];
    else x[i] = (double)(x0[i] + dx[i]);
}

// the solve's copies of the assembled matrix: values in the ELL slots of
// the iteration kernels (precision V), and for the FP32 path the FP32 CSR
template <typename V>
__global__ void k_prep_matrix(const double *aval, const int *csr_ell, V *ell_a, float *a32, int nnz) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nnz) return;
    const double v = aval[q];
    if (a32) a32[q] = (float)v;
    const int slot = csr_ell[q];
    if (slot >= 0) ell_a[slot] = (V)v;
}

// initial guess x = zn; clears the factorisation flag of this solve
template <typename S>
__global__ void k_guess(const S *zn, double *x, int n, int *ctrl) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) { ctrl[CT_FACTOR] = 0; ctrl[CT_ITS] = 0; ctrl[CT_NREF] = 0; ctrl[CT_REFCONV] = 0; }
    if (i < n) x[i] = (double)zn[i];
}

// FP32 path: initial guess extrapolated linearly in time from the levels at
// the start of this step (zn) and of the previous one (zprev), x = 2 zn -
// zprev (zn alone without a history); zprev <- zn.  The refinement's target
// is absolute (a fraction of |b|), so a closer start saves rounds; the
// solution it converges to does not depend on the start.
__global__ void k_guess_extrap(const float *zn, float *zprev, double *x, int n, int *ctrl, int have_prev) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) { ctrl[CT_FACTOR] = 0; ctrl[CT_ITS] = 0; ctrl[CT_NREF] = 0; ctrl[CT_REFCONV] = 0; }
    if (i >= n) return;
    const double z = (double)zn[i];
    x[i] = have_prev ? 2. * z - (double)zprev[i] : z;
    zprev[i] = zn[i];
}

// FP64 residual r64 = b - A x with partial |r64|^2 and |b|^2 (refinement)
__global__ __launch_bounds__(kThreads) void k_resid64(const int *rowptr, const int *cols, const double *A,
                                                       const double *b, const double *x, double *r64, float *r32,
                                                       int n, double *part, int nparts, const int *ctrl) {
    if (ctrl[CT_REFCONV]) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    double loc[2] = {0., 0.};
    if (i < n) {
        double t = 0.;
        for (int q = rowptr[i]; q < rowptr[i + 1]; q++) t = t + A[q] * x[cols[q]];
        const double r = b[i] - t;
        r64[i] = r;
        r32[i] = (float)r;
        loc[0] = r * r;
        loc[1] = b[i] * b[i];
    }
    store_partials<2>(loc, part, PR_R, nparts, blockIdx.x);
}

__global__ __launch_bounds__(kThreads) void k_resid_check(const double *part, int nparts, int n, double *scal,
                                                           int *ctrl, double tol) {
    if (ctrl[CT_REFCONV]) return;
    double rs[2];
    sum_partials<2>(part, PR_R, nparts, n, rs);
    if (threadIdx.x == 0) {
        // iterations of the inner solve just finished (round nref - 1),
        // negative when it stopped without converging (cut short)
        const int r = ctrl[CT_NREF];
        if (r >= 1 && r <= CT_NRITS) {
            const int its = (ctrl[CT_NMV] - 1) / 2;
            ctrl[CT_RITS + r - 1] = ctrl[CT_CONV] ? its : -its;
        }
        scal[SC_RES64] = sqrt(rs[0]);
        scal[SC_BNORM] = sqrt(rs[1]);
        const int conv = (sqrt(rs[0]) <= tol * sqrt(rs[1])) ? 1 : 0;
        ctrl[CT_REFCONV] = conv;
        if (!conv) ctrl[CT_NREF] += 1;
    }
}

// ---------------------------------------------------------------- one-launch solve
// The whole Krylov solve (and on the FP32 path the refinement around it) in
// one launch, one workgroup per diagonal block, one row per work-item: the
// row's matrix and factor entries and its vector elements stay in registers
// for the solve, and the workgroups exchange what the next half iteration
// needs through memory instead of ending the kernel.
//
// What bounds it: the chain of a half iteration -- product, triangular
// sweeps, one exchange -- not bytes (8 MB per product on 50k rows).  As two
// kernels per iteration the same chain also paid a kernel boundary and two
// rounds of loads of the matrix, factors and vectors every time: 16.4 us per
// FP64 iteration on the 50k-node lagoon (196 blocks), 9.7 us as one launch;
// a hydro step there 0.60 -> 0.37 ms, on 3k nodes 0.35 -> 0.21 ms, FP32 on
// 60k nodes 0.61 -> 0.40 ms.  Of the clocks of a half iteration (4.9 us) on
// 50k rows, 98 workgroups of 512, in all 11,400: 3,400 waiting for the slots,
// 4,100 in the rest of the exchange (sums, puts, barriers), 2,900 in the
// product and 3 sweeps; on 20k rows, 79 of 256, 9,600: 3,000, 3,200 and
// 2,200; on 3k rows, 12 of 256, 8,400: 2,000, 3,100 and 2,200.
//
// Exchange.  Each half iteration has an epoch.  A workgroup puts its partial
// sums into its own slots, and the elements of v (or t) that rows of other
// blocks multiply into theirs; the readers wait until a slot holds a value.
// Every slot is one machine word, written and read by relaxed agent-scope
// atomics (they go through to memory that all XCDs see), and an empty slot
// holds a NaN pattern that no put ever writes, so a word is its own flag and
// an exchange is one store and one load latency long.  Slots rotate over
// four buffers: at epoch e a workgroup has every partial of epoch e-1, so
// every workgroup has finished reading epoch e-2, and it empties its own
// slots of that buffer (next used at e+2), with the stores complete before
// it puts its partials of epoch e.  The factorisation kernel of each solve
// empties all slots.
//
// A block's neighbour rows in other blocks (its halo) are kept as well: the
// recurrences of p, r, s (and the correction) are run on them redundantly,
// with the same operations, so only v and t are exchanged and the halo
// values have the owner's bits.  The partial sums are those of the diagonal blocks
// and every workgroup adds them in the order of the two-kernel iteration, so
// all of them (and all runs) take the same decisions and the FP64 solve of
// blocks of 256 rows has that iteration's bits.
//
// The waits are bounded: the launch is made only when all its workgroups
// can be resident together (zeta_slots), and a wait that still runs out sets
// CT_WAIT and ends the workgroup.  Every other workgroup then runs out of
// its own wait, and the host makes the solve with the two-kernel iteration,
// and the next ones too (zeta_expired).
// The result counts only once every workgroup has written its part of it:
// each puts one more partial after its stores, and the workgroup that sets
// the convergence flags collects them first.
constexpr int kWaitExpired = -9;
constexpr int kSpinLimit = 1 << 17;      // polls of one wait (about 0.1 s), unless the model sets its own
constexpr int kZetaBufs = 4;
// Partial sums per diagonal block and buffer, and their copies: every
// workgroup reads all of them, so one copy makes all workgroups wait for the
// same few memory lines (196 workgroups: a half iteration of 5.8 us with one
// copy, 5.3 us with 16); each workgroup puts its sums into every copy and
// reads one.  Copies lie apart.
constexpr int kPartSlots = 5;
constexpr int kPartCopies = 16;
constexpr int kPartStride = 512 * 5;     // words per copy: [kPartSlots][512 blocks]

template <typename V>
struct Slot;
template <>
struct Slot<double> {
    using U = unsigned long long;
    static constexpr U empty = 0x7ff8a5a55a5a0001ull, nan = 0x7ff8000000000000ull;
};
template <>
struct Slot<float> {
    using U = unsigned;
    static constexpr U empty = 0x7fc0a5a5u, nan = 0x7fc00000u;
};
template <typename V>
__device__ inline void slot_put(typename Slot<V>::U *p, V v) {
    using U = typename Slot<V>::U;
    __hip_atomic_store(p, v == v ? __builtin_bit_cast(U, v) : Slot<V>::nan, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
template <typename U>
__device__ inline void slot_clear(U *p, U empty) {
    __hip_atomic_store(p, empty, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename U>
__device__ inline U slot_get(const U *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ inline unsigned long long *part_slot(unsigned long long *pslot, int buf, int copy, int k, int blk) {
    return pslot + ((size_t)buf * kPartCopies + copy) * kPartStride + k * 512 + blk;
}

// the slots of block blk empty in every buffer, and the solve's flags clear
template <typename V>
__device__ inline void zeta_empty_slots(const SolvArgs<V> &a, int blk, int b0, int nb) {
    auto *xch = (typename Slot<V>::U *)a.xch;
    for (int b = 0; b < kZetaBufs; b++) {
        for (int li = threadIdx.x; li < nb; li += blockDim.x)
            if (const int q = a.send[b0 + li]; q >= 0) slot_clear(xch + (size_t)b * a.nsend + q, Slot<V>::empty);
        if (threadIdx.x < kPartSlots * kPartCopies)
            slot_clear(part_slot(a.pslot, b, threadIdx.x % kPartCopies, threadIdx.x / kPartCopies, blk),
                       Slot<double>::empty);
    }
    if (blk == 0 && threadIdx.x == 0) {
        a.ctrl[CT_CONV] = 0; a.ctrl[CT_FAIL] = 0; a.ctrl[CT_MAXIT] = 0; a.ctrl[CT_WAIT] = 0;
    }
}

// the partial-sum slots of all workgroups empty (dense rows: more workgroups
// than blocks, too many slots for the few workgroups of the factorisation);
// one buffer's copy and sum per workgroup
__global__ __launch_bounds__(kThreads) void k_empty_partials(unsigned long long *pslot, int nsum) {
    const int b = blockIdx.x;
    unsigned long long *p = part_slot(pslot, b / (kPartCopies * kPartSlots), b / kPartSlots % kPartCopies,
                                      b % kPartSlots, 0);
    for (int i = threadIdx.x; i < nsum; i += kThreads) slot_clear(p + i, Slot<double>::empty);
}

// every store this work-item has issued is complete
__device__ __attribute__((always_inline)) inline void wait_stores() {
    __builtin_amdgcn_s_waitcnt(0x0F70);      // vmcnt(0)
}

struct ZetaArgs {
    int nwg, group;                      // workgroups, diagonal blocks of each
    int hmax;                            // halo stride per workgroup
    const unsigned *lcol;                // byte offsets of the row's columns, two per word [k/2][n]
    const int *hcol, *hslot, *hcnt;      // halo rows and their slots [wg*hmax + h], their number
    const int *send;                     // slot of a row in other workgroups' halos, or -1
    int nsend;                           // value slots per buffer
    // exact substitution: rows in its order, their chunks (stride per block)
    const int *rows_f, *rows_b;
    const unsigned *chunk_f, *chunk_b;
    const int *nch_f, *nch_b;
    int chmax;
    // dense rows of the block inverses: workgroups per block; the transposed
    // factors' entries (value's place | row << 16) in the order of rows_f and
    // rows_b [blk*dmax + e] and their starts by position [blk*(brows+1) + t]
    int members, dmax;
    const unsigned *dent_f, *dent_b;
    const int *dptr_f, *dptr_b;
    void *xch;                           // value slots [buf][nsend]
    unsigned long long *pslot;           // partial-sum slots [buf][kPartCopies][kPartStride]
    // FP32 path: the FP64 system and its refinement
    const double *rhs;
    double *x;
    double tol;
    int maxref;
    int maxit;                           // iterations of a Krylov solve (krylov_cap)
    int spins;                           // polls of one wait
};

// Exact substitution with one triangular factor of a block by one wavefront
// (wavefront g of the workgroup takes its block g): rows level by level (a level's rows depend only on earlier
// levels), up to 64 rows of a level at a time, one lane per row.  One
// wavefront needs no barrier between levels (its LDS accesses run in
// order).  The rows lie in LDS in the order of the substitution, their first
// kSubFirst entries slot-major with zero padding, so the next chunk's
// entries are read, at fixed offsets from one address, while the current
// chunk waits for its operands: a chunk costs one LDS gather and its chain of
// subtractions.  What bounds it is that chain times the number of levels
// (62 levels each way on the 41x21 basin: with a barrier of the workgroup
// per level and the factors in global memory a solve of 20 iterations took
// 3.7 ms, with the factors read in the list order by one wavefront 1.26 ms,
// in this layout 0.95 ms).
// A row's word: byte offset of its value | further entries << 16 (these few
// rows take them from the block's entry list).
constexpr int kSubFirst = 4;

template <typename V, int ROWS>
struct SubExact {
    const V *val, *piv;                  // [kSubFirst][ROWS], inverted pivots [ROWS]
    const unsigned *col;                 // byte offsets [kSubFirst / 2][ROWS], two per word
    const unsigned *row, *tail;          // the rows' words and first further entries [ROWS]
    const unsigned *chunk;               // first row | rows << 16 of each chunk of the block
    const V *lu;                         // the block's entries and local columns (global memory)
    const int *pcol;
    int nch, r0;                         // chunks and first row of the block

    template <bool BACK>
    __device__ __attribute__((always_inline)) inline void run(V *y) const {
        const int lane = threadIdx.x & 63;
        char *yb = reinterpret_cast<char *>(y);
        auto at = [&](unsigned o) __attribute__((always_inline)) -> V & { return *reinterpret_cast<V *>(yb + o); };
        V v[kSubFirst], p = 0, rhs;
        unsigned c[kSubFirst / 2], r, r1;
        unsigned w = chunk[0], w1 = chunk[1], w2 = chunk[2];      // (padded)
        // (lanes beyond a chunk's rows read some row and write nothing)
        auto pos = [&](unsigned c0) __attribute__((always_inline)) { return min(r0 + (int)(c0 & 0xffffu) + lane, ROWS - 1); };
        int t = pos(w), t1 = pos(w1);
        r = row[t];
        r1 = row[t1];
        auto entries = [&](int tt) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < kSubFirst; k++) v[k] = val[k * ROWS + tt];
#pragma unroll
            for (int k = 0; k < kSubFirst / 2; k++) c[k] = col[k * ROWS + tt];
            if (BACK) p = piv[tt];
        };
        entries(t);
        rhs = at(r & 0xffffu);
        for (int ch = 0; ch < nch; ch++) {
            V g[kSubFirst], vc[kSubFirst];
#pragma unroll
            for (int k = 0; k < kSubFirst; k++) {
                g[k] = at((k & 1) ? c[k / 2] >> 16 : c[k / 2] & 0xffffu);
                vc[k] = v[k];
            }
            V acc = rhs;
            const V pc = p;
            const unsigned rc = r;
            const int tc = t;
            const bool on = lane < (int)(w >> 16);
            // ahead: the next chunk's entries, the one after's row word
            w = w1; w1 = w2; w2 = chunk[ch + 3];
            t = t1; r = r1;
            entries(t);
            rhs = at(r & 0xffffu);
            t1 = pos(w1);
            r1 = row[t1];
#pragma unroll
            for (int k = 0; k < kSubFirst; k++) acc = acc - vc[k] * g[k];
            const int more = on ? (int)(rc >> 16) : 0;
            if (__any(more)) {
                const int q = (int)tail[tc];
                for (int k = 0; k < more; k++) acc = acc - lu[q + k] * y[r0 + pcol[q + k]];
            }
            if (on) at(rc & 0xffffu) = BACK ? pc * acc : acc;
        }
    }
};

// Triangular solves of the one-launch kernel: Jacobi sweeps with the factor
// row in registers, exact substitution, or exact by dense rows of the blocks'
// inverses.  The last: substitution is a chain of up to 80 levels each way
// (23 us per half iteration on 861 rows, 46 us on 256-row blocks of an 80 x 40
// basin), so where the device has room each block is given to several
// workgroups; each computes kOwn rows of the block's (LU)^-1 once per solve,
// keeps them in registers, and applies them to the block's whole right-hand
// side, which it forms itself (the vectors of all the block's rows are kept
// by each of its workgroups, the rows applied elsewhere come with the halo).
// A step of the 41 x 21 basin (861 rows, one block) 1.09 -> 0.56 ms, of an 80
// x 40 basin 2.38 -> 0.48 ms, FP64, against the substitution.  The rows are
// computed in 20 to 30 us; of the 18,200 clocks of a half iteration on 861
// rows 7,800 are the product (the matrix row read from cache) and the dense
// rows, 6,200 the exchange outside its wait, 2,300 the wait.
enum { kSwept = 0, kSubst = 1, kDense = 2 };
template <int T>
struct DenseShape {                      // 512: blocks of up to 256 rows; 1024: of up to 1024
    static constexpr int kOwn = T == 512 ? 64 : 12;           // rows per workgroup (what LDS holds at set-up)
    static constexpr int kRows = T == 512 ? 8 : 1;            // per wavefront
    static constexpr int kLanes = 64 / kRows;                 // lanes per row
    static constexpr int kCols = (T == 512 ? 256 : 1024) / kLanes;   // columns per lane
    static constexpr bool kRegs = T == 512;                   // rows in registers, else in LDS
};

// One row of the solve and its block's halo entries, in registers (1024
// work-items have half the registers of 256 each: they read the matrix row
// from cache in every product instead of spilling).  The entries of a row
// are padded with zeros at the row's own column, so that all operands are
// read at once and the terms added without a test per entry (a test each
// made every entry wait for its own LDS read: 2.8 us of product and sweeps
// per half iteration on 256 rows, 1.6 us without); the last slots, which few rows
// fill, are taken only by the wavefronts that hold such a row.
constexpr int kRowFirst = 8;             // matrix entries always taken
constexpr int kTriWidth = kFacWidth - 1; // entries of a row on one side of the diagonal
constexpr int kTriFirst = 6;             // of these always taken

template <typename V, int T, int KH, int MODE>
struct ZetaRow {
    using U = typename Slot<V>::U;
    static constexpr bool kHold = T <= 512;
    static constexpr int kTri = MODE == kSwept ? kTriWidth : 1, kTriWords = (kTri + 1) / 2;
    using D = DenseShape<T>;
    // matrix row; (sweeps) factor row: L and U entries, inverted pivot
    V a[kHold ? kEllWidth : 1], l[kTri], u[kTri], dinv = 0;
    unsigned lc[kHold ? kEllWidth / 2 : 1], llc[kTriWords], uc[kTriWords];
    const V *ga;
    const unsigned *glc;
    bool more_a = false, more_l = false, more_u = false;   // some row of the wavefront fills the last slots
    int i, wg, nh, nsum, n, sweeps, send, nsend;   // nsum: partial sums of all workgroups
    bool mine;
    int hslot[KH];
    // LDS: operand (rows, then halo), two row buffers; exact: block factors
    V *X, *y, *w;
    SubExact<V, T> sf, sb;
    // dense: this lane's part of its row of the block inverse, and the rows
    // of the block that this workgroup applies
    V pinv[MODE == kDense && D::kRegs ? D::kCols : 1];
    const V *plds;
    int own0 = 0, nown = 0;
    bool own;                                // this work-item's row is one of them (else: every row)
    int rows, group;
    U *xch;
    unsigned long long *pslot;
    int epoch = 0, spins;
    int *dead;

    // byte offset k of the offsets packed two per word
    __device__ static __attribute__((always_inline)) inline unsigned off(const unsigned *words, int k) {
        return (k & 1) ? words[k / 2] >> 16 : words[k / 2] & 0xffffu;
    }
    __device__ static __attribute__((always_inline)) inline V at(const V *base, unsigned o) {
        return *reinterpret_cast<const V *>(reinterpret_cast<const char *>(base) + o);
    }
    // t + SIGN * (terms K0 .. K1-1 of the row v, c), in order
    template <int K0, int K1, int SIGN>
    __device__ static __attribute__((always_inline)) inline V terms(V t, const V *v, const unsigned *c, const V *x) {
        V g[K1 - K0];
#pragma unroll
        for (int k = K0; k < K1; k++) g[k - K0] = at(x, off(c, k));
#pragma unroll
        for (int k = K0; k < K1; k++) t = SIGN > 0 ? t + v[k] * g[k - K0] : t - v[k] * g[k - K0];
        return t;
    }
    // operand of the product: this row's element and its halo entries
    __device__ __attribute__((always_inline)) inline void operand(V own, const V (&h)[KH]) {
        if (mine) X[threadIdx.x] = own;
#pragma unroll
        for (int k = 0; k < KH; k++)
            if ((int)threadIdx.x + k * T < nh) X[rows + threadIdx.x + k * T] = h[k];
    }
    // A X of this row, terms in column order
    __device__ __attribute__((always_inline)) inline V product() {
        V t = 0;
        if constexpr (kHold) {
            __syncthreads();
            t = terms<0, kRowFirst, 1>(t, a, lc, X);
            if (more_a) t = terms<kRowFirst, kEllWidth, 1>(t, a, lc, X);
        } else {
            V av[kEllWidth];
            unsigned cv[kEllWidth / 2];
#pragma unroll
            for (int k = 0; k < kEllWidth; k++) av[k] = mine ? ga[(size_t)k * n + i] : (V)0;
            columns(cv);
            __syncthreads();
            t = terms<0, kRowFirst, 1>(t, av, cv, X);
            if (more_a) t = terms<kRowFirst, kEllWidth, 1>(t, av, cv, X);
        }
        return t;
    }
    __device__ __attribute__((always_inline)) inline void columns(unsigned (&cv)[kEllWidth / 2]) const {
#pragma unroll
        for (int k = 0; k < kEllWidth / 2; k++) {
            if constexpr (kHold) cv[k] = lc[k];
            else cv[k] = mine ? glc[(size_t)k * n + i] : 0u;
        }
    }
    // (LU)^-1 of the block applied to the rows' values t: this row's result
    // (the operations of FacRow::lusol and block_lusol)
    __device__ __attribute__((always_inline)) inline V precond(V t) {
        if (mine) y[threadIdx.x] = t;
        __syncthreads();
        if constexpr (MODE == kDense) {
            // row w * kRows + lane / kLanes: the lanes of a row take every
            // kLanes-th column
            const int lane = threadIdx.x & 63, part = lane % D::kLanes;
            V acc = 0;
            if constexpr (D::kRegs) {
#pragma unroll
                for (int j = 0; j < D::kCols; j++) acc = acc + pinv[j] * y[part + D::kLanes * j];
            } else if ((threadIdx.x >> 6) < D::kOwn) {
                const V *p = plds + (size_t)(threadIdx.x >> 6) * (D::kLanes * D::kCols) + part;
#pragma unroll
                for (int j = 0; j < D::kCols; j++) acc = acc + p[D::kLanes * j] * y[part + D::kLanes * j];
            }
            double sum = (double)acc;
            if constexpr (D::kLanes == 64) {
                sum = wave_sum(sum);
            } else {
                sum = sum + dpp_f64<0xB1>(sum);
                sum = sum + dpp_f64<0x4E>(sum);
                sum = sum + dpp_f64<0x141>(sum);
            }
            if (part == 0) w[(threadIdx.x >> 6) * D::kRows + lane / D::kLanes] = (V)sum;
            __syncthreads();
            return own ? w[threadIdx.x - own0] : (V)0;
        } else if constexpr (MODE == kSubst) {
            if ((int)threadIdx.x < 64 * group) {
                sf.template run<false>(y);
                sb.template run<true>(y);
            }
            __syncthreads();
            return mine ? y[threadIdx.x] : (V)0;
        } else {
            V *src = y, *dst = w, bl = t, cur = t;
            for (int s = 1; s < sweeps; s++) {
                cur = terms<0, kTriFirst, -1>(bl, l, llc, src);
                if (more_l) cur = terms<kTriFirst, kTri, -1>(cur, l, llc, src);
                if (mine) dst[threadIdx.x] = cur;
                __syncthreads();
                V *sw = src; src = dst; dst = sw;
            }
            bl = cur;
            cur = dinv * bl;
            for (int s = 1; s < sweeps; s++) {
                if (mine) dst[threadIdx.x] = cur;
                __syncthreads();
                V *sw = src; src = dst; dst = sw;
                cur = terms<0, kTriFirst, -1>(bl, u, uc, src);
                if (more_u) cur = terms<kTriFirst, kTri, -1>(cur, u, uc, src);
                cur = dinv * cur;
            }
            return cur;
        }
    }
    // Exchange of one epoch: the workgroups' partial sums of q (totals
    // returned to everyone) and, with HALO, the rows' values v (the halo
    // entries returned in h; dense: v of the block's other rows too).  False
    // when a wait ran out.
    template <int NQ, bool HALO>
    __device__ __attribute__((always_inline)) inline bool exchange(double (&q)[NQ], V &v, V (&h)[KH]) {
        // the wavefronts' sums
        __shared__ double red[NQ][T / 64], tot[NQ][kWaves], hi[NQ][T > kThreads ? kThreads : 1];
#pragma unroll
        for (int k = 0; k < NQ; k++) q[k] = wave_sum(q[k]);
        const int buf = epoch & (kZetaBufs - 1);
        U *vs = xch + (size_t)buf * nsend;
        wait_stores();          // the slots emptied after the last exchange
        if (HALO && own && send >= 0) slot_put<V>(vs + send, v);
        if ((threadIdx.x & 63) == 0)
#pragma unroll
            for (int k = 0; k < NQ; k++) red[k][threadIdx.x >> 6] = q[k];
        __syncthreads();
        // Each block's sum: its wavefronts' in order (a workgroup with more
        // than one block has blocks of whole wavefronts).
        const int bw = group == 1 ? T / 64 : rows / (64 * group);
        if (nsum == 1) {
#pragma unroll
            for (int k = 0; k < NQ; k++) {
                q[k] = red[k][0];
                for (int w = 1; w < bw; w++) q[k] += red[k][w];
            }
            return true;
        }
        for (int e = threadIdx.x; e < NQ * group * kPartCopies; e += T) {
            const int copy = e % kPartCopies, g = e / kPartCopies % group, k = e / (kPartCopies * group);
            double t = red[k][g * bw];
            for (int w = 1; w < bw; w++) t += red[k][g * bw + w];
            if (wg * group + g < nsum) slot_put<double>(part_slot(pslot, buf, copy, k, wg * group + g), t);
        }
        const unsigned long long *ps = part_slot(pslot, buf, wg % kPartCopies, 0, threadIdx.x);
        unsigned long long pv[NQ];
        U hv[KH], rv = 0;
        const bool recv = MODE == kDense && HALO && mine && !own;
        const bool hasp = (int)threadIdx.x < nsum;
        int spin = 0;
        for (;;) {
            bool ok = true;
            if (hasp)
#pragma unroll
                for (int k = 0; k < NQ; k++) pv[k] = slot_get(ps + k * 512);
            if (HALO)
#pragma unroll
                for (int k = 0; k < KH; k++)
                    if ((int)threadIdx.x + k * T < nh) hv[k] = slot_get(vs + hslot[k]);
            if (recv) rv = slot_get(vs + send);
            if (hasp)
#pragma unroll
                for (int k = 0; k < NQ; k++) ok = ok && pv[k] != Slot<double>::empty;
            if (HALO)
#pragma unroll
                for (int k = 0; k < KH; k++)
                    if ((int)threadIdx.x + k * T < nh) ok = ok && hv[k] != Slot<V>::empty;
            if (recv) ok = ok && rv != Slot<V>::empty;
            if (ok) break;
            if (++spin > spins) {
                *dead = 1;
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        // the total, in the order of Partials: work-item i holds partials i
        // and i + 256, then the wavefronts' sums, then these in order
#pragma unroll
        for (int k = 0; k < NQ; k++) q[k] = hasp ? 0. + __builtin_bit_cast(double, pv[k]) : 0.;
        if (recv) v = __builtin_bit_cast(V, rv);
        if (T > kThreads && nsum > kThreads) {
            if (threadIdx.x >= kThreads && threadIdx.x < 2 * kThreads)
#pragma unroll
                for (int k = 0; k < NQ; k++) hi[k][threadIdx.x - kThreads] = q[k];
            __syncthreads();
            if (threadIdx.x < kThreads)
#pragma unroll
                for (int k = 0; k < NQ; k++) q[k] += hi[k][threadIdx.x];
        }
        if (threadIdx.x < kThreads) {
#pragma unroll
            for (int k = 0; k < NQ; k++) q[k] = wave_sum(q[k]);
            if ((threadIdx.x & 63) == 0)
#pragma unroll
                for (int k = 0; k < NQ; k++) tot[k][threadIdx.x >> 6] = q[k];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < NQ; k++) {
            double t = tot[k][0];
#pragma unroll
            for (int w = 1; w < kWaves; w++) t += tot[k][w];
            q[k] = t;
        }
        if (HALO)
#pragma unroll
            for (int k = 0; k < KH; k++)
                h[k] = (int)threadIdx.x + k * T < nh ? __builtin_bit_cast(V, hv[k]) : (V)0;
        if (*dead) return false;
        // every workgroup has put its partials of this epoch, so the slots
        // of the epoch before are read out: empty them for epoch + 3, and
        // have that done before the next epoch's partials (one barrier later)
        if (epoch >= 1) {
            const int b1 = (epoch - 1) & (kZetaBufs - 1);
            if (own && send >= 0) slot_clear(xch + (size_t)b1 * nsend + send, Slot<V>::empty);
            for (int e = threadIdx.x; e < kPartSlots * group * kPartCopies; e += T) {
                const int g = e / kPartCopies % group;
                if (wg * group + g < nsum)
                    slot_clear(part_slot(pslot, b1, e % kPartCopies, e / (kPartCopies * group), wg * group + g),
                               Slot<double>::empty);
            }
        }
        epoch++;
        return true;
    }
};

// dynamic LDS of k_zeta
struct ZetaLds {
    size_t x, y, w, p, sub[2], total;
};
template <typename V>
__host__ __device__ inline ZetaLds zeta_lds(int rows, int group, int hmax, int chmax, int threads, int mode, int dmax) {
    const bool exact = mode == kSubst;
    const size_t sub = (size_t)threads * ((kSubFirst + 1) * sizeof(V) + (kSubFirst / 2 + 2) * sizeof(unsigned)) +
                       (size_t)group * chmax * sizeof(unsigned);
    auto up = [](size_t b) { return (b + 15) & ~(size_t)15; };
    ZetaLds l;
    size_t o = 0;
    // the operand also holds the FP64 residual's (rows and halo)
    l.x = o; o += up((size_t)(rows + hmax) * sizeof(double));
    l.y = o; o += up((size_t)(mode == kDense ? (threads == 512 ? 256 : 1024) : rows) * sizeof(V));
    l.w = o; o += exact ? 0 : up((size_t)(mode == kDense && rows < 64 ? 64 : rows) * sizeof(V));
    l.p = o; o += mode == kDense && threads == 1024 ? (size_t)DenseShape<1024>::kOwn * 1024 * sizeof(V) : 0;
    for (int d = 0; d < 2; d++) { l.sub[d] = o; o += exact ? up(sub) : 0; }
    l.total = o;
    // the inverse's rows are computed before the solve uses its LDS
    if (mode == kDense) {
        const size_t setup = up((size_t)rows * (threads == 512 ? DenseShape<512>::kOwn : DenseShape<1024>::kOwn) * sizeof(V)) + up((size_t)dmax * sizeof(V)) +
                             up((size_t)rows * sizeof(V)) + (size_t)(dmax + 3 * rows + 4) * sizeof(unsigned short);
        if (setup > l.total) l.total = setup;
    }
    return l;
}

// Rows own0 .. own0+nown-1 of the inverse of block blk's factors, this lane's
// columns of its row into p: e^T U^-1 L^-1 by the transposed factors, a level
// at a time for all the rows at once (work-items take a level's unknowns
// times the rows; a level of L is a level of U^T).
template <typename V, int T, bool BACK>
__device__ __attribute__((always_inline)) inline void dense_pass(const SolvArgs<V> &a, const ZetaArgs &z, int blk,
                                                                 int nb, int own0, V *xs, V *tv, const V *dv,
                                                                 unsigned short *tk, unsigned short *ep,
                                                                 unsigned short *rows, unsigned short *lp) {
    constexpr int R = DenseShape<T>::kOwn;
    const int stride = a.brows + 1;
    const int *ptr = (BACK ? z.dptr_b : z.dptr_f) + (size_t)blk * stride;
    const unsigned *ent = (BACK ? z.dent_b : z.dent_f) + (size_t)blk * z.dmax;
    const int *order = (BACK ? z.rows_b : z.rows_f) + (size_t)blk * a.brows;
    const int *lptr = (BACK ? a.blptr : a.flptr) + (size_t)blk * stride;
    const int nlev = (BACK ? a.bnlev : a.fnlev)[blk];
    const V *lu = a.lu + (size_t)blk * a.mx;
    for (int e = threadIdx.x; e < ptr[nb]; e += T) {
        const unsigned w = ent[e];
        tv[e] = lu[w & 0xffffu];
        tk[e] = (unsigned short)(w >> 16);
    }
    for (int t = threadIdx.x; t <= nb; t += T) {
        ep[t] = (unsigned short)ptr[t];
        if (t < nb) rows[t] = (unsigned short)order[t];
    }
    for (int l = threadIdx.x; l <= nlev; l += T) lp[l] = (unsigned short)lptr[l];
    __syncthreads();
    for (int l = 0; l < nlev; l++) {
        const int t0 = lp[l], n = (lp[l + 1] - t0) * R;
        for (int e = threadIdx.x; e < n; e += T) {
            const int t = t0 + e / R, r = e % R, j = rows[t];
            V acc = BACK ? xs[(size_t)j * R + r] : (j == own0 + r ? (V)1 : (V)0);
            for (int q = ep[t]; q < ep[t + 1]; q++) acc = acc - tv[q] * xs[(size_t)tk[q] * R + r];
            xs[(size_t)j * R + r] = BACK ? acc : acc * dv[j];
        }
        __syncthreads();
    }
}

template <typename V, int T>
__device__ __attribute__((always_inline)) inline void dense_rows(const SolvArgs<V> &a, const ZetaArgs &z, int blk,
                                                                 int nb, int own0, unsigned char *lds,
                                                                 V (&p)[DenseShape<T>::kCols]) {
    using D = DenseShape<T>;
    constexpr int R = D::kOwn;
    auto up = [](size_t b) { return (b + 15) & ~(size_t)15; };
    V *xs = reinterpret_cast<V *>(lds);
    V *tv = reinterpret_cast<V *>(lds + up((size_t)a.brows * R * sizeof(V)));
    V *dv = reinterpret_cast<V *>(reinterpret_cast<unsigned char *>(tv) + up((size_t)z.dmax * sizeof(V)));
    unsigned short *tk = reinterpret_cast<unsigned short *>(reinterpret_cast<unsigned char *>(dv) +
                                                            up((size_t)a.brows * sizeof(V)));
    unsigned short *ep = tk + z.dmax, *rows = ep + a.brows + 1, *lp = rows + a.brows;
    for (int t = threadIdx.x; t < nb; t += T)
        dv[t] = a.lu[(size_t)blk * a.mx + a.pdg[(size_t)blk * a.brows + t]];
    dense_pass<V, T, false>(a, z, blk, nb, own0, xs, tv, dv, tk, ep, rows, lp);
    dense_pass<V, T, true>(a, z, blk, nb, own0, xs, tv, dv, tk, ep, rows, lp);
    const int lane = threadIdx.x & 63, r = (threadIdx.x >> 6) * D::kRows + lane / D::kLanes;
#pragma unroll
    for (int j = 0; j < D::kCols; j++) {
        const int c = lane % D::kLanes + D::kLanes * j;
        p[j] = c < nb && r < R ? xs[(size_t)c * R + r] : (V)0;
    }
    __syncthreads();
}

// the rows of the workgroup's blocks into LDS, in the order of one substitution
template <typename V, int T, bool BACK>
__device__ __attribute__((always_inline)) inline SubExact<V, T> stage_sub(const SolvArgs<V> &a, const ZetaArgs &z,
                                                                          int wg, unsigned char *lds) {
    SubExact<V, T> s;
    V *val = reinterpret_cast<V *>(lds), *piv = val + kSubFirst * T;
    unsigned *col = reinterpret_cast<unsigned *>(piv + T), *row = col + (kSubFirst / 2) * T, *tail = row + T,
             *chunk = tail + T;
    const int *nch = BACK ? z.nch_b : z.nch_f;
    const unsigned *chunks = BACK ? z.chunk_b : z.chunk_f;
    // position t: row rows[..] of the block t / brows
    const int t = threadIdx.x, g = t / a.brows, r0 = g * a.brows, blk = wg * z.group + g;
    const bool on = g < z.group && blk < a.nblk && blk * a.brows + t - r0 < a.n;
    const V *lu = a.lu + (on ? (size_t)blk * a.mx : 0);
    const int *pcol = a.pcol + (on ? (size_t)blk * a.mx : 0);
    int li = 0, d = 0, e0 = 0, cnt = 0;
    if (on) {
        const int *rp = a.prp + (size_t)blk * (a.brows + 1);
        li = (BACK ? z.rows_b : z.rows_f)[blk * a.brows + t - r0];
        d = a.pdg[(size_t)blk * a.brows + li];
        e0 = BACK ? d + 1 : rp[li];
        cnt = BACK ? rp[li + 1] - e0 : d - e0;
    }
    unsigned c[kSubFirst];
#pragma unroll
    for (int k = 0; k < kSubFirst; k++) {
        val[k * T + t] = k < cnt ? lu[e0 + k] : (V)0;
        c[k] = on ? (unsigned)((r0 + (k < cnt ? pcol[e0 + k] : li)) * (int)sizeof(V)) : 0u;
    }
#pragma unroll
    for (int k = 0; k < kSubFirst / 2; k++) col[k * T + t] = c[2 * k] | c[2 * k + 1] << 16;
    piv[t] = BACK && on ? lu[d] : (V)0;
    row[t] = on ? (unsigned)((r0 + li) * (int)sizeof(V)) | (unsigned)max(0, cnt - kSubFirst) << 16 : 0u;
    tail[t] = (unsigned)(e0 + kSubFirst);
    for (int e = t; e < z.group * z.chmax; e += T) {
        const int b = wg * z.group + e / z.chmax;
        chunk[e] = b < a.nblk ? chunks[(size_t)b * z.chmax + e % z.chmax] : 0u;
    }
    s.val = val; s.piv = piv; s.col = col; s.row = row; s.tail = tail;
    // this wavefront's block
    const int w = min((int)threadIdx.x >> 6, z.group - 1), wb = wg * z.group + w;
    s.chunk = chunk + w * z.chmax;
    s.r0 = w * a.brows;
    s.nch = wb < a.nblk ? nch[wb] : 0;
    s.lu = a.lu + (wb < a.nblk ? (size_t)wb * a.mx : 0);
    s.pcol = a.pcol + (wb < a.nblk ? (size_t)wb * a.mx : 0);
    return s;
}

template <typename V, int T, int KH, int MODE>
__global__ __launch_bounds__(T) void k_zeta(SolvArgs<V> a, ZetaArgs z) {
    constexpr bool REFINE = sizeof(V) == 4;
    extern __shared__ double smem[];
    __shared__ int dead;
    unsigned char *lds = reinterpret_cast<unsigned char *>(smem);
    const ZetaLds L = zeta_lds<V>(z.group * a.brows, z.group, z.hmax, z.chmax, T, MODE, z.dmax);
    const int tid = threadIdx.x;
    if (tid == 0) dead = 0;
    ZetaRow<V, T, KH, MODE> R;
    R.wg = xcd_block(blockIdx.x, gridDim.x);
    R.nsum = MODE == kDense ? z.nwg : a.nblk;
    R.n = a.n; R.sweeps = a.sweeps; R.rows = z.group * a.brows; R.group = z.group;
    // the workgroup's rows: its blocks, or (dense) its block of several workgroups
    const int part = MODE == kDense ? R.wg / z.members : R.wg;
    const int b0 = part * R.rows, nb = min(a.n, b0 + R.rows) - b0;
    R.i = b0 + tid;
    R.mine = tid < nb;
    R.own = R.mine;
    if (MODE == kDense) {
        R.own0 = R.wg % z.members * DenseShape<T>::kOwn;
        R.own = R.mine && tid >= R.own0 && tid < R.own0 + DenseShape<T>::kOwn;
    }
    R.nh = z.hcnt[part];
    R.X = reinterpret_cast<V *>(lds + L.x);
    R.y = reinterpret_cast<V *>(lds + L.y);
    R.w = reinterpret_cast<V *>(lds + L.w);
    R.xch = (typename Slot<V>::U *)z.xch;
    R.pslot = z.pslot;
    R.dead = &dead;
    R.spins = z.spins;
    R.send = -1;
    R.nsend = z.nsend;
    int hcol[KH];
    double *X64 = reinterpret_cast<double *>(lds + L.x);
    const size_t n = a.n;
    const int i = R.i;
#pragma unroll
    for (int k = 0; k < KH; k++) {
        const bool on = tid + k * T < R.nh;
        const size_t h = (size_t)part * z.hmax + tid + k * T;
        hcol[k] = on ? z.hcol[h] : 0;
        R.hslot[k] = on ? z.hslot[h] : 0;
    }
    constexpr bool HOLD = ZetaRow<V, T, KH, MODE>::kHold;
    R.ga = a.ell_a;
    R.glc = z.lcol;
#pragma unroll
    for (int k = 0; k < (HOLD ? kEllWidth : 1); k++) R.a[k] = 0;
#pragma unroll
    for (int k = 0; k < (HOLD ? kEllWidth / 2 : 1); k++) R.lc[k] = 0;
    double a64[REFINE && HOLD ? kEllWidth : 1] = {};
    int q64 = 0;
    double b64 = 0., x64 = 0., xh64[KH] = {};
    V bown = 0;
    int len = 0;
    if (R.mine) {
        R.send = z.send[i];
        len = a.ell_len[i];
        if constexpr (HOLD) {
#pragma unroll
            for (int k = 0; k < kEllWidth; k++) R.a[k] = a.ell_a[(size_t)k * n + i];
#pragma unroll
            for (int k = 0; k < kEllWidth / 2; k++) R.lc[k] = z.lcol[(size_t)k * n + i];
        }
        if (REFINE) {
            q64 = a.rowptr[i];
            if constexpr (HOLD) {
#pragma unroll
                for (int k = 0; k < kEllWidth; k++)
                    if (k < len) a64[k] = a.aval[q64 + k];
            }
            b64 = z.rhs[i];
            x64 = z.x[i];
        } else {
            bown = a.b[i];
            x64 = (double)a.x0[i];
        }
    }
#pragma unroll
    for (int k = 0; k < KH; k++)
        if (tid + k * T < R.nh) xh64[k] = REFINE ? z.x[hcol[k]] : (double)a.x0[hcol[k]];
    R.more_a = __any(len > kRowFirst);
#pragma unroll
    for (int k = 0; k < R.kTri; k++) R.l[k] = R.u[k] = 0;
#pragma unroll
    for (int k = 0; k < R.kTriWords; k++) R.llc[k] = R.uc[k] = 0;
    if constexpr (MODE == kDense) {
        using D = DenseShape<T>;
        if constexpr (D::kRegs) {
            dense_rows<V, T>(a, z, part, nb, R.own0, lds, R.pinv);
        } else {
            V p[D::kCols], *pl = reinterpret_cast<V *>(lds + L.p);
            dense_rows<V, T>(a, z, part, nb, R.own0, lds, p);
            R.plds = pl;
            if ((tid >> 6) < D::kOwn)
#pragma unroll
                for (int j = 0; j < D::kCols; j++) pl[(size_t)(tid >> 6) * (D::kLanes * D::kCols) + (tid & 63) + D::kLanes * j] = p[j];
        }
        // the right-hand side's unused columns: zeros
        for (int t = tid; t < DenseShape<T>::kLanes * DenseShape<T>::kCols; t += T) R.y[t] = 0;
        if (tid == 0) dead = 0;
        __syncthreads();
    } else if constexpr (MODE == kSubst) {
        R.sf = stage_sub<V, T, false>(a, z, R.wg, lds + L.sub[0]);
        R.sb = stage_sub<V, T, true>(a, z, R.wg, lds + L.sub[1]);
    } else {
        int nl = 0, nu = 0;
        if (R.mine) {
            const int meta = a.fs_meta[i], self = tid, r0 = tid / a.brows * a.brows;
            nl = meta & 255;
            nu = (meta >> 8) - nl - 1;
            R.dinv = a.fs_val[i];
#pragma unroll
            for (int k = 0; k < kTriWidth; k++) {
                const bool hl = k < nl, hu = k < nu;
                const size_t sl = (size_t)(k + 1) * n + i, su = (size_t)(nl + 1 + k) * n + i;
                const unsigned cl = (unsigned)((hl ? r0 + a.fs_col[sl] : self) * (int)sizeof(V));
                const unsigned cu = (unsigned)((hu ? r0 + a.fs_col[su] : self) * (int)sizeof(V));
                R.l[k] = hl ? a.fs_val[sl] : (V)0;
                R.u[k] = hu ? a.fs_val[su] : (V)0;
                R.llc[k / 2] |= cl << (16 * (k & 1));
                R.uc[k / 2] |= cu << (16 * (k & 1));
            }
        }
        R.more_l = __any(nl > kTriFirst);
        R.more_u = __any(nu > kTriFirst);
    }
    int conv = 0, fail = 0, maxit = 0, nmv = 1, its = 0, nref = 0, refconv = 0;
    double rn = 0.;
    V dx = 0;
    for (;;) {
        V rhs, hdx[KH];
        if (REFINE) {
            // FP64 residual of the current x and its test (k_resid64, k_resid_check)
            __syncthreads();
            if (R.mine) X64[tid] = x64;
#pragma unroll
            for (int k = 0; k < KH; k++)
                if (tid + k * T < R.nh) X64[R.rows + tid + k * T] = xh64[k];
            __syncthreads();
            double t = 0.;
            unsigned cv[kEllWidth / 2];
            R.columns(cv);
#pragma unroll
            for (int k = 0; k < kEllWidth; k++)
                if (k < len) t = t + (HOLD ? a64[HOLD ? k : 0] : a.aval[q64 + k]) * X64[R.off(cv, k) / sizeof(V)];
            const double r = b64 - t;
            double rs[2] = {R.own ? r * r : 0., R.own ? b64 * b64 : 0.};
            V none[KH], nov = 0;
            if (!R.template exchange<2, false>(rs, nov, none)) { fail = kWaitExpired; break; }
            rn = sqrt(rs[0]);
            if (rn <= z.tol * sqrt(rs[1])) { refconv = 1; break; }
            if (nref >= z.maxref) break;
            nref++;
            rhs = (V)r;
        } else {
            // b - A x0
            V h[KH];
#pragma unroll
            for (int k = 0; k < KH; k++) h[k] = (V)xh64[k];
            R.operand((V)x64, h);
            const V t = R.product();
            rhs = bown - t;
        }
        // r0 = M^-1 rhs
        V r = R.precond(rhs), p = 0, v = 0, s = 0, t = 0;
        V hr[KH], hp[KH], hv[KH], hs[KH], ht[KH];
#pragma unroll
        for (int k = 0; k < KH; k++) { hp[k] = hv[k] = hs[k] = ht[k] = 0; hdx[k] = 0; }
        if (!R.mine) r = 0;
        dx = 0;
        conv = fail = maxit = 0;
        double q5[5] = {0., 0., 0., 0., 0.}, q1[1] = {(double)r * (double)r};
        if (!R.template exchange<1, true>(q1, r, hr)) { fail = kWaitExpired; break; }
        const V r0 = r;
        double target = 0., alpha = 0., rho = q1[0], rho_prev = 0., omega = 0.;
        for (int it = 0;; it++) {
            if (it == 0) {
                rn = sqrt(q1[0]);
                target = a.rtol * rn + a.atol;
            } else {
                // q5: (t,t) (t,s) (s,s) (r0,s) (r0,t)
                if (breakdown(q5[0])) { fail = -3; break; }
                omega = q5[1] / q5[0];
                if (breakdown(omega)) { fail = -3; break; }
                rn = sqrt(fmax(0., q5[2] - 2. * omega * q5[1] + omega * omega * q5[0]));
                rho = q5[3] - omega * q5[4];
                const V va = (V)alpha, vo = (V)omega;
                dx = dx + (va * p + vo * s);
                r = s - vo * t;
#pragma unroll
                for (int k = 0; k < KH; k++) {
                    if (REFINE) hdx[k] = hdx[k] + (va * hp[k] + vo * hs[k]);
                    hr[k] = hs[k] - vo * ht[k];
                }
                its++;
            }
            nmv = 1 + 2 * it;
            if (!(rn > target)) { conv = 1; break; }
            if (it > 0 && a.itermax > 0 && 1 + 2 * it >= a.itermax) { maxit = 1; break; }
            // without an itermax nothing else ends a recurrence that
            // stagnates above its target (no convergence: the host's errors)
            if (it >= z.maxit) break;
            if (it == 0) {
                p = r;
#pragma unroll
                for (int k = 0; k < KH; k++) hp[k] = hr[k];
            } else {
                if (breakdown(rho)) { fail = -3; break; }
                const V vb = (V)(rho * alpha / (omega * rho_prev)), vo = (V)omega;
                p = r + vb * (p - vo * v);
#pragma unroll
                for (int k = 0; k < KH; k++) hp[k] = hr[k] + vb * (hp[k] - vo * hv[k]);
            }
            rho_prev = rho;
            R.operand(p, hp);
            v = R.precond(R.product());
            q1[0] = R.own ? (double)r0 * (double)v : 0.;
            if (!R.template exchange<1, true>(q1, v, hv)) { fail = kWaitExpired; break; }
            if (breakdown(q1[0])) { fail = -3; break; }
            alpha = rho / q1[0];
            const V va = (V)alpha;
            s = r - va * v;
#pragma unroll
            for (int k = 0; k < KH; k++) hs[k] = hr[k] - va * hv[k];
            R.operand(s, hs);
            t = R.precond(R.product());
            const double tv = R.own ? (double)t : 0., sv = R.own ? (double)s : 0., r0v = (double)r0;
            q5[0] = tv * tv;
            q5[1] = tv * sv;
            q5[2] = sv * sv;
            q5[3] = r0v * sv;
            q5[4] = r0v * tv;
            if (!R.template exchange<5, true>(q5, t, ht)) { fail = kWaitExpired; break; }
        }
        if (!REFINE || fail == kWaitExpired) break;
        if (tid == 0 && R.wg == 0 && nref <= CT_NRITS) a.ctrl[CT_RITS + nref - 1] = (nmv - 1) / 2;
        // x += correction
        x64 = x64 + (double)dx;
#pragma unroll
        for (int k = 0; k < KH; k++) xh64[k] = xh64[k] + (double)hdx[k];
    }
    if (fail == kWaitExpired) {
        if (tid == 0) a.ctrl[CT_WAIT] = 1;
        return;
    }
    if (R.own) {
        if (REFINE) z.x[i] = x64;
        else a.dx[i] = dx;
    }
    // commit: workgroup 0 sets the flags after everyone's stores
    if (z.nwg > 1) {
        const int buf = R.epoch & (kZetaBufs - 1);
        unsigned long long *ps = part_slot(z.pslot, buf, 0, 0, 0);
        wait_stores();
        __syncthreads();
        if (tid == 0) slot_put<double>(ps + R.wg, 1.);
        if (R.wg != 0) return;
        if (tid < z.nwg) {
            int spin = 0;
            while (slot_get(ps + tid) == Slot<double>::empty) {
                if (++spin > z.spins) {
                    dead = 1;
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
            }
        }
        __syncthreads();
        if (dead) {
            if (tid == 0) a.ctrl[CT_WAIT] = 1;
            return;
        }
    }
    if (tid == 0 && R.wg == 0) {
        a.ctrl[CT_STOPIT] = 1;
        a.ctrl[CT_CONV] = conv;
        a.ctrl[CT_FAIL] = fail;
        a.ctrl[CT_MAXIT] = maxit;
        a.ctrl[CT_NMV] = nmv;
        a.ctrl[CT_ITS] = its;
        a.ctrl[CT_NREF] = nref;
        a.ctrl[CT_REFCONV] = refconv;
        a.scal[REFINE ? SC_RES64 : SC_RNORM] = rn;
    }
}

// ---------------------------------------------------------------- host driver
// The solver's control words and the device error words into the host's
// pinned memory, then the number of this report: the host waits for it
// (wait_report) instead of two copies and a stream synchronisation.
// go (may be null): whether the solve converged (word `conv`), no error is
// set and no element changed its wet/dry state, for the kernels enqueued
// behind the report.
__global__ __launch_bounds__(64) void k_report(const int *ctrl, const int *err, int *host, int seq, int conv, int *go) {
    const int t = threadIdx.x;
    if (t == 0 && go) {
        const bool ok = ctrl[conv] && !ctrl[CT_FACTOR] && !err[0] && !err[1] &&
                        (conv == CT_REFCONV || !(ctrl[CT_FAIL] || ctrl[CT_MAXIT]));
        *go = ok;
        host[HP_GO] = ok;
    }
    if (t < CT_WORDS) host[HP_CTRL + t] = ctrl[t];
    else if (t < CT_WORDS + 2) host[HP_ERR + t - CT_WORDS] = err[t - CT_WORDS];
    __threadfence_system();
    __syncthreads();
    if (t == 0) __hip_atomic_store(host + HP_SEQ, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// the work before it on the stream has ended
__global__ void k_mark(int *host, int seq) {
    __hip_atomic_store(host, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// one read-back: the solver's control words and the device error word and
// counter d_err[0..1] (into h_pinned[HP_ERR..])
static int read_ctrl(Model &M, int *out, int n, const std::function<int(const int *)> *after = nullptr,
                     int conv = CT_CONV) {
    const int seq = ++M.report_seq;
    int *go = after ? M.d_err + kErrGo : nullptr;
    hipLaunchKernelGGL(k_report, dim3(1), dim3(64), 0, M.stream, (const int *)M.sv.ctrl, (const int *)M.d_err,
                       M.h_pinned, seq, conv, go);
    HIPCHK(M, hipGetLastError());
    if (after && (*after)(go)) return 1;
    if (wait_report(M, HP_SEQ, seq)) return 1;
    for (int i = 0; i < n; i++) out[i] = M.h_pinned[HP_CTRL + i];
    return 0;
}

static constexpr size_t kLdsLimit = 64 * 1024;
static constexpr size_t kLdsStatic = 3 * kThreads * sizeof(double);   // reduction buffers

// dynamic LDS of the kernels that apply the preconditioner: with the block
// staged, or y and w only (blocks too large to stage read factors from
// global memory)
template <typename V>
static bool stage_fits(const Model &M) {
    return staged_lds<V>(M.sv.brows, M.sv.max_blk_nnz) + kLdsStatic <= kLdsLimit;
}

template <typename V>
static size_t apply_lds(const Model &M) {
    return stage_fits<V>(M) ? staged_lds<V>(M.sv.brows, M.sv.max_blk_nnz) : 2 * (size_t)M.sv.brows * sizeof(V);
}

// dynamic LDS of the iteration kernels: with halos y, w and the operand
template <typename V, int MODE>
static size_t iter_lds(const Model &M) {
    return MODE == 3 ? (3 * (size_t)M.sv.brows + M.sv.zeta_hmax) * sizeof(V) : apply_lds<V>(M);
}

// block factors of the current matrix (exact block ILU(0)), every solve: the
// wet/dry state changes rows of the zeta matrix from one step to the next
// (dry-element rows, level boundaries), and factors of an earlier matrix
// then no longer precondition it.
// LDS of the factorisation: the block's values, and when they fit the
// descriptors, pairs and level starts
// sweeps of a warm start (four reach the iteration counts of exact factors
// on the 50k-node lagoon, two do not), and exact factorisations at least
// every kWarmRefresh solves
constexpr int kMaxRefine = 40;          // FP64 refinement rounds of a solve
constexpr int kWarmSweeps = 4;
constexpr int kWarmRefresh = 16;

template <typename V>
static int factor(Model &M, SolvArgs<V> &a) {
    const int sweeps = (kWarmSweeps > 0 && M.sv.have_lu && M.sv.max_blk_nnz <= kWarmEntries * kFactorThreads)
                           ? kWarmSweeps : 0;
    M.sv.last_warm = sweeps > 0;
    if (sweeps == 0) M.sv.solves_since_exact = 0;
    const size_t vals = (((size_t)M.sv.max_blk_nnz * sizeof(V) + 15) & ~(size_t)15) * (sweeps > 0 ? 2 : 1);
    const size_t lists = (size_t)M.sv.max_blk_nnz * sizeof(int4) + (size_t)M.sv.max_blk_pairs * sizeof(int2) +
                         (size_t)(M.sv.max_elev + 1) * sizeof(int);
    const int stage = vals + lists <= kLdsLimit ? 1 : 0;
    launch_timed(M, T_FACTOR, k_bilu_factor<V>, dim3(M.sv.nblk), dim3(kFactorThreads), stage ? vals + lists : vals,
                 M.stream, a, stage, sweeps);
    if (M.sv.zeta_members > 0)
        hipLaunchKernelGGL(k_empty_partials, dim3(kZetaBufs * kPartCopies * kPartSlots), dim3(kThreads), 0, M.stream,
                           M.sv.pslot, M.sv.zeta_nwg);
    HIPCHK(M, hipGetLastError());
    M.sv.have_lu = true;
    return 0;
}

// iterations and errors of a finished BiCGStab solve from its control words
static int krylov_outcome(Model &M, const int *c, int *iters, int slot) {
    if (iters) *iters = (c[CT_NMV] - 1) / 2;
    M.sv.last_its[slot] = (c[CT_NMV] - 1) / 2;
    if (c[CT_FACTOR] != 0) {
        M.err = "zeta solver: zero pivot in the block factorisation (row " + std::to_string(c[CT_FACTOR]) + ")";
        return 2;
    }
    if (c[CT_FAIL] != 0 || c[CT_MAXIT] != 0) {
        M.err = "zeta solver: BiCGStab failed (code " + std::to_string(c[CT_FAIL] ? c[CT_FAIL] : -1) + ")";
        return 2;
    }
    if (!c[CT_CONV]) {
        M.err = "zeta solver: no convergence";
        return 2;
    }
    return 0;
}

// The iterations it0 .. it0 + n - 1 in pieces of about 0.3 ms, no more than
// two of them enqueued and not finished.
//
// Streams share a few hardware queues (four per process), each of which runs
// what it was given in order: a stream that shares a queue waits behind all
// that the other has enqueued, every time that its own host waits.  A solve
// of 500 iterations on 331k nodes is 25 ms; with all of it enqueued at once, 9
// small runs in one model beside it took 10.5 s (median), 4.4 s where the
// streams had queues of their own; 7.4 s with pieces of 32 iterations (0.8
// ms), 5.9 s of 12.  The device does not idle, since the host waits for the piece before
// the last; a mark per piece costs 3 us.
constexpr int kPieceRows = 4000000, kPieceLeast = 12;
template <typename F>
static int in_pieces(Model &M, int it0, int n, F piece) {
    const int most = std::max(kPieceLeast, kPieceRows / M.nkn);
    int q = 0, before = 0;
    for (; n - q > most + most / 2; q += most) {
        if (piece(it0 + q, most)) return 1;
        const int seq = ++M.report_seq;
        hipLaunchKernelGGL(k_mark, dim3(1), dim3(1), 0, M.stream, M.h_pinned + HP_PIECE, seq);
        HIPCHK(M, hipGetLastError());
        if (before && wait_report(M, HP_PIECE, before)) return 1;
        before = seq;
    }
    return piece(it0 + q, n - q);
}

// Iterations of one Krylov solve at most (FP32: of one refinement round),
// also without an itermax.
static int krylov_cap(const Model &M) {
    if (M.prec == SHYHIP_FP64) return M.p.itermax > 0 ? (M.p.itermax + 1) / 2 + 1 : 100000;
    return M.p.itermax > 0 ? (M.p.itermax + 1) / 2 : 500;
}

// One iteration is two kernels (k_bicg_a, k_bicg_b).  Iterations are
// enqueued in chunks between host checks of the device flags;
// the first chunk is the iteration count of the previous solve of the same
// kind (`slot`), so a converging solve usually needs a single round trip.
// Kernels enqueued after convergence return immediately.  `tail` enqueues
// the work that follows a converged solve, switched on by its flag, before
// each check.
// MODE of the iteration kernels: 0 block factors read from global memory,
// 1 staged in LDS, 2 factor rows in registers (the init kernel stages), 3 the
// same with the blocks' halos in LDS
template <typename V, int MODE>
static int bicgstab_t(Model &M, SolvArgs<V> &a, int *iters, int slot, int zero_x0,
                      const std::function<int()> &tail) {
    const int g = a.nblk;
    const size_t lds = apply_lds<V>(M), ilds = iter_lds<V, MODE>(M);
    int it = 0, c[CT_WORDS] = {};
    const int maxit = krylov_cap(M);
    int chunk = std::max(2, M.sv.last_its[slot] + 1);
    for (;;) {
        // the chunk's iterations (after the initialisation, for the first),
        // each piece as one replayed launch sequence
        auto piece = [&](int it0, int n) -> int {
            auto launches = [&]() -> int {
                if (it0 == 0)
                    hipLaunchKernelGGL((k_bicg_init<V, MODE != 0>), dim3(g), dim3(kThreads), lds, M.stream, a, zero_x0);
                for (int q = 0; q < n; q++) {
                    launch_timed(M, T_BICG_A, k_bicg_a<V, MODE>, dim3(g), dim3(kThreads), ilds, M.stream, a, it0 + q);
                    launch_timed(M, T_BICG_B, k_bicg_b<V, MODE>, dim3(g), dim3(kThreads), ilds, M.stream, a, it0 + q);
                }
                HIPCHK(M, hipGetLastError());
                return 0;
            };
            std::string key("bicgstab");
            key_add(key, a);
            key_add(key, MODE);
            key_add(key, lds);
            key_add(key, it0);
            key_add(key, n);
            key_add(key, zero_x0);
            return graph_run(M, M.stream, key, launches);
        };
        if (in_pieces(M, it, chunk, piece)) return 1;
        it += chunk;
        if (tail && tail()) return 1;
        if (read_ctrl(M, c, CT_WORDS)) return 1;
        if (c[CT_CONV] || c[CT_FAIL] || c[CT_MAXIT] || it >= maxit) break;
        chunk = 2;
    }
    return krylov_outcome(M, c, iters, slot);
}

template <typename V>
static int iter_mode(const Model &M, const SolvArgs<V> &a) {
    if (!stage_fits<V>(M)) return 0;
    return (a.fs_val && a.brows <= kThreads) ? (a.hcol ? 3 : 2) : 1;
}

template <typename V>
static int bicgstab(Model &M, SolvArgs<V> &a, int *iters, int slot, int zero_x0, const std::function<int()> &tail) {
    switch (iter_mode(M, a)) {
    case 3: return bicgstab_t<V, 3>(M, a, iters, slot, zero_x0, tail);
    case 2: return bicgstab_t<V, 2>(M, a, iters, slot, zero_x0, tail);
    case 1: return bicgstab_t<V, 1>(M, a, iters, slot, zero_x0, tail);
    default: return bicgstab_t<V, 0>(M, a, iters, slot, zero_x0, tail);
    }
}

// one inner FP32 solve of the refinement, enqueued without host checks:
// init from a zero correction, then `chunk` iterations (no-ops once
// converged or once the refinement has converged)
template <typename V, int MODE>
static int enqueue_inner_t(Model &M, SolvArgs<V> &a, int chunk) {
    const int g = a.nblk;
    const size_t lds = apply_lds<V>(M), ilds = iter_lds<V, MODE>(M);
    auto piece = [&](int it0, int n) -> int {
        auto launches = [&]() -> int {
            if (it0 == 0)
                hipLaunchKernelGGL((k_bicg_init<V, MODE != 0>), dim3(g), dim3(kThreads), lds, M.stream, a, 1);
            for (int it = it0; it < it0 + n; it++) {
                launch_timed(M, T_BICG_A, k_bicg_a<V, MODE>, dim3(g), dim3(kThreads), ilds, M.stream, a, it);
                launch_timed(M, T_BICG_B, k_bicg_b<V, MODE>, dim3(g), dim3(kThreads), ilds, M.stream, a, it);
            }
            HIPCHK(M, hipGetLastError());
            return 0;
        };
        // one replayed launch sequence per argument set and piece
        std::string key("inner");
        key_add(key, a);
        key_add(key, MODE);
        key_add(key, lds);
        key_add(key, it0);
        key_add(key, n);
        return graph_run(M, M.stream, key, launches);
    };
    return in_pieces(M, 0, chunk, piece);
}

template <typename V>
static int enqueue_inner(Model &M, SolvArgs<V> &a, int chunk) {
    switch (iter_mode(M, a)) {
    case 3: return enqueue_inner_t<V, 3>(M, a, chunk);
    case 2: return enqueue_inner_t<V, 2>(M, a, chunk);
    case 1: return enqueue_inner_t<V, 1>(M, a, chunk);
    default: return enqueue_inner_t<V, 0>(M, a, chunk);
    }
}


// The one-launch solve: kernel of the workgroup size, the halo entries per
// work-item and the kind of triangular solve.
template <typename V>
using ZetaKernel = void (*)(SolvArgs<V>, ZetaArgs);
static int zeta_mode(const Model &M) {
    return M.p.tri_sweeps > 0 ? kSwept : (M.sv.zeta_members > 0 ? kDense : kSubst);
}
template <typename V>
static ZetaKernel<V> zeta_kernel(const Model &M) {
    const int mode = zeta_mode(M);
    // (exact substitution in FP64 only, see host_zeta_tables)
    if constexpr (std::is_same<V, double>::value) {
        if (mode == kDense) return M.sv.zeta_t == 1024 ? k_zeta<V, 1024, 1, kDense> : k_zeta<V, 512, 1, kDense>;
        if (mode == kSubst)
            return M.sv.zeta_t == 1024 ? k_zeta<V, 1024, 1, kSubst>
                                       : (M.sv.zeta_t == 512 ? k_zeta<V, 512, 1, kSubst>
                                                             : (M.sv.zeta_hmax <= 256 ? k_zeta<V, 256, 1, kSubst>
                                                                                      : k_zeta<V, 256, 2, kSubst>));
    }
    if (M.sv.zeta_t == 512) return k_zeta<V, 512, 1, kSwept>;
    return M.sv.zeta_hmax <= 256 ? k_zeta<V, 256, 1, kSwept> : k_zeta<V, 256, 2, kSwept>;
}

// Workgroups of the one-launch solve wait for each other, so a launch is
// made only when all of them can be resident together with those of every
// other such launch of this process: each takes its share of the device's
// compute units (workgroups / workgroups that fit one unit) out of the
// units that are not taken, and waits for them otherwise (a solve holds
// them for some hundred microseconds).  Launches that need no other
// workgroup to proceed (everything else) end by themselves and only delay it.
namespace {
UnitBudget &zeta_units() {
    static UnitBudget u;
    return u;
}
struct ZetaHold {
    int dev;
    long parts;
    ZetaHold(int d, long n, long budget) : dev(d), parts(n) { zeta_units().take(dev, parts, budget); }
    ~ZetaHold() { zeta_units().give(dev, parts); }
    ZetaHold(const ZetaHold &) = delete;
    ZetaHold &operator=(const ZetaHold &) = delete;
};
}  // namespace

constexpr size_t kZetaStatic = 20480;         // at least the kernels' static LDS

// LDS, device share and capacity of this model's next one-launch solve under
// its current parameters; cost < 0: it cannot run (the two-kernel iteration does)
struct ZetaPlan {
    size_t lds = 0;
    int dev = 0;
    long cost = -1, cap = 0;
};
template <typename V>
static ZetaPlan zeta_plan(Model &M) {
    ZetaPlan p;
    Solver &v = M.sv;
    if (v.zeta_t == 0) return p;
    if (v.zeta_rest > 0) {                        // see zeta_expired
        v.zeta_rest--;
        return p;
    }
    const int mode = zeta_mode(M), exact = mode != kSwept;
    if (exact && sizeof(V) == 4) return p;        // FP64 only (see host_zeta_tables)
    // sweeps keep the factor row in registers (and need its slot-major copy),
    // and a basin laid out for dense rows has one block's work-items per workgroup
    if (!exact && (!v.fs_val || v.brows > kThreads || v.zeta_members > 0)) return p;
    p.lds = zeta_lds<V>(v.zeta_group * v.brows, v.zeta_group, v.zeta_hmax, v.zeta_chmax, v.zeta_t, mode, v.zeta_dmax).total;
    if (v.zeta_occ[exact] == 0) {
        // asked once per model and kind
        int dev = 0, cus = 0, occ = 0, lds_max = 0;
        const void *fn = (const void *)zeta_kernel<V>(M);
        // (the limit belongs to the kernel, which models of several sizes
        // share: always the most that any of them may ask for)
        const bool ok =
            hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
            hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) == hipSuccess &&
            p.lds + kZetaStatic <= (size_t)lds_max &&
            (p.lds <= kLdsLimit || hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                       lds_max - (int)kZetaStatic) == hipSuccess) &&
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, fn, v.zeta_t, p.lds) == hipSuccess && occ >= 1;
        v.zeta_occ[exact] = ok ? occ : -1;
        if (!ok) {
            (void)hipGetLastError();     // (a refusal is no error of the launches that follow)
            return p;
        }
        v.zeta_dev = dev;
        v.zeta_cus = cus;
    }
    if (v.zeta_occ[exact] < 1) return p;
    p.dev = v.zeta_dev;
    p.cap = unit_budget(v.zeta_cus);
    const long cost = unit_parts(v.zeta_nwg, v.zeta_occ[exact]);
    if (cost <= p.cap) p.cost = cost;
    return p;
}

// A wait that expired costs the solve about 0.1 s, and what kept its
// workgroups apart (another process's work on the device) may last: the next
// solves are made with the two-kernel iteration, twice as many after each
// further expiry.
constexpr int kZetaBackFirst = 16, kZetaBackMost = 1024;
static void zeta_expired(Model &M) {
    M.solver_retries++;
    M.sv.zeta_back = std::min(kZetaBackMost, std::max(kZetaBackFirst, 2 * M.sv.zeta_back));
    M.sv.zeta_rest = M.sv.zeta_back;
}

// the launch, `tail` and the read-back of the control words; *done false
// when a wait expired
template <typename V>
static int zeta_run(Model &M, const ZetaPlan &p, SolvArgs<V> &a, const std::function<int()> &tail,
                    const std::function<int(const int *)> *after, int *c, bool *done) {
    ZetaArgs z;
    std::memset(&z, 0, sizeof z);
    z.nwg = M.sv.zeta_nwg; z.group = M.sv.zeta_group;
    z.hmax = M.sv.zeta_hmax; z.chmax = M.sv.zeta_chmax;
    z.lcol = M.m.z_lcol; z.hcol = M.m.z_hcol; z.hslot = M.m.z_hslot; z.hcnt = M.m.z_hcnt;
    z.send = M.m.z_send; z.nsend = M.sv.zeta_nsend;
    z.rows_f = M.m.fwd_rows; z.rows_b = M.m.bwd_rows;
    z.members = M.sv.zeta_members; z.dmax = M.sv.zeta_dmax;
    z.dent_f = M.m.z_dentf; z.dent_b = M.m.z_dentb; z.dptr_f = M.m.z_dptrf; z.dptr_b = M.m.z_dptrb;
    z.chunk_f = M.m.z_chf; z.chunk_b = M.m.z_chb; z.nch_f = M.m.z_nchf; z.nch_b = M.m.z_nchb;
    z.xch = M.sv.xch; z.pslot = M.sv.pslot;
    z.rhs = M.s.rhs; z.x = M.s.x; z.tol = M.p.refine_rtol; z.maxref = kMaxRefine; z.maxit = krylov_cap(M);
    z.spins = M.sv.zeta_spins >= 0 ? M.sv.zeta_spins : kSpinLimit;
    ZetaHold hold(p.dev, p.cost, p.cap);
    static_assert(kZetaSlotWords == (size_t)kZetaBufs * kPartCopies * kPartStride, "partial slots");
    hipLaunchKernelGGL(zeta_kernel<V>(M), dim3(M.sv.zeta_nwg), dim3(M.sv.zeta_t), p.lds, M.stream, a, z);
    HIPCHK(M, hipGetLastError());
    if (tail && tail()) return 1;
    if (read_ctrl(M, c, CT_WORDS, after, std::is_same<V, double>::value ? CT_CONV : CT_REFCONV)) return 1;
    *done = c[CT_CONV] || c[CT_REFCONV] || !c[CT_WAIT];
    if (*done) M.sv.zeta_back /= 2;
    else zeta_expired(M);
    return 0;
}

int solver_setup(Model &M) { (void)M; return 0; }

// the words of one zeta solve, for a second attempt at it
__global__ void k_ctrl_restart(int *ctrl) {
    if (threadIdx.x == 0) {
        ctrl[CT_FACTOR] = 0; ctrl[CT_ITS] = 0; ctrl[CT_NREF] = 0; ctrl[CT_REFCONV] = 0;
    }
}

// one zeta solve; fed: the row assembly already wrote its inputs (or a
// first attempt did)
static int solve_once(Model &M, int *iters, int *refinements, int wetdry_bnew, bool fed,
                      const std::function<int(const int *)> *after) {
    const int n = M.nkn;
    const int g1 = (n + kThreads - 1) / kThreads;
    int it_total = 0, nref = 0;
    // system_get + setweg(1) behind the solve, gated by its convergence flag
    auto wetdry = [&](const int *gate, const double *dx) -> int {
        if (wetdry_bnew < 0) return 0;
        timer_begin(M, T_WETDRY);
        const int rc = launch_system_get_setweg1(M, wetdry_bnew, gate, dx);
        timer_end(M);
        return rc;
    };
    if (M.prec == SHYHIP_FP64) {
        // initial guess = current level (system_solve passes znv); the Krylov
        // x0 vector is the FP64 solution array itself
        if (!fed) {
            hipLaunchKernelGGL(k_guess<double>, dim3(g1), dim3(kThreads), 0, M.stream, (const double *)M.s.zn, M.s.x,
                               n, M.sv.ctrl);
            hipLaunchKernelGGL(k_prep_matrix<double>, dim3((M.nnz + kThreads - 1) / kThreads), dim3(kThreads), 0,
                               M.stream, (const double *)M.s.aval, (const int *)M.m.csr_ell, (double *)M.sv.ell_a,
                               (float *)nullptr, M.nnz);
        }
        auto a = solv_args<double>(M, M.s.aval, M.s.rhs, M.s.x);
        if (factor<double>(M, a)) return 1;
        int its = 0;
        auto tail = [&]() -> int {
            // x = x0 + dx: inside system_get when it follows, else on its own
            if (wetdry_bnew >= 0) return wetdry(M.sv.ctrl + CT_CONV, a.dx);
            hipLaunchKernelGGL(k_bicg_finish<double>, dim3(g1), dim3(kThreads), 0, M.stream, (const double *)M.s.x,
                               (const double *)a.dx, M.s.x, n, 0, (const int *)M.sv.ctrl);
            HIPCHK(M, hipGetLastError());
            return 0;
        };
        int rc = 0;
        bool done = false;
        const ZetaPlan plan = zeta_plan<double>(M);
        if (plan.cost >= 0) {
            int c[CT_WORDS] = {};
            if (zeta_run<double>(M, plan, a, tail, after, c, &done)) return 1;
            if (done) rc = krylov_outcome(M, c, &its, 0);
        }
        if (!done) rc = bicgstab<double>(M, a, &its, 0, 0, tail);
        it_total = its;
        if (rc) return rc;
    } else {
        // FP32 BiCGStab on the FP32-rounded matrix inside FP64 refinement:
        // x <- x + A32^-1 (b - A64 x) until |b - A64 x| <= refine_rtol |b|;
        // each inner solve starts from a zero correction and runs at most
        // `chunk` iterations (a partial correction still refines).  The
        // rounds of the previous solve are enqueued at once; the flags are
        // read after them.
        float *a32 = (float *)M.sv.a32;
        if (!fed) {
            hipLaunchKernelGGL(k_guess_extrap, dim3(g1), dim3(kThreads), 0, M.stream, (const float *)M.s.zn,
                               (float *)M.sv.zprev, M.s.x, n, M.sv.ctrl, M.sv.have_prev ? 1 : 0);
            M.sv.have_prev = true;
            hipLaunchKernelGGL(k_prep_matrix<float>, dim3((M.nnz + kThreads - 1) / kThreads), dim3(kThreads), 0,
                               M.stream, (const double *)M.s.aval, (const int *)M.m.csr_ell, (float *)M.sv.ell_a, a32,
                               M.nnz);
        }
        float *b32 = (float *)M.sv.b, *x0 = (float *)M.sv.x0;
        auto a = solv_args<float>(M, a32, b32, x0);
        if (factor<float>(M, a)) return 1;
        a.rtol = M.p.inner_rtol;
        a.atol = 0.0;
        const int maxref = kMaxRefine;
        const int itmax_inner = krylov_cap(M);
        // iterations enqueued for round r: that round's count in the previous
        // solve plus one (kernels beyond convergence return at once but
        // still cost a launch); a round cut short by its chunk leaves a
        // partial correction and the next round continues from it
        auto chunk_of = [&](int r) {
            const int prev = r < CT_NRITS ? M.sv.round_its[r] : 0;
            const int c0 = prev > 0 ? prev + 1 : std::max(4, M.sv.last_its[1] + 3);
            return std::min(itmax_inner, std::max(2, c0));
        };
        auto resid = [&]() -> int {
            hipLaunchKernelGGL(k_resid64, dim3(g1), dim3(kThreads), 0, M.stream, M.m.rowptr, M.m.cols,
                               (const double *)M.s.aval, (const double *)M.s.rhs, (const double *)M.s.x, M.sv.r64,
                               b32, n, M.sv.part, M.sv.nparts, (const int *)M.sv.ctrl);
            hipLaunchKernelGGL(k_resid_check, dim3(1), dim3(kThreads), 0, M.stream, (const double *)M.sv.part,
                               M.sv.nparts, g1, M.sv.scal, M.sv.ctrl, M.p.refine_rtol);
            HIPCHK(M, hipGetLastError());
            return 0;
        };
        // boost: the rounds enqueued so far did not reach the target (their
        // chunks, sized from the previous solve, cut them short or the system
        // changed), so each later round gets twice the iterations of the last
        int plan = std::min((int)CT_NRITS, std::max(1, M.sv.last_nref)), enq = 0, c[CT_WORDS] = {}, boost = 1;
        const ZetaPlan zp = zeta_plan<float>(M);
        bool done = false;
        if (zp.cost >= 0) {
            auto tail = [&]() -> int { return wetdry(M.sv.ctrl + CT_REFCONV, nullptr); };
            if (zeta_run<float>(M, zp, a, tail, after, c, &done)) return 1;
            if (done) enq = maxref;       // all its rounds are behind it
        }
        for (;;) {
            if (!done) {
                for (int r = 0; r < plan && enq < maxref; r++, enq++) {
                    if (resid() || enqueue_inner<float>(M, a, std::min(itmax_inner, chunk_of(enq) * boost))) return 1;
                    hipLaunchKernelGGL(k_bicg_finish<float>, dim3(g1), dim3(kThreads), 0, M.stream, (const float *)x0,
                                       (const float *)a.dx, M.s.x, n, 1, (const int *)M.sv.ctrl);
                }
                if (resid()) return 1;
                if (wetdry(M.sv.ctrl + CT_REFCONV, nullptr)) return 1;
                if (read_ctrl(M, c, CT_WORDS)) return 1;
            }
            if (c[CT_FACTOR] != 0) {
                M.err = "zeta solver: zero pivot in the block factorisation (row " + std::to_string(c[CT_FACTOR]) + ")";
                return 2;
            }
            if (c[CT_REFCONV]) break;
            if (enq >= maxref) {
                double sc[16] = {};
                (void)hipMemcpyAsync(sc, M.sv.scal, sizeof sc, hipMemcpyDeviceToHost, M.stream);
                (void)hipStreamSynchronize(M.stream);
                std::string its;
                for (int r = 0; r < std::min((int)CT_NRITS, c[CT_NREF]); r++) its += " " + std::to_string(c[CT_RITS + r]);
                char buf[160];
                std::snprintf(buf, sizeof buf, " (|b - Ax| %.3e, |b| %.3e after %d rounds, %d iterations; first rounds:",
                              sc[SC_RES64], sc[SC_BNORM], c[CT_NREF], c[CT_ITS]);
                M.err = std::string("zeta solver: FP64 refinement did not reach the residual target") + buf + its + ")";
                return 2;
            }
            plan = 1;
            boost = std::min(2 * boost, 64);
        }
        nref = c[CT_NREF];
        it_total = c[CT_ITS];
        M.sv.last_nref = nref;
        M.sv.last_its[1] = nref > 0 ? (it_total + nref - 1) / nref : 0;
        for (int r = 0; r < CT_NRITS; r++) {
            const int its_r = r < nref ? c[CT_RITS + r] : 0;
            // a round cut short by its chunk gets more next time
            M.sv.round_its[r] = its_r < 0 ? 2 - its_r : its_r;
        }
    }
    if (iters) *iters = it_total;
    if (refinements) *refinements = nref;
    return 0;
}

// The block factors are refined from the previous solve's (warm) except on
// the first solve and every kWarmRefresh-th, which factorise exactly.  A
// solve that fails with refined factors (a matrix that changed too much for
// the sweeps: rows switched by wetting and drying) is done again with exact
// factors from where it stopped, so the warm start can cost iterations but
// never a solve.
int solver_solve(Model &M, int *iters, int *refinements, int wetdry_bnew,
                 const std::function<int(const int *)> *after) {
    // inputs already written by the row assembly of this step's system?
    const bool fed = M.sv.fed;
    M.sv.fed = false;
    if (++M.sv.solves_since_exact >= kWarmRefresh) M.sv.have_lu = false;
    const int rc = solve_once(M, iters, refinements, wetdry_bnew, fed, after);
    if (rc != 2 || !M.sv.last_warm) return rc;
    M.solver_retries++;
    M.sv.have_lu = false;
    hipLaunchKernelGGL(k_ctrl_restart, dim3(1), dim3(64), 0, M.stream, M.sv.ctrl);
    HIPCHK(M, hipGetLastError());
    M.err.clear();
    return solve_once(M, iters, refinements, wetdry_bnew, true, after);
}

}  // namespace shy

// pcg.hip -- Jacobi-PCG for gfx950: FP64 (reference op order) and the
// mixed form (FP32 inner iteration, FP64 residual replacement).
//
// Reference loop (src/fcgalg/cel_cgalg_module.f90:206-304):
//   r = b - A x ; p = jac*r ; alpha = r.p ; norm2 = ||r||
//   while k < iter_max and |alpha| > 1.1 eps_mach and norm2 > eps:
//     v = A p ; k++ ; sigma = alpha / (v.p)
//     x = x + sigma p ; r = r + (-sigma) v ; z = jac*r
//     beta = (r.z)/alpha ; alpha = r.z ; p = beta p + z ; norm2 = ||r||
//
// One iteration is three streaming kernels:
//   K1  v = A p (LDS-staged CSR tile, DIA rows or JAD), one partial of v.p
//       per block
//   K2  sigma = alpha / sum(v.p) ; r = r + (-sigma) v ; z = jac*r ;
//       partials of r.z and r.r
//   K3  beta = sum(r.z)/alpha ; x = x + sigma p ; p = beta p + jac*r ;
//       alpha, norm2, k, loop decision
// (the x update sits in K3 because K3 reads p anyway; x never feeds back
// into the iteration and each element is the reference's formula).
//
// No kernel waits on another block of the same launch: there are no grid
// barriers, atomics or device-scope fences in the loop.  The scalars travel
// as a small token along the ring of kernels -- every kernel reads the token
// its predecessor wrote and block 0 writes the token for its successor -- and
// a kernel that needs a dot product sums the predecessor's per-block
// partials itself, in every block, in the same fixed order.  All blocks
// therefore hold bit-identical scalars, the sums do not depend on which
// block finished first, and the device never waits for the host, which
// stays a few iterations ahead by a progress word in its own memory.  A
// stopped token is forwarded unchanged, so a captured chunk of iterations
// can be replayed as a hipGraph and runs past convergence as no-ops.
//
// Per element the arithmetic is the reference's (products rounded before the
// add, -ffp-contract=off); only the summation order of the dot products
// differs from the reference (fixed tree here, worker chunks there).
#include <algorithm>
#include <chrono>
#include <cmath>
#include <thread>
#include <vector>

#include "cel_internal.hpp"
#include "spmv_device.hpp"

namespace cel {

// Token passed along the kernel ring.
struct Ctrl {
    double alpha, sigma, beta, norm2, eps, norm0, bnorm, rnorm_ref;
    int run;     // 1 while the loop continues
    int iter;    // completed iterations
    int status;  // 0 or a CEL_ERR_* code
    int reduce;  // partials the next K1 must fold in first: 0 none, 1 set-up, 2 replacement
    int ru;      // mixed: replace the residual at the end of this iteration
    int outer;   // mixed: replacements done
    int since;   // mixed: iterations since the last replacement
    int stall;   // mixed: consecutive replacements that did not halve the FP64 residual
    int slots;   // finished slots (launch groups of one iteration or replacement)
    int pad;
};

// Constant solver parameters.
struct Prm {
    double tol, small, ru_delta;
    int tol_mode, iter_max, ru_restart, hist_cap, alpha_stop, ru_max_inner;
    double* hist;
};

// the reference's absolute test |alpha| > 1.1 eps_mach (optional)
__device__ __forceinline__ bool alpha_ok(const Prm& P, double alpha)
{
    return !P.alpha_stop || fabs(alpha) > P.small;
}

enum { kReduceNone = 0, kReduceSetup = 1, kReduceReplace = 2 };

// ------------------------------------------------------------------ helpers
__device__ __forceinline__ double eps_from(const Prm& P, double bnorm, double r0)
{
    if (P.tol_mode == CEL_TOL_REL_B) return P.tol * bnorm;
    if (P.tol_mode == CEL_TOL_REL_R0) return P.tol * r0;
    return P.tol;
}

// Every thread of the block reads the token (written by the previous kernel).
// Field by field: as one struct copy, the fields a kernel only forwards stay
// in a private array, which the compiler moves to LDS and indexes with the
// work-group sizes of the dispatch packet -- a read of host memory that held
// every launch of more than 64 blocks back by 12 us (an otherwise empty
// kernel that copies the token: 14.7 us so, 2.6 us field by field).
__device__ __forceinline__ Ctrl read_ctrl(const Ctrl* __restrict__ p)
{
    Ctrl c;
    c.alpha = p->alpha;
    c.sigma = p->sigma;
    c.beta = p->beta;
    c.norm2 = p->norm2;
    c.eps = p->eps;
    c.norm0 = p->norm0;
    c.bnorm = p->bnorm;
    c.rnorm_ref = p->rnorm_ref;
    c.run = p->run;
    c.iter = p->iter;
    c.status = p->status;
    c.reduce = p->reduce;
    c.ru = p->ru;
    c.outer = p->outer;
    c.since = p->since;
    c.stall = p->stall;
    c.slots = p->slots;
    c.pad = 0;
    return c;
}

__device__ __forceinline__ void write_ctrl(Ctrl* __restrict__ dst, const Ctrl& c)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        dst->alpha = c.alpha;
        dst->sigma = c.sigma;
        dst->beta = c.beta;
        dst->norm2 = c.norm2;
        dst->eps = c.eps;
        dst->norm0 = c.norm0;
        dst->bnorm = c.bnorm;
        dst->rnorm_ref = c.rnorm_ref;
        dst->run = c.run;
        dst->iter = c.iter;
        dst->status = c.status;
        dst->reduce = c.reduce;
        dst->ru = c.ru;
        dst->outer = c.outer;
        dst->since = c.since;
        dst->stall = c.stall;
        dst->slots = c.slots;
        dst->pad = c.pad;
    }
}

// End of a slot, in its last kernel: the token, and the host's progress
// word (may be null): slots finished, or -1 once the solve has stopped.
__device__ __forceinline__ void end_slot(Ctrl* __restrict__ dst, Ctrl& c, int* progress)
{
    c.slots = c.slots + 1;
    write_ctrl(dst, c);
    if (progress && blockIdx.x == 0 && threadIdx.x == 0)
        __hip_atomic_store(progress, c.run ? c.slots : -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// A fresh token.
__global__ void k_token(Ctrl* c)
{
    Ctrl t{};
    t.run = 1;
    write_ctrl(c, t);
}

// Sum of G partials in fixed order, returned to every thread of the block.
// red: as block_sum_all.
__device__ __forceinline__ double all_sum(const double* __restrict__ part, int G, double* red)
{
    return block_sum_all(strided_sum(part, G), red);
}

// Two folds at once, each in all_sum's order, from the threads' parts.
__device__ __forceinline__ void all_sum2(double sa, double sb, double* red /* 2*kWaves */, double& a, double& b)
{
    sa = wave_sum(sa);
    sb = wave_sum(sb);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) {
        red[wave] = sa;
        red[kWaves + wave] = sb;
    }
    __syncthreads();
    a = b = 0.0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        a = a + red[w];
        b = b + red[kWaves + w];
    }
}

// Balanced contiguous ranges: logical block lb of G owns units [u0, u1).
__device__ __forceinline__ void unit_range(long long nunits, int G, int lb, long long& u0,
                                           long long& u1)
{
    u0 = nunits * lb / G;
    u1 = nunits * (lb + 1) / G;
}

// ------------------------------------------------------------------ set-up
__global__ void k_fill(long long n, double* __restrict__ x, double v)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        x[i] = v;
}

// dst[k] = src[perm[k]] (to the permuted row order) and back
template <typename T>
__global__ void k_perm_gather(long long n, const int* __restrict__ perm, const T* __restrict__ src,
                              T* __restrict__ dst)
{
    for (long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x; k < n;
         k += (long long)gridDim.x * blockDim.x)
        dst[k] = src[perm[k]];
}

template <typename T>
__global__ void k_perm_scatter(long long n, const int* __restrict__ perm, const T* __restrict__ src,
                               T* __restrict__ dst)
{
    for (long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x; k < n;
         k += (long long)gridDim.x * blockDim.x)
        dst[perm[k]] = src[k];
}

struct MatView {
    int n, mmax;
    int coo;  // the local block is applied as COO: v(row) += a p entry by entry from v = 0
    long long jnnz;
    const int *xadj, *cols;
    const double* vals;
    const float* vals32;
    const int *jbegin, *jcols, *jperm;
    const double* jvals;
    const float* jvals32;
    // DIA: values [nd][n], presence mask, ascending offsets
    const double* dvals;
    const float* dvals32;
    const uint32_t* dmask;   // presence bits, more than 8 diagonals
    const uint8_t* dmask8;   // presence bits, at most 8 diagonals
    int nd;
    int dzero;               // index of the diagonal with offset 0, or -1
    int doff[32];
    int dwide;                    // the K1 walks the diagonals with several rows per lane
    long long dbase[kClassDiag];  // then entry (i, d) is dvals[dbase[d] + i] (dia_bases)
    // row classes (rowclass.hip), with the diagonals above
    const uint8_t* cls;
    RowClasses ctab;
    int band;         // window K1s: the largest |column - row|
    const int* walk;  // by K1 block, wide walks: the walk it takes (null: its own)
    // halo (FP64 only)
    const int *hrow_tile, *hrows, *hrowq, *hptr, *hcols;
    const double* hvals;
    const double* ghost;
    const double* hrec;     // per compact halo row: {p1, p2}
    const uint8_t* hflag;   // per row: min(halo entries, 255); hflag[n] = 0
    const int* hwq;         // per 64-row group: compact index of its first halo row
    int hnq;                // rows with halo entries
};

// The halo records of this SpMV (after the ghost values arrived; here
// after the face pack): one thread per row with halo entries, in compact
// order.
__global__ __launch_bounds__(kBlock) void k_halo_rec(int nq, const int* __restrict__ hptr,
                                                     const int* __restrict__ hcols,
                                                     const double* __restrict__ hvals,
                                                     const double* __restrict__ ghost,
                                                     double* __restrict__ rec,
                                                     const Ctrl* __restrict__ cin)
{
    if (!cin->run) return;  // uniform: the iteration does not run
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nq) return;
    const int j0 = hptr[q];
    const int c = hptr[q + 1] - j0;
    double w[kHaloRec] = {0.0, 0.0};
#pragma unroll
    for (int k = 0; k < kHaloRec; ++k)
        if (k < c) w[k] = hvals[j0 + k] * ghost[hcols[j0 + k]];
    double* o = rec + 2 * (size_t)q;  // compact: the K1s find q from their wavefront
    o[0] = w[0];
    o[1] = w[1];
}

template <typename VT>
__device__ __forceinline__ const VT* csr_vals(const MatView& A);
template <>
__device__ __forceinline__ const double* csr_vals<double>(const MatView& A) { return A.vals; }
template <>
__device__ __forceinline__ const float* csr_vals<float>(const MatView& A) { return A.vals32; }
template <typename VT>
__device__ __forceinline__ const VT* dia_vals(const MatView& A);
template <>
__device__ __forceinline__ const double* dia_vals<double>(const MatView& A) { return A.dvals; }
template <>
__device__ __forceinline__ const float* dia_vals<float>(const MatView& A) { return A.dvals32; }

// A solve's matrix as row classes: a form of its own beside CEL_FMT_*.
constexpr int kFmtClass = 64;

template <typename VT>
__device__ __forceinline__ void load_classes(const MatView& A, ClassTab<VT>& t);
template <>
__device__ __forceinline__ void load_classes<double>(const MatView& A, ClassTab<double>& t)
{
    t.load(A.ctab.val64, A.ctab.mask);
}
template <>
__device__ __forceinline__ void load_classes<float>(const MatView& A, ClassTab<float>& t)
{
    t.load(A.ctab.val32, A.ctab.mask);
}

// The LDS a form's tile walk uses.
template <typename VT, int FMT, bool LONG>
struct StageOf {
    using T = typename CsrStreamOf<VT, LONG>::Stage;
};
template <typename VT, bool LONG>
struct StageOf<VT, kFmtClass, LONG> {
    using T = ClassTab<VT>;
};
struct NoStage {};
template <typename VT, bool LONG>
struct StageOf<VT, CEL_FMT_DIA, LONG> {
    using T = NoStage;
};

template <typename VT>
__device__ __forceinline__ const VT* jad_vals(const MatView& A);
template <>
__device__ __forceinline__ const double* jad_vals<double>(const MatView& A) { return A.jvals; }
template <>
__device__ __forceinline__ const float* jad_vals<float>(const MatView& A) { return A.jvals32; }

// Walks the tiles [t0, t1) of one block in the requested format and
// returns, per tile, the calling thread's row sum and its row.  For CSR
// row = r0 + tid (the next tile's loads are issued while this tile's
// gathers wait); for JAD row = perm[r0 + tid].  HALO adds the halo entries
// after the local sum ((0 + local) + halo...).  With xrow, x[row] is
// loaded too (before the next tile's loads).  next() contains
// __syncthreads() for CSR: every thread of the block calls it.
template <typename VT, typename AT, int FMT, bool HALO, bool LONG>
struct TileWalk {
    using Stage = typename StageOf<VT, FMT, LONG>::T;
    typename CsrStreamOf<VT, LONG>::Stream cs;

    // Contains __syncthreads() for CSR: every thread of the block calls it.
    __device__ __forceinline__ void start(const MatView& A, long long t0, long long t1, Stage& sm)
    {
        if constexpr (FMT == CEL_FMT_CSR) {
            if (t0 < t1)  // uniform across the block
                cs.open(A.n, (int)t0, t0 + 1 < t1 ? (int)t0 + 1 : -1, A.xadj, A.cols,
                        csr_vals<VT>(A), sm);
        }
        if constexpr (FMT == kFmtClass) load_classes<VT>(A, sm);
    }

    __device__ __forceinline__ AT next(const MatView& A, long long t, long long t1,
                                       const VT* __restrict__ x, Stage& sm, int& row, VT* xrow)
    {
        const int r0 = (int)t * kTileRows;
        AT s;
        if constexpr (FMT == CEL_FMT_CSR) {
            const int nxt = (t + 1 < t1) ? (int)(t + 1) : -1;
            const int aft = (t + 2 < t1) ? (int)(t + 2) : -1;
            row = r0 + threadIdx.x;
            s = cs.template rows<AT>(A.n, (int)t, nxt, aft, A.xadj, A.cols, csr_vals<VT>(A), XPlain<VT>{x}, sm,
                                     row, xrow);
            cs.advance(nxt, sm);
            // CSR: r = 0; r = r + tmp.  COO: the entries were added to 0 one
            // by one (the same bits but for the sign of a zero sum)
            s = A.coo ? s : AT(0) + s;
            if constexpr (HALO) {
                if (row < A.n)
                    s = halo_row<AT>(row, (int)t, s, A.hrow_tile, A.hrows, A.hptr, A.hcols,
                                     A.hvals, A.ghost);
            }
        } else if constexpr (FMT == kFmtClass) {
            row = r0 + threadIdx.x;
            s = AT(0);
            if (row < A.n) {
                const int r[1] = {row};
                VT sum[1];
                class_rows<VT, 1>(A.n, A.nd, A.doff, A.cls, sm, r, XPlain<VT>{x}, sum);
                s = AT(0) + sum[0];
            }
        } else {
            // JAD solves keep their vectors in the permuted row order, with
            // the columns renumbered into it: row k of the permuted system
            const int k = r0 + threadIdx.x;
            s = AT(0);
            row = A.n;
            if (k < A.n) {
                VT xr = VT(0);
                if (xrow) xr = x[k];
                s = jad_row<VT, AT>(k, A.mmax, A.jbegin, A.jcols, jad_vals<VT>(A), x);
                row = k;
                if (xrow) *xrow = xr;
            }
        }
        return s;
    }
};

// ------------------------------------------------------------------ residual
// r = b - A x with the FP64 operator; per-block partials: r.z, r.r, b.b.
// FP64 form: r and p = z = jac*r stored in FP64.  Mixed form (OUT_T =
// float): r rounded to FP32, z = jac32 * r32 (p = z at the start or on a
// restart), e = 0 at the start, the norm taken in FP64 before rounding.
// The next K1 folds the partials into the token.
template <typename OUT_T>
struct ResArgs {
    const double *x, *b, *jac;
    const float* jac32;
    OUT_T *r, *p;
    float* e;
    double* part;
    int G;  // blocks of the partials
};

// Block lb of a.G: its contiguous tiles and its partials.
template <typename OUT_T, int FMT, bool HALO, bool REPLACE, bool LONG>
__device__ __forceinline__ void residual_block(const MatView& A, const ResArgs<OUT_T>& a, int lb,
                                               bool restart, typename StageOf<double, FMT, LONG>::T& sm,
                                               double* red /* 3*kWaves */)
{
    const int G = a.G;
    const long long ntiles = (A.n + kTileRows - 1) / kTileRows;
    long long t0, t1;
    unit_range(ntiles, G, lb, t0, t1);
    double arz = 0.0, arr = 0.0, abb = 0.0;
    TileWalk<double, double, FMT, HALO, LONG> walk;
    walk.start(A, t0, t1, sm);
    for (long long t = t0; t < t1; ++t) {
        int row;
        double s = walk.next(A, t, t1, a.x, sm, row, nullptr);
        if (row < A.n) {
            const double bi = a.b[row];
            const double ri = bi - s;  // r = 0; r = r + A x; r = b - r
            double bb = bi * bi;  // a non-finite b makes this sum non-finite
            abb = abb + bb;
            double rr = ri * ri;
            arr = arr + rr;
            if constexpr (sizeof(OUT_T) == 8) {
                const double zi = ri * a.jac[row];
                a.r[row] = ri;
                a.p[row] = zi;
                double rz = ri * zi;
                arz = arz + rz;
            } else {
                const float rf = (float)ri;
                const float zf = rf * a.jac32[row];
                a.r[row] = rf;
                if (!REPLACE || restart) a.p[row] = zf;
                if (!REPLACE) a.e[row] = 0.0f;
                double rz = (double)rf * (double)zf;
                arz = arz + rz;
            }
        }
    }
    block_sum2(arz, arr, red);
    const double sbb = block_sum(abb, red + 2 * kWaves);
    if (threadIdx.x == 0) {
        a.part[lb] = arz;
        a.part[G + lb] = arr;
        a.part[2 * G + lb] = sbb;
    }
}

// Set-up of a solve: r0, p0, partials.
template <typename OUT_T, int FMT, bool HALO, bool LONG>
__global__ __launch_bounds__(kBlock) void k_residual(MatView A, ResArgs<OUT_T> a,
                                                     const Ctrl* __restrict__ cin,
                                                     Ctrl* __restrict__ cout)
{
    Ctrl c = read_ctrl(cin);
    __shared__ typename StageOf<double, FMT, LONG>::T sm;
    __shared__ double red[3 * kWaves];
    residual_block<OUT_T, FMT, HALO, false, LONG>(A, a, logical_block(), false, sm, red);
    c.reduce = kReduceSetup;
    c.ru = 0;
    write_ctrl(cout, c);
}

// Mixed form, requested replacement (token's ru): the FP64 residual in place
// of the product of a K1 launch.  The K1's blocks share the a.G blocks of
// the partials (the set-up's grid, so the sums are grouped alike).  A
// launch of its own per iteration, almost always with nothing to do, cost
// 1 us at 32^3 (mixed 15.2 against 14.4 us per iteration) to 7 us on larger
// grids (600k-row mesh solve 9.13 against 8.80 ms).
template <int FMT, bool LONG>
__device__ __forceinline__ void replace_residual(const MatView& A, const ResArgs<float>& a, Ctrl& c,
                                                 const Prm& P, typename StageOf<double, FMT, LONG>::T& sm,
                                                 double* red)
{
    for (int vb = blockIdx.x; vb < a.G; vb += gridDim.x) {
        const int lb = a.G % kXcds ? vb : (vb % kXcds) * (a.G / kXcds) + vb / kXcds;
        residual_block<float, FMT, false, true, LONG>(A, a, lb, P.ru_restart, sm, red);
        __syncthreads();  // the stage is free again
    }
    c.reduce = kReduceReplace;
    c.ru = 0;
}

// The CSR, DIA and JAD K1s walk their tiles in group_tile's order
// (spmv_device.hpp).  The CSR and DIA K1s add a thread's rows to the block
// partial in that order, so their partials and solves are bit-identical;
// the JAD K1's tiles hold permuted rows, so it shares only the order of the
// tiles, and its solves agree with the others to rounding.  (Groups of 4
// tiles measured: FP64 DIA solve 1% faster, mixed DIA 1% slower.)

// Folds pending set-up or replacement partials into the token (every block,
// same order) and decides whether the iteration runs.
__device__ __forceinline__ void fold_pending(Ctrl& c, const double* __restrict__ rpart, int Gr,
                                             const Prm& P, double* red /* 2*kWaves */)
{
    double rz, rr;
    all_sum2(strided_sum(rpart, Gr), strided_sum(rpart + Gr, Gr), red, rz, rr);
    const double rn = sqrt(rr);
    __syncthreads();
    if (c.reduce == kReduceSetup) {
        const double bb = all_sum(rpart + 2 * Gr, Gr, red);
        c.bnorm = sqrt(bb);
        c.norm0 = rn;
        c.eps = eps_from(P, c.bnorm, rn);
        c.iter = 0;
        c.outer = 0;
        if (!isfinite(bb) && c.status == 0) c.status = CEL_ERR_NONFINITE;
        if (blockIdx.x == 0 && threadIdx.x == 0 && P.hist_cap > 0) P.hist[0] = rn;
    } else {
        c.outer = c.outer + 1;
        // attainable accuracy: two cycles in a row that fail to halve the
        // FP64 residual end the solve (not converged)
        c.stall = (rn > 0.5 * c.rnorm_ref) ? c.stall + 1 : 0;
    }
    c.since = 0;
    c.alpha = rz;
    c.norm2 = rn;
    c.rnorm_ref = rn;
    c.reduce = kReduceNone;
    c.run = (c.status == 0 && c.iter < P.iter_max && alpha_ok(P, c.alpha) &&
             c.norm2 > c.eps && c.stall < 2)
                ? 1
                : 0;
}

// The scalars after r.z and r.r of an iteration: beta, alpha = r.z, norm2,
// k++, history, loop decision (FP64) or replacement request (mixed).
template <bool MIXED>
__device__ __forceinline__ void next_scalars(Ctrl& c, double rz, double rr, const Prm& P)
{
    c.beta = rz / c.alpha;
    c.alpha = rz;
    c.norm2 = sqrt(rr);
    c.iter = c.iter + 1;
    if (blockIdx.x == 0 && threadIdx.x == 0 && c.iter < P.hist_cap) P.hist[c.iter] = c.norm2;
    if (!MIXED) {
        c.run = (c.iter < P.iter_max && alpha_ok(P, c.alpha) && c.norm2 > c.eps) ? 1 : 0;
    } else {
        // replace the FP32 residual by the FP64 one when it has dropped by
        // ru_delta since the last replacement, looks converged, the budget
        // is spent, or the FP32 recurrence has stopped tracking the FP64
        // residual (grown past it, or a cycle far longer than expected);
        // the stop decision is taken on the FP64 norm
        c.since = c.since + 1;
        const bool drop = c.norm2 < P.ru_delta * c.rnorm_ref;
        const bool astray = c.norm2 > 2.0 * c.rnorm_ref || c.since >= P.ru_max_inner;
        c.ru = (drop || astray || c.norm2 <= c.eps || c.iter >= P.iter_max ||
                !alpha_ok(P, c.alpha) || !isfinite(c.norm2))
                   ? 1
                   : 0;
    }
}

// Most tile groups a wide walk sums per step: with 2, the four waves have one
// 16-byte task each in FP32 and two in FP64.
constexpr int kWideGroups = 2;

// What the tile walk of a K1 does with the rows besides the product: nothing,
// or (k_pcg_step) p_new and x += sigma p of the thread's rows.
template <typename VT>
struct StepRows {
    VT* pout;
    VT* x;
    VT sigma;
    bool upd;  // x is updated (uniform; false right after a set-up or replacement)
};

// LDS of a wide walk: the rows' terms of v.d, two steps of them.
struct WideStage {
    double prod[2][kWideGroups * kTileGroup * kTileRows];
};
template <int FMT, bool HALO, bool STEP>
constexpr bool wide_form = FMT == kFmtClass || (FMT == CEL_FMT_DIA && !HALO && !STEP);
template <bool WIDE>
struct WideStageOf {
    using T = NoStage;
};
template <>
struct WideStageOf<true> {
    using T = WideStage;
};

// k1_tiles of row classes and of symmetric diagonal storage: v = A d with E =
// 16 / sizeof(VT) consecutive rows per lane.  What bounds a product of so few
// bytes per row (classes: x, v and a byte) is the work per row: one row per
// lane took 7 loads, 8 LDS reads and 90 instructions, 56.6 us on the 256^3
// block in FP32 (151 MB); this one takes 7/4 loads, 3 LDS reads and 45
// instructions, 35.8 us (4.2 TB/s).  The rows of a step are those of the
// row-per-thread kernels (NG groups of kTileGroup tiles) and their terms of
// v.d go through LDS to the threads that add them there, so the partials are
// the same bit for bit.  Waves that hold a row without all of its neighbours
// in [0, n) (the ends of the matrix) take loads that are checked one by one
// (edge).  AHEAD: the next step's loads are issued before the sums of this
// one, into a second set of registers: for diagonals in FP64, whose loads are
// memory's (200^3 192 us per iteration without, 181 with); by classes it
// measured slower (FP64 100^3 27.8 against 28.9 us), in FP32 it spills (K1 of
// 256^3 50 us).
// Per iteration, before and after, classes: mixed 256^3 150.6 -> 130.2 us,
// 200^3 79.5 -> 68.5, 128^3 30.5 -> 29.8, 100^3 23.7 -> 23.7; FP64 256^3 283
// -> 244, 200^3 141 -> 120, 128^3 47 -> 43, 100^3 28.7 -> 27.5.  Symmetric
// diagonals: FP64 256^3 454 -> 407, 200^3 208 -> 181, 128^3 58.3 -> 51.8,
// 820,911 rows 29.5 -> 27.2; mixed 128^3 36.7 -> 33.0.
template <typename VT, int ND, int NG, bool AHEAD, typename SRC, typename EDGE>
__device__ __forceinline__ double k1_wide(const MatView& A, const VT* __restrict__ x, VT* __restrict__ v,
                                          const SRC& src, const EDGE& edge, WideStage& st, int walk)
{
    constexpr int E = WideOf<VT>::E, WR = 64 * E;        // rows of a wave's task
    constexpr int GR = kTileGroup * kTileRows;           // rows of a group
    constexpr int WPG = GR / WR, U = NG * WPG / kWaves;  // tasks of a group, and of a wave per step
    static_assert(NG <= kWideGroups && NG * WPG % kWaves == 0 && GR % WR == 0, "whole tasks");
    using V = typename WideOf<VT>::T;
    const long long ngroups = ((long long)A.n + GR - 1) / GR, G = gridDim.x;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int omin = min(0, A.doff[0]), omax = max(0, A.doff[A.nd - 1]);
    // the first rows that have all neighbours, as a multiple of E: what a task
    // loads that is summed row by row (loads under a branch would be waited
    // for at its end)
    const int safe = (-omin + E - 1) / E * E;
    struct Step {
        WideRows<VT, ND, U, SRC> R;
        V xr[U];
        int row[U];
        bool inside;  // uniform across the wave
    };
    // the u-th task of the step at q: its first row, and the place of its terms
    auto first_row = [&](long long q, int u) -> long long {
        const int task = u * kWaves + wave;
        return (q + task / WPG * G) * GR + task % WPG * WR;
    };
    auto place = [&](int u) { return (u * kWaves + wave) * WR + lane * E; };
    auto fetch = [&](long long q, Step& T) {
        T.inside = true;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const long long w0 = first_row(q, u);
            T.inside = T.inside && w0 + omin >= 0 && w0 + WR + omax <= A.n;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) T.row[u] = (T.inside ? (int)first_row(q, u) : safe) + lane * E;
        T.R.load(T.row, A.doff, x, src);
#pragma unroll
        for (int u = 0; u < U; ++u) T.xr[u] = ld_at<V>(x, (unsigned)T.row[u] * (unsigned)sizeof(VT));
    };
    double acc = 0.0;
    int buf = 0;
    auto sum = [&](long long q, const Step& T) {
        double* prod = st.prod[buf];
        buf ^= 1;
        if (T.inside) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                V vv;
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    const VT s = T.R.sum(u, e, src);
                    vv[e] = s;
                    prod[place(u) + e] = double(s) * double(T.xr[u][e]);
                }
                *reinterpret_cast<V*>(v + T.row[u]) = vv;
            }
        } else {
#pragma unroll 1
            for (int u = 0; u < U; ++u) {
                const long long r0 = first_row(q, u) + lane * E;
                int r[E];
                VT s[E], pr[E];
#pragma unroll
                for (int e = 0; e < E; ++e) r[e] = (int)min(r0 + e, (long long)A.n);
                if (r[0] < A.n) edge(r, s, pr);
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    double t = 0.0;
                    if (r[e] < A.n) {
                        const VT d = A.dzero >= 0 ? pr[e] : x[r[e]];
                        const VT sk = VT(0) + s[e];
                        v[r[e]] = sk;
                        t = double(sk) * double(d);
                    }
                    prod[place(u) + e] = t;
                }
            }
        }
        __syncthreads();  // one per step: the next one writes the other half
#pragma unroll
        for (int k = 0; k < NG * kTileGroup; ++k) acc = acc + prod[k * kTileRows + threadIdx.x];
    };
    if ((long long)safe + WR + omax > A.n) {  // no such rows (uniform across the grid)
        Step T;
        T.inside = false;
        for (long long q = walk; q < ngroups; q += NG * G) sum(q, T);
    } else if constexpr (!AHEAD) {
        for (long long q = walk; q < ngroups; q += NG * G) {
            Step T;
            fetch(q, T);
            sum(q, T);
        }
    } else {
        // two sets of registers by turns: a copy would wait for the loads
        Step T0, T1;
        if (walk < ngroups) fetch(walk, T0);
        for (long long q = walk; q < ngroups; q += 2 * NG * G) {
            fetch(q + NG * G, T1);
            __builtin_amdgcn_sched_barrier(0);
            sum(q, T0);
            if (q + NG * G >= ngroups) break;
            fetch(q + 2 * NG * G, T0);
            __builtin_amdgcn_sched_barrier(0);
            sum(q + NG * G, T1);
        }
    }
    return acc;
}

// The tile stream of a step's CSR walk.  In FP64 it is opened (a tile's entries
// to LDS) before the step's scalars are there: per iteration, after / before
// them, FP64 20^3 11.2 / 10.7 us, 32^3 11.35 / 10.9, 64^3 15.1 / 14.6; in the
// mixed form, whose registers it takes, 32^3 12.7 / 13.0, 64^3 14.4 / 14.6.
template <typename VT>
constexpr bool kOpenAhead = sizeof(VT) == 8;
template <typename VT, int FMT, bool LONG, bool KEEP>
struct StepStream {
    __device__ __forceinline__ void open(const MatView&, typename StageOf<VT, FMT, LONG>::T&) {}
};
template <typename VT, bool LONG, bool KEEP>
struct StepStream<VT, CEL_FMT_CSR, LONG, KEEP> {
    typename CsrStreamOf<VT, LONG, KEEP>::Stream cs;
    __device__ __forceinline__ void open(const MatView& A, typename CsrStreamOf<VT, LONG>::Stage& sm)
    {
        const long long ntiles = (A.n + kTileRows - 1) / kTileRows;
        const int t = (int)group_tile(0, ntiles);
        if (t >= 0)  // uniform across the block
            cs.open(A.n, t, (int)group_tile(1, ntiles), A.xadj, A.cols, csr_vals<VT>(A), sm);
    }
};

// v = A d over the block's tiles, d the vector of the accessor X; returns the
// thread's part of v.d.  STEP: X is XDirection, and d and the updated x of
// every row are stored as well.  (Taking a step's scalars behind the first
// tile's gathers instead of before them measured slower, 32^3 12.7 against
// 12.3 us per iteration.)  KEEP: keep_matrix(); TAIL: deep_rows().
template <typename VT, int FMT, bool HALO, bool LONG, bool STEP, bool KEEP, int TAIL, typename X>
__device__ __forceinline__ double k1_tiles(const MatView& A, const X& x, VT* __restrict__ v,
                                           StepStream<VT, FMT, LONG, KEEP>& first,
                                           typename StageOf<VT, FMT, LONG>::T& sm,
                                           typename WideStageOf<wide_form<FMT, HALO, STEP>>::T& wide,
                                           const StepRows<VT>& st, int walk = 0)
{
    const long long ntiles = (A.n + kTileRows - 1) / kTileRows;
    double acc = 0.0;
    static_assert(!(STEP && FMT == kFmtClass), "large systems only");
    // one finished row: its value, and in a step its direction and x
    auto finish = [&](int row, VT s, const typename X::Raw& raw, VT xo) {
        const VT d = x.value(raw);
        v[row] = s;
        if constexpr (STEP) {
            st.pout[row] = d;
            if (st.upd) {
                const VT t = st.sigma * raw.p;
                st.x[row] = xo + t;
            }
        }
        double prod = double(s) * double(d);
        acc = acc + prod;
    };
    if constexpr (FMT == CEL_FMT_CSR) {
        // halo rows (HALO): a row's halo record (count and products, in
        // block order) is added after its local sum.  Its flag loads one
        // step ahead, behind the previous tile's entries; the record loads
        // in the row's own step, behind the gathers (so the wait for the
        // gathers does not include it) and ahead of the next tile's entries
        // (whose wait, for the stage, covers it).  Unflagged rows load no
        // record and read count 0.  Each loaded value is used once in the
        // step after it, in place: a copy of a register still being loaded
        // would wait for every load issued before it.
        typename CsrStreamOf<VT, LONG, KEEP, TAIL>::Stream own;
        auto& cs = [&]() -> auto& {
            if constexpr (STEP && kOpenAhead<VT>) return first.cs;
            else return own;
        }();
        const VT* vals = csr_vals<VT>(A);
        const long long tfirst = group_tile(0, ntiles);
        const auto rrec = tile_rsrc(HALO ? A.hrec : nullptr, HALO ? A.hnq * 16 : 0);
        // flag index of this thread's row of tile t (rows past n read hflag[n] = 0)
        auto fidx = [&](long long t) {
            const long long r = t * kTileRows + threadIdx.x;
            return t >= 0 && r < A.n ? (int)r : A.n;
        };
        // the halo flag (entry count) of this thread's row of the tile being
        // summed, and its wavefront's first compact halo index
        int hf = 0, hq = 0;
        if (tfirst >= 0) {  // uniform across the block
            if constexpr (HALO) {
                hf = A.hflag[fidx(tfirst)];
                hq = A.hwq[fidx(tfirst) >> 6];
            }
            if constexpr (!(STEP && kOpenAhead<VT>)) cs.open(A.n, (int)tfirst, (int)group_tile(1, ntiles), A.xadj, A.cols, vals, sm);
        }
        long long k = 0;
        for (long long t = tfirst; t >= 0; t = group_tile(++k, ntiles)) {
            const int nxt = (int)group_tile(k + 1, ntiles);
            const int aft = (int)group_tile(k + 2, ntiles);
            const int row = (int)t * kTileRows + threadIdx.x;
            typename X::Raw pr{};
            VT xo = VT(0);
            HaloRec hw{};
            int hc = 0;
            auto recs = [&]() {
                if constexpr (STEP) xo = st.x[row < A.n ? row : 0];
                if constexpr (HALO) {
                    hc = hf;
                    hw = halo_rec_load(rrec, hq, hc);
                    hf = A.hflag[fidx(nxt)];
                    hq = A.hwq[fidx(nxt) >> 6];
                }
            };
            VT s = cs.template rows<VT>(A.n, (int)t, nxt, aft, A.xadj, A.cols, vals, x, sm, row,
                                        &pr, VT(0), recs);
            s = A.coo ? s : VT(0) + s;
            if constexpr (HALO) {
                bool over = false;
                const VT sh = halo_rec_add<VT>(s, hw, hc, over);
                s = over ? halo_row<VT>(row, (int)t, s, A.hrow_tile, A.hrows, A.hptr, A.hcols, A.hvals,
                                        A.ghost)
                         : sh;
            }
            cs.advance(nxt, sm);
            if (row < A.n) finish(row, s, pr, xo);
        }
    } else if constexpr (FMT == kFmtClass) {
        // (the table is in LDS: k_pcg_spmv loads it before it has the token)
        const WideClasses<VT> src{A.cls, &sm};
        auto edge = [&](const int (&r)[WideOf<VT>::E], VT (&s)[WideOf<VT>::E], VT (&pr)[WideOf<VT>::E]) {
            class_rows<VT, WideOf<VT>::E>(A.n, A.nd, A.doff, A.cls, sm, r, x, s, pr, A.dzero);
        };
        acc = A.nd <= 7 ? k1_wide<VT, 7, 2, false>(A, x.x, v, src, edge, wide, walk)
                        : k1_wide<VT, 8, 2, false>(A, x.x, v, src, edge, wide, walk);
    } else if constexpr (FMT == CEL_FMT_DIA) {
        if constexpr (!HALO && !STEP) {
            if (A.dwide) {  // uniform
                const WideDiags<VT, KEEP> src{dia_vals<VT>(A), A.dbase, A.dmask8};
                auto edge = [&](const int (&r)[WideOf<VT>::E], VT (&s)[WideOf<VT>::E], VT (&pr)[WideOf<VT>::E]) {
                    dia_rows<VT, WideOf<VT>::E, (WideOf<VT>::E >= 4 ? 4 : 8), KEEP>(
                        A.n, A.nd, A.doff, dia_vals<VT>(A), A.dmask8, nullptr, r, x, s, pr, A.dzero);
                };
                constexpr bool F64 = sizeof(VT) == 8;
                constexpr int NG = F64 ? 1 : 2;
                return A.nd <= 7 ? k1_wide<VT, 7, NG, F64>(A, x.x, v, src, edge, wide, walk)
                                 : k1_wide<VT, 8, NG, F64>(A, x.x, v, src, edge, wide, walk);
            }
        }
        // all tiles of a group per step, one row of each per thread; the
        // rows are added to the partial in tile order, as in the CSR K1.
        // Halo rows (HALO): as in the CSR K1, a row's record is added after
        // its local sum.  The records of a step load at the end of the step
        // before (after its products, into the registers those just freed)
        // and the flags one step earlier still, so both are in by the time
        // the step's products are and neither is copied while in flight.
        constexpr int R = kTileGroup;
        const long long ngroups = (ntiles + R - 1) / R;
        const auto rrec = tile_rsrc(HALO ? A.hrec : nullptr, HALO ? A.hnq * 16 : 0);
        // flag index of this thread's row of tile t (rows past n read hflag[n] = 0)
        auto fidx = [&](long long t) {
            const long long r = t * kTileRows + threadIdx.x;
            return t < ntiles && r < A.n ? (int)r : A.n;
        };
        // flags and first compact halo indices of the next group, entry
        // counts and records of this group
        int hf[R], hq[R], hc[R];
        HaloRec hr[R];
        auto load_flags = [&](long long q) {
#pragma unroll
            for (int k = 0; k < R; ++k) {
                hf[k] = A.hflag[fidx(R * q + k)];
                hq[k] = A.hwq[fidx(R * q + k) >> 6];
            }
        };
        // a wave without halo rows in a tile skips that tile's record load
        auto load_recs = [&]() {
#pragma unroll
            for (int k = 0; k < R; ++k) {
                hc[k] = hf[k];
                hr[k] = HaloRec{};
                if (__builtin_amdgcn_ballot_w64(hc[k] != 0)) hr[k] = halo_rec_load(rrec, hq[k], hc[k]);
            }
        };
        if constexpr (HALO) {
            const long long q0 = blockIdx.x;
            load_flags(q0);
            load_recs();
            load_flags(q0 + gridDim.x);
        }
        for (long long q = blockIdx.x; q < ngroups; q += gridDim.x) {
            int r[R];
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const long long t = R * q + k;
                r[k] = t < ntiles ? (int)t * kTileRows + threadIdx.x : A.n;
            }
            if (r[0] < A.n) {
                VT s[R], xo[R];
                typename X::Raw pr[R];
                if constexpr (STEP) {
#pragma unroll
                    for (int k = 0; k < R; ++k) xo[k] = st.x[r[k] < A.n ? r[k] : r[0]];
                }
                // x[row] comes from the loads of the diagonal with offset 0
                dia_rows<VT, R, (R >= 4 ? 4 : 8), KEEP>(A.n, A.nd, A.doff, dia_vals<VT>(A), A.dmask8,
                                                        A.dmask, r, x, s, pr, A.dzero);
#pragma unroll
                for (int k = 0; k < R; ++k) {
                    if (r[k] < A.n) {
                        const typename X::Raw pk = A.dzero >= 0 ? pr[k] : x.load(r[k]);
                        VT sk = VT(0) + s[k];
                        if constexpr (HALO) {
                            bool over = false;
                            sk = halo_rec_add<VT>(sk, hr[k], hc[k], over);
                            if (over) {  // more than kHaloRec entries: the compact lists
                                VT s0 = VT(0) + s[k];
                                const int hq = A.hrowq[r[k]];
                                for (int j = A.hptr[hq]; j < A.hptr[hq + 1]; ++j) {
                                    VT prod = VT(A.hvals[j]) * VT(A.ghost[A.hcols[j]]);
                                    s0 = s0 + prod;
                                }
                                sk = s0;
                            }
                        }
                        finish(r[k], sk, pk, STEP ? xo[k] : VT(0));
                    }
                }
            }
            if constexpr (HALO) {  // the next group's records, the flags of the one after
                load_recs();
                load_flags(q + 2 * (long long)gridDim.x);
            }
        }
    } else {
        // JAD in the permuted row order: the CSR K1's tile-pair order, one
        // row per thread and tile, the next tile's row loaded while this
        // one's gathers are in flight
        JadStream<VT, X, KEEP> js;
        js.init(A.n, A.mmax, A.jnnz, A.jbegin, A.jcols, jad_vals<VT>(A), x);
        long long k = 0;
        long long t = group_tile(0, ntiles);
        if (t >= 0) js.fetch((int)t * kTileRows + threadIdx.x);
        for (; t >= 0; t = group_tile(++k, ntiles)) {
            const long long tn = group_tile(k + 1, ntiles);
            const int row = (int)t * kTileRows + threadIdx.x;
            const int rn = tn >= 0 ? (int)tn * kTileRows + threadIdx.x : A.n;
            typename X::Raw pr;
            VT xo = VT(0);
            if constexpr (STEP) xo = st.x[row < A.n ? row : 0];
            VT s = js.template row<VT>(row, rn, A.mmax, A.jbegin, A.jcols, jad_vals<VT>(A), x, pr);
            // the reference's JAD product overwrites v (y(perm(k)) = tmp(k))
            if (row < A.n) finish(row, s, pr, xo);
        }
    }
    return acc;
}

// The FP64 K1 of long rows in a narrow band: x of a tile group's columns in
// LDS.  CsrLongStream is bound by its gathers (11 per row of a mesh, a line
// of L2 each); 2 * band + 512 values loaded in order are a fraction of those
// bytes, and the gathers then read LDS.  The rows, blocks and orders are the
// K1's, so the partials are the same.  Two blocks per CU (kWindowCap).
// Per iteration, from L2 / from LDS: 1,000,003 rows of 13 entries in a band of
// 3500 76.7 / 55.9 us, of 1400 61.7 / 53.9, 2,000,003 rows in 1400 128.8 /
// 104.9, 200,003 in 3420 25.4 / 21.7 (27 entries 40.2 / 30.6), 300,007 in 700
// 29.6 / 27.8, 100,003 in 3420 19.5 / 18.5 and in 1000 17.7 / 18.0, 20,011 in
// 700 16.8 / 17.1: hence kWindowRows.  Not in the mixed form, whose values are
// half as wide (600,011 rows 38.6 / 38.0, 300,007 28.9 / 30.2).
constexpr int kWindowCap = 7680;  // values: 60 KB beside the tile's stage, twice in 160 KB
constexpr int kWindowRows = 120000;
static bool window_fits(const Mat& A)
{
    return A.band >= 0 && 2LL * A.band + kTileGroup * kTileRows + 4 <= kWindowCap;
}

template <bool KEEP>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2, 8))) void k_pcg_window(
    MatView A, const double* __restrict__ p, double* __restrict__ v, double* __restrict__ part, ResArgs<double> R,
    const Ctrl* __restrict__ cin, Ctrl* __restrict__ cout, Prm P)
{
    __shared__ struct {
        CsrLongStage<double> tile;
        alignas(16) double win[kWindowCap];
    } sm;
    __shared__ double red[3 * kWaves];
    __shared__ double fred[2 * kWaves];
    Ctrl c = read_ctrl(cin);
    if (c.reduce != kReduceNone) fold_pending(c, R.part, R.G, P, fred);
    if (!c.run) {
        write_ctrl(cout, c);
        return;
    }
    const long long ntiles = (A.n + kTileRows - 1) / kTileRows;
    const double* vals = A.vals;
    CsrLongStream<double, KEEP> cs;
    const long long tfirst = group_tile(0, ntiles);
    if (tfirst >= 0) cs.open(A.n, (int)tfirst, (int)group_tile(1, ntiles), A.xadj, A.cols, vals, sm.tile);
    double acc = 0.0;
    XWindow<double> x{sm.win, 0, 0};
    long long k = 0;
    for (long long t = tfirst; t >= 0; t = group_tile(++k, ntiles)) {
        if (k % kTileGroup == 0) {  // a new group: its columns
            const int r0 = (int)t * kTileRows;
            x.w0 = max(0, r0 - A.band) & ~1;
            const int w1 = min(A.n, r0 + kTileGroup * kTileRows + A.band);
            x.last = w1 - x.w0 - 1;
            // (16 bytes per load; past w1 it returns 0)
            const auto rx = tile_rsrc(p + x.w0, (w1 - x.w0) * 8);
            __syncthreads();  // the group before is done with the window
            constexpr int kAt = kWindowCap / 2 / kBlock;
            U32x4 w[kAt];
#pragma unroll
            for (int i = 0; i < kAt; ++i)
                w[i] = __builtin_amdgcn_raw_buffer_load_b128(rx, 16 * (int)threadIdx.x, 16 * kBlock * i, 0);
#pragma unroll
            for (int i = 0; i < kAt; ++i)
                reinterpret_cast<U32x4*>(sm.win)[threadIdx.x + kBlock * i] = w[i];
            __syncthreads();
        }
        const int nxt = (int)group_tile(k + 1, ntiles);
        const int aft = (int)group_tile(k + 2, ntiles);
        const int row = (int)t * kTileRows + threadIdx.x;
        double pr = 0.0;
        double s = cs.template rows<double>(A.n, (int)t, nxt, aft, A.xadj, A.cols, vals, x, sm.tile, row, &pr);
        s = A.coo ? s : 0.0 + s;
        if (row < A.n) {
            v[row] = s;
            const double prod = s * pr;
            acc = acc + prod;
        }
    }
    const double bs = block_sum(acc, red);
    if (threadIdx.x == 0) part[logical_block()] = bs;
    write_ctrl(cout, c);
}

// LDS of a K1: its tile stage and that of a wide walk; in the mixed form the
// FP64 stage of a replacement residual takes the same place.
template <typename VT, int FMT, bool LONG, bool WIDE>
union K1Stage {
    struct {
        typename StageOf<VT, FMT, LONG>::T tile;
        typename WideStageOf<WIDE>::T wide;
    };
    typename StageOf<double, FMT == CEL_FMT_DIA ? CEL_FMT_CSR : FMT, LONG>::T res;
};

// Waves per SIMD the K1s are compiled for.  The FP64 wide walks hold the loads
// of two tasks or steps in registers; the FP64 K1s run on 2 blocks per CU
// (kK1BlocksPerCuF64), so it may take the registers of 2 waves.
template <typename VT, int FMT>
constexpr int k1_waves = sizeof(VT) == 8 && (FMT == kFmtClass || FMT == CEL_FMT_DIA) ? 2 : 4;

// K1: v = A p, per-block partial of v.p.  Mixed: a requested replacement
// residual takes the place of the product (K2 and K3 then do nothing, and
// the next K1 folds its partials).  LONG of a DIA K1: its residual's.
template <typename VT, int FMT, bool HALO, bool LONG, bool KEEP = false, int TAIL = 1>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(k1_waves<VT, FMT>, 8))) void k_pcg_spmv(MatView A, const VT* __restrict__ p,
                                                     VT* __restrict__ v, double* __restrict__ part,
                                                     ResArgs<VT> R,
                                                     const Ctrl* __restrict__ cin,
                                                     Ctrl* __restrict__ cout, Prm P)
{
    constexpr bool MIXED = sizeof(VT) == 4;
    __shared__ K1Stage<VT, FMT, LONG, wide_form<FMT, HALO, false>> sm;
    __shared__ double red[3 * kWaves];
    __shared__ double fred[2 * kWaves];
    Ctrl c = read_ctrl(cin);
    if constexpr (FMT == kFmtClass) load_classes<VT>(A, sm.tile);
    if (c.reduce != kReduceNone) fold_pending(c, R.part, R.G, P, fred);
    if (!c.run) {
        write_ctrl(cout, c);
        return;
    }
    if constexpr (MIXED) {
        if (c.ru) {  // uniform
            replace_residual<FMT == CEL_FMT_DIA ? CEL_FMT_CSR : FMT, LONG>(A, R, c, P, sm.res, red);
            write_ctrl(cout, c);
            return;
        }
    }
    // the walk (first group, and the partial's slot) of this block: a wide one
    // may be another block's
    int walk = blockIdx.x, slot = logical_block();
    if constexpr (wide_form<FMT, HALO, false>) {
        if (A.walk) {
            walk = A.walk[blockIdx.x];
            slot = gridDim.x % kXcds ? walk : (walk % kXcds) * (gridDim.x / kXcds) + walk / kXcds;
        }
    }
    StepStream<VT, FMT, LONG, KEEP> none;
    const double acc = k1_tiles<VT, FMT, HALO, LONG, false, KEEP, TAIL>(A, XPlain<VT>{p}, v, none, sm.tile, sm.wide, StepRows<VT>{}, walk);
    const double bs = block_sum(acc, red);
    if (threadIdx.x == 0) part[slot] = bs;
    write_ctrl(cout, c);
}

// A group of CSR tiles of the step kernel, one row of each tile per thread,
// every row read by its own thread: a block's chain is three round trips
// (row bounds, entries, gathers) for all of its rows, without LDS and
// barriers, and none of them waits for the step's scalars.  A lane's entries
// lie 28 to 84 bytes from the next one's, so every load touches the lines of
// all of a wave's rows, which pays as long as few blocks share the caches.
// Per iteration, tiles in LDS / so: FP64 20^3 10.4 / 9.8 us, 32^3 10.5 / 9.95,
// 40^3 11.8 / 11.2, 44^3 12.2 / 12.8, 64^3 14.4 / 15.0; mixed 20^3 12.1 / 11.3,
// 32^3 11.8 / 10.9, 48^3 12.5 / 12.2, 52^3 13.6 / 14.1, 64^3 13.7 / 15.0; hence
// the lines in step_direct, 70,000 and 120,000 rows.
template <typename VT>
struct DirectGroup {
    static constexpr int R = kTileGroup;
    int r[R], lo[R], hi[R];
    VT a[R][kGather], xo[R];
    typename XDirection<VT>::Raw xv[R][kGather], own[R];

    __device__ __forceinline__ void load(const MatView& A, long long q, const XDirection<VT>& d, const VT* x)
    {
        const VT* vals = csr_vals<VT>(A);
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const long long i = (R * q + k) * kTileRows + threadIdx.x;
            r[k] = i < A.n ? (int)i : A.n;
            const int rc = r[k] < A.n ? r[k] : 0;
            lo[k] = A.xadj[rc];
            hi[k] = A.xadj[rc + 1];
        }
        int c[R][kGather];
#pragma unroll
        for (int k = 0; k < R; ++k)
#pragma unroll
            for (int i = 0; i < kGather; ++i) {
                const int at = lo[k] + i < hi[k] ? lo[k] + i : 0;
                c[k][i] = A.cols[at];
                a[k][i] = vals[at];
            }
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int rc = r[k] < A.n ? r[k] : 0;
            own[k] = d.load(rc);
            xo[k] = x[rc];
        }
#pragma unroll
        for (int k = 0; k < R; ++k)
#pragma unroll
            for (int i = 0; i < kGather; ++i) xv[k][i] = d.load(c[k][i]);
    }
    // the row's sum in column order (rows of more than kGather entries read
    // the others here)
    __device__ __forceinline__ VT sum(int k, const MatView& A, const XDirection<VT>& d) const
    {
        VT s = VT(0);
#pragma unroll
        for (int i = 0; i < kGather; ++i) {
            const VT prod = a[k][i] * d.value(xv[k][i]);
            const VT t = s + prod;
            s = lo[k] + i < hi[k] ? t : s;
        }
        const VT* vals = csr_vals<VT>(A);
        for (int j = lo[k] + kGather; j < hi[k]; ++j) {
            const VT prod = vals[j] * d.value(d.load(A.cols[j]));
            s = s + prod;
        }
        return s;
    }
};

// K3 and the next iteration's K1 in one launch, for small systems (rule at
// step_form): beta and the loop decision from K2's partials, x += sigma p,
// p_new = beta p + z, v = A p_new and the partials of v.p_new.  A block
// needs p_new of its neighbours' rows as well, so every gather reads p and
// z and forms p_new itself (the same roundings as K3), and p_new goes to a
// second buffer.  The rows, blocks and orders are the K1's, so the solve is
// bit for bit the three-kernel one.  An iteration that stops or requests
// the FP64 residual (mixed) only updates the vectors; the request's flush
// (x64 += e, e = 0) is K3's, and the next launch forms the residual.  What
// it saves is a launch and K3's second look at p; what it costs is a second
// gather per entry.
template <typename VT, int FMT, bool DIRECT = false>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(sizeof(VT) == 4 ? 4 : 2, 8))) void k_pcg_step(
    MatView A, const VT* __restrict__ p, const VT* __restrict__ z, VT* __restrict__ pout,
    VT* __restrict__ x, double* __restrict__ x64, VT* __restrict__ v, double* __restrict__ part,
    ResArgs<VT> R, const double* __restrict__ part2, int G2, const Ctrl* __restrict__ cin,
    Ctrl* __restrict__ cout, Prm P)
{
    constexpr bool MIXED = sizeof(VT) == 4;
    __shared__ K1Stage<VT, FMT, false, false> sm;
    __shared__ double red[3 * kWaves];
    __shared__ double fred[2 * kWaves];
    Ctrl c = read_ctrl(cin);
    // the partials' loads do not wait for the token
    const Parts<MIXED ? false : FMT == CEL_FMT_CSR> sz(part2, G2), sr(part2 + G2, G2);
    StepStream<VT, FMT, false, true> first;
    if constexpr (!DIRECT && kOpenAhead<VT>) first.open(A, sm.tile);
    DirectGroup<VT> grp;
    const long long ngroups = ((long long)A.n + kTileGroup * kTileRows - 1) / (kTileGroup * kTileRows);
    if constexpr (DIRECT) grp.load(A, blockIdx.x, XDirection<VT>{p, z, VT(0), false}, x);
    if (!c.run) {
        write_ctrl(cout, c);
        return;
    }
    if constexpr (MIXED) {
        if (c.ru) {  // uniform; the direction moves on to the next slot's buffer
            replace_residual<FMT == CEL_FMT_DIA ? CEL_FMT_CSR : FMT, false>(A, R, c, P, sm.res, red);
            if (!P.ru_restart)
                for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < A.n;
                     i += (long long)gridDim.x * kBlock)
                    pout[i] = p[i];
            write_ctrl(cout, c);
            return;
        }
    }
    const bool pending = c.reduce != kReduceNone;
    if (pending) {
        fold_pending(c, R.part, R.G, P, fred);
    } else {
        double rz, rr;
        all_sum2(sz.sum(), sr.sum(), fred, rz, rr);
        next_scalars<MIXED>(c, rz, rr, P);
    }
    const VT sigma = VT(c.sigma), beta = VT(c.beta);
    if (!c.run || (MIXED && c.ru)) {  // uniform: no product
        const bool flush = MIXED && c.ru;
        if (!pending)
            for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < A.n;
                 i += (long long)gridDim.x * kBlock) {
                const VT pi = p[i];
                const VT t = sigma * pi;
                VT xi = x[i] + t;
                if (flush) {
                    const double tt = (double)xi;
                    x64[i] = x64[i] + tt;
                    xi = VT(0);
                }
                x[i] = xi;
                const VT bp = beta * pi;
                pout[i] = bp + z[i];
            }
        write_ctrl(cout, c);
        return;
    }
    double acc = 0.0;
    const XDirection<VT> d{p, z, beta, pending};
    if constexpr (DIRECT) {
        for (long long q = blockIdx.x; q < ngroups; q += gridDim.x) {
            if (q != blockIdx.x) grp.load(A, q, d, x);
#pragma unroll
            for (int k = 0; k < kTileGroup; ++k) {
                const int row = grp.r[k];
                if (row >= A.n) continue;
                VT s = grp.sum(k, A, d);
                s = A.coo ? s : VT(0) + s;
                const VT dk = d.value(grp.own[k]);
                v[row] = s;
                pout[row] = dk;
                if (!pending) {
                    const VT t = sigma * grp.own[k].p;
                    x[row] = grp.xo[k] + t;
                }
                const double prod = double(s) * double(dk);
                acc = acc + prod;
            }
        }
    } else {
        acc = k1_tiles<VT, FMT, false, false, true, true, 1>(A, d, v, first, sm.tile, sm.wide,
                                                          StepRows<VT>{pout, x, sigma, !pending});
    }
    const double bs = block_sum(acc, red);
    if (threadIdx.x == 0) part[logical_block()] = bs;
    write_ctrl(cout, c);
}

// 16-byte vectors for the streaming kernels
template <typename VT>
struct Vec;
template <>
struct Vec<double> {
    using T = double2;
    static constexpr int W = 2;
};
template <>
struct Vec<float> {
    using T = float4;
    static constexpr int W = 4;
};

template <typename VT>
__device__ __forceinline__ VT lane(const typename Vec<VT>::T& a, int k)
{
    if constexpr (Vec<VT>::W == 2) {
        return k == 0 ? a.x : a.y;
    } else {
        return k == 0 ? a.x : k == 1 ? a.y : k == 2 ? a.z : a.w;
    }
}

template <typename VT>
__device__ __forceinline__ void set_lane(typename Vec<VT>::T& a, int k, VT v)
{
    if constexpr (Vec<VT>::W == 2) {
        if (k == 0) a.x = v;
        else a.y = v;
    } else {
        if (k == 0) a.x = v;
        else if (k == 1) a.y = v;
        else if (k == 2) a.z = v;
        else a.w = v;
    }
}

// The Jacobi values of W consecutive elements: from the vector, or (CLS)
// from the rows' classes and their table in LDS.
template <typename VT, bool CLS>
struct JacOf {
    using Raw = typename Vec<VT>::T;
    const VT* jac;
    __device__ __forceinline__ Raw load(long long i) const { return *reinterpret_cast<const Raw*>(jac + i); }
    __device__ __forceinline__ VT value(const Raw& r, int k) const { return lane<VT>(r, k); }
    __device__ __forceinline__ VT at(long long i) const { return jac[i]; }
};
template <typename VT>
struct JacOf<VT, true> {
    using Raw = unsigned;  // W class bytes
    const uint8_t* cls;
    VT* tab;  // LDS
    // the table to LDS; every thread of the block; it synchronises
    __device__ __forceinline__ void table(const VT* __restrict__ jac) const
    {
        tab[threadIdx.x] = jac[threadIdx.x];  // kMaxClass == kBlock
        __syncthreads();
    }
    __device__ __forceinline__ Raw load(long long i) const
    {
        if constexpr (Vec<VT>::W == 2) return *reinterpret_cast<const uint16_t*>(cls + i);
        else return *reinterpret_cast<const uint32_t*>(cls + i);
    }
    __device__ __forceinline__ VT value(Raw r, int k) const { return tab[(r >> (8 * k)) & 255u]; }
    __device__ __forceinline__ VT at(long long i) const { return tab[cls[i]]; }
};

template <typename VT, bool CLS>
__device__ __forceinline__ JacOf<VT, CLS> jac_of(const VT* __restrict__ jac, const uint8_t* __restrict__ cls,
                                                 VT* lds)
{
    if constexpr (CLS) return JacOf<VT, true>{cls, lds};
    else return JacOf<VT, false>{jac};
}
static_assert(kMaxClass == kBlock, "one table entry per thread");

// Whole 16-byte units per thread and loop step in the vector kernels (all
// their loads in flight together).  Measured on the 256^3 solves (two
// interleaved repetitions, one box): FP32 4 (mixed CSR 304-305 ms against
// 309-310 with 1, 308-310 with 2), FP64 2 (CSR 497-501 against 503-507
// with 1, 501-506 with 4).
template <typename VT>
constexpr int kVecUnrollOf = sizeof(VT) == 4 ? 4 : 2;

// Which vectors K2 and K3 keep in the infinity cache, by the bytes of the
// vectors an iteration touches (x, p, r, v, and the Jacobi vector or the
// class bytes).  A vector that is marked as read once leaves its room to the
// others: kStreamX: x, which only K3 touches; kStreamAll: also v and r where
// they are read, so that what stays is what the next kernel reads (v from K1
// to K2, r from K2 to K3, p from K3 to K1).  Measured per iteration with
// none / x / all marked, Poisson cubes on row classes: FP64 180^3 (192 MB)
// 88.2 / 90.0 / 92.5 us, 200^3 (264) 124.9 / 116.2 / 119.8, 216^3 (333) 154.7
// / 144.3 / 147.9, 232^3 (412) 205.6 / 181.5 / 177.1; mixed 232^3 (212) 97.7 /
// 99.9 / 102.2, 256^3 (285) 138.8 / 126.8 / 129.4, 288^3 (406) 210.0 / 183.7 /
// 180.7; general variable coefficients FP64 176^3 (218) 146 / 147 / 149, 192^3 (283)
// 189 / 186 / 188, 216^3 (403) 285 / 267 / 264, 256^3 (671) 521 / 494 / 459.
// The values of a symmetric block (`arrays` of them) are kept as well and
// share the cache, so there the line is one on both together: 144^3 (215 MB)
// 65.8 / 67.0 / 68.4 us, 160^3 (295) 98.2 / 91.6 / 90.9, 176^3 (392) 125.1 /
// 122.9 / 122.0, 200^3 (576) 192.3 / 185.7 / 177.9, 230^3 (876) 311 / 295 / 279.
enum StreamLevel { kStreamNone = 0, kStreamX = 1, kStreamAll = 2 };
static int stream_level(long long n, bool mixed, bool cls, int arrays)
{
    const double vb = mixed ? 4.0 : 8.0;
    const double bytes = ((cls ? 4.0 : 5.0) * vb + (cls ? 1.0 : 0.0)) * (double)n;
    if (arrays) return bytes + arrays * vb * (double)n > 240e6 ? kStreamAll : kStreamNone;
    return bytes > 380e6 ? kStreamAll : bytes > 240e6 ? kStreamX : kStreamNone;
}

// K2: sigma = alpha / sum(v.p) ; r = r + (-sigma) v ; z = jac*r ;
// per-block partials of r.z and r.r.  ZOUT: z is stored too (for k_pcg_step).
// STREAM: stream_level (K2 knows none and all).
template <typename VT, bool ZOUT, bool CLS, int STREAM = kStreamNone>
__global__ __launch_bounds__(kBlock) void k_pcg_update_r(long long n, VT* __restrict__ r,
                                                         const VT* __restrict__ v,
                                                         const VT* __restrict__ jac,
                                                         const uint8_t* __restrict__ cls,
                                                         VT* __restrict__ z,
                                                         double* __restrict__ part,
                                                         const double* __restrict__ vpart, int G1,
                                                         const Ctrl* __restrict__ cin,
                                                         Ctrl* __restrict__ cout, int* progress)
{
    __shared__ double red[2 * kWaves];
    __shared__ double fred[kWaves];
    Ctrl c = read_ctrl(cin);
    // (in the two-kernel form K2 ends the slot)
    auto done = [&]() {
        if constexpr (ZOUT) end_slot(cout, c, progress);
        else write_ctrl(cout, c);
    };
    // AHEAD: the block's first elements are loaded with the partials, before
    // the token is looked at, and a step's at the end of the one before.
    // Per iteration without / with it, FP64 32^3 11.9 / 11.6 us, JAD 61x47x73
    // 15.5 / 15.2, DIA 128^3 50.9 / 50.3, 200^3 186.7 / 184.7; by classes 100^3
    // 26.7 / 27.1, mixed 100^3 22.0 / 23.1 (the registers of 4 units).
    const Parts<sizeof(VT) == 8> sv(vpart, G1);
    using V = typename Vec<VT>::T;
    constexpr int W = Vec<VT>::W;
    __shared__ VT jlds[CLS ? kMaxClass : 1];
    const JacOf<VT, CLS> J = jac_of<VT, CLS>(jac, cls, jlds);
    constexpr bool AHEAD = sizeof(VT) == 8 && !CLS;
    const int lb = logical_block();
    const int G = gridDim.x;
    const long long unit = (long long)kBlock * W;
    long long u0, u1;
    unit_range((n + unit - 1) / unit, G, lb, u0, u1);
    const long long lo = u0 * unit, hi = min(u1 * unit, n);
    long long i = lo + (long long)threadIdx.x * W;
    constexpr int kVecUnroll = kVecUnrollOf<VT>;
    V vv[kVecUnroll], rv[kVecUnroll];
    typename JacOf<VT, CLS>::Raw jv[kVecUnroll];
    // units i, i + unit, ... of the block, as far as they are whole vectors
    auto load = [&]() {
#pragma unroll
        for (int u = 0; u < kVecUnroll; ++u) {
            const long long at = i + u * unit < hi && i + u * unit + W <= n ? i + u * unit : 0;
            vv[u] = ld_vec<STREAM == kStreamAll, V>(v + at);
            rv[u] = ld_vec<STREAM == kStreamAll, V>(r + at);
            jv[u] = J.load(at);
        }
    };
    if (AHEAD && n >= W) load();  // uniform
    // a slot without a product: a replacement was requested (ru) or its
    // residual is pending (reduce)
    if (!c.run || c.ru || c.reduce != kReduceNone) {
        done();
        return;
    }
    const double vp = block_sum_all(sv.sum(), fred);
    const double sigma = c.alpha / vp;
    if (!(vp > 0.0) || !isfinite(sigma)) {
        c.status = CEL_ERR_BREAKDOWN;
        c.run = 0;
        done();
        return;
    }
    c.sigma = sigma;
    if constexpr (CLS) J.table(jac);
    if (!AHEAD && n >= W) load();
    const VT ms = VT(-sigma);
    double arz = 0.0, arr = 0.0;
    auto element = [&](VT vj, VT& rj, VT jj, VT& zj) {
        const VT t = ms * vj;
        const VT ri = rj + t;
        rj = ri;
        const VT zi = ri * jj;
        zj = zi;
        const double rz = double(ri) * double(zi);
        arz = arz + rz;
        const double rr = double(ri) * double(ri);
        arr = arr + rr;
    };
    auto vec = [&](int u, long long at) {
        V zv{};
#pragma unroll
        for (int k = 0; k < W; ++k) {
            VT ri = lane<VT>(rv[u], k), zi;
            element(lane<VT>(vv[u], k), ri, J.value(jv[u], k), zi);
            set_lane<VT>(rv[u], k, ri);
            if constexpr (ZOUT) set_lane<VT>(zv, k, zi);
        }
        *reinterpret_cast<V*>(r + at) = rv[u];
        if constexpr (ZOUT) *reinterpret_cast<V*>(z + at) = zv;
    };
    // kVecUnroll units per step while they are whole vectors (all their
    // loads in flight together), added to the partials in unit order
    while (i + (kVecUnroll - 1) * unit + W <= hi) {
#pragma unroll
        for (int u = 0; u < kVecUnroll; ++u) vec(u, i + u * unit);
        i += kVecUnroll * unit;
        load();
    }
#pragma unroll
    for (int u = 0; u < kVecUnroll; ++u) {
        const long long at = i + u * unit;
        if (at < hi) {
            if (at + W <= n) {
                vec(u, at);
            } else {
                for (long long j = at; j < hi; ++j) {
                    VT rj = r[j], zj;
                    element(v[j], rj, J.at(j), zj);
                    r[j] = rj;
                    if constexpr (ZOUT) z[j] = zj;
                }
            }
        }
    }
    block_sum2(arz, arr, red);
    if (threadIdx.x == 0) {
        part[lb] = arz;
        part[G + lb] = arr;
    }
    done();
}

// K3: beta = sum(r.z)/alpha ; x = x + sigma p ; p = beta p + jac*r ;
// alpha = r.z, norm2, k++, history, loop decision (FP64) or replacement
// request (mixed).  STREAM: stream_level.
template <typename VT, bool MIXED, bool CLS, int STREAM>
__global__ __launch_bounds__(kBlock) void k_pcg_update_xp(long long n, VT* __restrict__ x,
                                                          VT* __restrict__ p,
                                                          const VT* __restrict__ r,
                                                          const VT* __restrict__ jac,
                                                          const uint8_t* __restrict__ cls,
                                                          double* __restrict__ x64,
                                                          const double* __restrict__ rpart, int G2,
                                                          const Ctrl* __restrict__ cin,
                                                          Ctrl* __restrict__ cout, Prm P, int* progress)
{
    __shared__ double red[2 * kWaves];
    Ctrl c = read_ctrl(cin);
    const Parts<!MIXED> sz(rpart, G2), sr(rpart + G2, G2);
    using V = typename Vec<VT>::T;
    constexpr int W = Vec<VT>::W;
    __shared__ VT jlds[CLS ? kMaxClass : 1];
    const JacOf<VT, CLS> J = jac_of<VT, CLS>(jac, cls, jlds);
    constexpr bool AHEAD = sizeof(VT) == 8 && !CLS;
    const int lb = logical_block();
    const long long unit = (long long)kBlock * W;
    long long u0, u1;
    unit_range((n + unit - 1) / unit, gridDim.x, lb, u0, u1);
    const long long lo = u0 * unit, hi = min(u1 * unit, n);
    long long i = lo + (long long)threadIdx.x * W;
    constexpr int kVecUnroll = kVecUnrollOf<VT>;
    V pv[kVecUnroll], rv[kVecUnroll];
    typename JacOf<VT, CLS>::Raw jv[kVecUnroll];
    VT xs[kVecUnroll][W];
    // units i, i + unit, ... of the block, as far as they are whole vectors;
    // the first ones before the token is looked at (as in K2)
    auto load = [&]() {
#pragma unroll
        for (int u = 0; u < kVecUnroll; ++u) {
            const long long at = i + u * unit < hi && i + u * unit + W <= n ? i + u * unit : 0;
            pv[u] = *reinterpret_cast<const V*>(p + at);
            rv[u] = ld_vec<STREAM == kStreamAll, V>(r + at);
            jv[u] = J.load(at);
#pragma unroll
            for (int k = 0; k < W; ++k)
                xs[u][k] = STREAM != kStreamNone ? __builtin_nontemporal_load(x + at + k) : x[at + k];
        }
    };
    if (AHEAD && n >= W) load();  // uniform
    if (!c.run || c.reduce != kReduceNone) {
        end_slot(cout, c, progress);
        return;
    }
    double rz, rr;
    all_sum2(sz.sum(), sr.sum(), red, rz, rr);
    const VT sigma = VT(c.sigma);
    // scalars of the next iteration (they do not depend on the vectors)
    next_scalars<MIXED>(c, rz, rr, P);
    const VT beta = VT(c.beta);
    if constexpr (CLS) J.table(jac);
    if (!AHEAD && n >= W) load();
    // mixed, replacement iteration: the FP32 correction is folded into the
    // FP64 solution here (x64 = x64 + e, e = 0) instead of in a kernel of
    // its own; same arithmetic
    const bool flush = MIXED && c.ru;
    auto vec = [&](int u, long long at) {
#pragma unroll
        for (int k = 0; k < W; ++k) {
            const VT pi = lane<VT>(pv[u], k);
            VT t = VT(sigma * pi);
            xs[u][k] = xs[u][k] + t;
            VT zi = lane<VT>(rv[u], k) * J.value(jv[u], k);
            VT bp = beta * pi;
            set_lane<VT>(pv[u], k, bp + zi);
        }
        if (flush) {
#pragma unroll
            for (int k = 0; k < W; ++k) {
                double t = (double)xs[u][k];
                x64[at + k] = x64[at + k] + t;
                xs[u][k] = VT(0);
            }
        }
#pragma unroll
        for (int k = 0; k < W; ++k) {
            if constexpr (STREAM != kStreamNone) __builtin_nontemporal_store(xs[u][k], x + at + k);
            else x[at + k] = xs[u][k];
        }
        *reinterpret_cast<V*>(p + at) = pv[u];
    };
    // kVecUnroll units per step while they are whole vectors
    while (i + (kVecUnroll - 1) * unit + W <= hi) {
#pragma unroll
        for (int u = 0; u < kVecUnroll; ++u) vec(u, i + u * unit);
        i += kVecUnroll * unit;
        load();
    }
#pragma unroll
    for (int u = 0; u < kVecUnroll; ++u) {
        const long long at = i + u * unit;
        if (at < hi) {
            if (at + W <= n) {
                vec(u, at);
            } else {
                for (long long j = at; j < hi; ++j) {
                    const VT pi = p[j];
                    VT t = VT(sigma * pi);
                    VT xj = x[j] + t;
                    if (flush) {
                        double tt = (double)xj;
                        x64[j] = x64[j] + tt;
                        xj = VT(0);
                    }
                    x[j] = xj;
                    VT zi = r[j] * J.at(j);
                    VT bp = beta * pi;
                    p[j] = bp + zi;
                }
            }
        }
    }
    end_slot(cout, c, progress);
}

// Mixed form, replacement step 1: x64 = x64 + e32 ; e32 = 0.
__global__ __launch_bounds__(kBlock) void k_ru_flush(long long n, double* __restrict__ x,
                                                     float* __restrict__ e,
                                                     const Ctrl* __restrict__ cin,
                                                     Ctrl* __restrict__ cout, int force)
{
    const Ctrl c = read_ctrl(cin);
    write_ctrl(cout, c);
    if (!force && (!c.run || !c.ru)) return;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x) {
        double t = (double)e[i];
        x[i] = x[i] + t;
        e[i] = 0.0f;
    }
}

// ------------------------------------------------------------------ host side
struct Workspace {
    DevBuf<double> r, p, v, x, b, part1, part2, rpart, ghost, sendbuf, hist;
    DevBuf<float> r32, p32, v32, e32;
    // two-kernel iterations: the second direction buffer and z = jac*r
    DevBuf<double> p2, z;
    DevBuf<float> p2_32, z32;
    // JAD solves: b, x and the Jacobi vector in the permuted row order
    DevBuf<double> bp, xp, jacp;
    DevBuf<int> walk;  // row-class solves: the K1 blocks' walks
    // halo solves: per-row halo records {count, p1, p2, p3}
    DevBuf<double> hrec;
    DevBuf<float> jacp32;
    DevBuf<Ctrl> ctrl;
    DevBuf<int> hrow_tile;
    // pinned: the progress word the kernels write and the final token
    struct Host {
        int progress;
        int pad[31];
        Ctrl ctrl;
    };
    Host* host = nullptr;
    int host_alloc()
    {
        if (host) return CEL_OK;
        void* q = nullptr;
        if (hipHostMalloc(&q, sizeof(Host), hipHostMallocCoherent) != hipSuccess)
            return fail(CEL_ERR_OOM, "hipHostMalloc failed");
        host = static_cast<Host*>(q);
        return CEL_OK;
    }
    ~Workspace()
    {
        if (host) (void)hipHostFree(host);
    }
};

// Waits until the solve's kernels have finished `upto` slots (1), or stopped
// (0), or there is an error (< 0).  The word is in host memory, so looking
// at it costs the stream nothing.  It looks without a pause for 100 us, the
// slots of a small system (yielding from the first look on cost 32^3 0.25 us
// per iteration of 11.2); after that it gives the core to any other thread
// that wants it, every time round.
static int wait_progress(hipStream_t s, const volatile int* progress, long long upto)
{
    const auto begin = std::chrono::steady_clock::now();
    auto last = begin;
    for (;;) {
        for (int k = 0; k < 512; ++k) {
            const int v = *progress;
            if (v < 0) return 0;
            if (v >= upto) return 1;
            __builtin_ia32_pause();
        }
        const auto now = std::chrono::steady_clock::now();
        if (now - begin > std::chrono::microseconds(100)) std::this_thread::yield();
        if (now - last < std::chrono::milliseconds(1)) continue;
        last = now;
        const hipError_t e = hipStreamQuery(s);
        if (e == hipErrorNotReady) continue;
        if (e != hipSuccess) return fail(CEL_ERR_HIP, std::string("the solve's kernels: ") + hipGetErrorString(e));
        return *progress < 0 ? 0 : 1;  // everything enqueued has run
    }
}

static Workspace& ws_of(Mat& A)
{
    if (!A.ws) A.ws = new Workspace();
    return *A.ws;
}

// Compact halo rows per 256-row tile: hrow_tile[t] = first compact row >= t*256.
static int build_hrow_tile(const Mat& A, Workspace& W, int ntiles)
{
    std::vector<int> hrows(A.halo_nrows);
    if (A.halo_nrows)
        CEL_HIP(hipMemcpy(hrows.data(), A.halo_rows.p, sizeof(int) * A.halo_nrows,
                          hipMemcpyDeviceToHost));
    std::vector<int> ht(ntiles + 1, 0);
    int q = 0;
    for (int t = 0; t <= ntiles; ++t) {
        while (q < A.halo_nrows && hrows[q] < t * kTileRows) ++q;
        ht[t] = q;
    }
    CEL_TRY(W.hrow_tile.reserve(ntiles + 1));
    CEL_HIP(hipMemcpy(W.hrow_tile.p, ht.data(), sizeof(int) * (ntiles + 1), hipMemcpyHostToDevice));
    return CEL_OK;
}

// Blocks per CU of the vector kernels (K2, K3).  Measured on the 256^3
// solve: larger grids of these kernels, and K1 grids larger than the
// resident blocks, were slower -- every consumer block sums all producer
// partials, so more blocks cost more reduction work.
constexpr int kVecBlocksPerCu = 4;

// Blocks per CU of the K1s.  Measured on the
// 256^3 block (mean K1 time over 100-iteration solves, three interleaved
// repetitions on one box): FP32 4 per CU (CSR 206-223 us, DIA 121-127 us,
// against 223-230 / 136-145 us with every resident block), FP64 2 per CU
// (CSR 349-352 against 376 us, DIA 260-264 against 266-271 us).
constexpr int kK1BlocksPerCuF32 = 4;
constexpr int kK1BlocksPerCuF64 = 2;

// Blocks per CU of the residual kernels: the set-up's and the replacement's
// sums are grouped by them.  As many as were resident when it was measured.
constexpr int kResBlocksPerCu = 6;
constexpr int kResBlocksPerCuJad = 7;

// At most per_cu blocks per CU, a multiple of the XCDs.  A constant, not the
// occupancy of the kernel: every dot product is grouped by its grid, and a
// register more would otherwise change the last bits of every solve.
static int fixed_grid(int per_cu, long long work)
{
    const long long g = std::max(1LL, std::min((long long)rt().num_cus * per_cu, work));
    return (int)(g >= kXcds ? g / kXcds * kXcds : g);
}

// The K1s' grid: the CSR and DIA forms share it, with and without halo, so
// that their partials, and the solves, stay bitwise equal.
static int k1_grid(long long ntiles, bool mixed)
{
    return fixed_grid(mixed ? kK1BlocksPerCuF32 : kK1BlocksPerCuF64, ntiles);
}

// The K1 of a form.
template <typename VT>
using K1Fn = void (*)(MatView, const VT*, VT*, double*, ResArgs<VT>, const Ctrl*, Ctrl*, Prm);

// keep: the same kernel with ordinary loads of the matrix (keep_matrix); it
// runs on the other one's grid.  deep: deep_rows().
template <typename VT>
static K1Fn<VT> k1_kernel(int fmt, bool halo, bool lr, bool keep = false, bool deep = false)
{
    if (deep)
        return keep ? k_pcg_spmv<VT, CEL_FMT_CSR, false, false, true, kGather>
                    : k_pcg_spmv<VT, CEL_FMT_CSR, false, false, false, kGather>;
    if (keep && !halo && fmt != kFmtClass) {
        if (fmt == CEL_FMT_JAD) return k_pcg_spmv<VT, CEL_FMT_JAD, false, false, true>;
        if constexpr (sizeof(VT) == 4)
            if (fmt == CEL_FMT_DIA && lr) return k_pcg_spmv<VT, CEL_FMT_DIA, false, true, true>;
        if (fmt == CEL_FMT_DIA) return k_pcg_spmv<VT, CEL_FMT_DIA, false, false, true>;
        return lr ? k_pcg_spmv<VT, CEL_FMT_CSR, false, true, true> : k_pcg_spmv<VT, CEL_FMT_CSR, false, false, true>;
    }
    if (fmt == CEL_FMT_JAD) return k_pcg_spmv<VT, CEL_FMT_JAD, false, false>;
    if (fmt == kFmtClass) return k_pcg_spmv<VT, kFmtClass, false, false>;
    if constexpr (sizeof(VT) == 8) {  // halo blocks: FP64 only
        if (halo && fmt == CEL_FMT_DIA) return k_pcg_spmv<VT, CEL_FMT_DIA, true, false>;
        if (halo) return lr ? k_pcg_spmv<VT, CEL_FMT_CSR, true, true> : k_pcg_spmv<VT, CEL_FMT_CSR, true, false>;
        if (fmt == CEL_FMT_DIA) return k_pcg_spmv<VT, CEL_FMT_DIA, false, false>;
    } else if (fmt == CEL_FMT_DIA) {
        return lr ? k_pcg_spmv<VT, CEL_FMT_DIA, false, true> : k_pcg_spmv<VT, CEL_FMT_DIA, false, false>;
    }
    return lr ? k_pcg_spmv<VT, CEL_FMT_CSR, false, true> : k_pcg_spmv<VT, CEL_FMT_CSR, false, false>;
}

// Whether the K1s load the matrix (nd > 0: nd diagonals) so that it stays in
// the infinity cache: what an iteration touches, matrix and vectors, is at
// most kKeepBytes.  Above it the matrix would push out the vectors, which
// are touched more than once an iteration, and come from HBM all the same.
// Measured per iteration on 7-point cubes, marked as read once / kept, by
// the bytes touched: CSR FP64 112^3 (185 MB) 51.3 / 46.9 us, 128^3 (277)
// 71.5 / 65.8, 136^3 (332) 84.0 / 86.0, 144^3 (395) 96.6 / 101.9; DIA FP64
// 128^3 (218) 65.3 / 58.2, 144^3 (311) 85.4 / 84.9, 152^3 (365) 99.1 / 103.9;
// CSR mixed 144^3 (251) 62.9 / 58.7, 152^3 (295) 74.3 / 73.4, 160^3 (344)
// 85.8 / 88.2; DIA mixed 160^3 (230) 63.5 / 62.3, 176^3 (305) 80.9 / 81.9;
// JAD FP64 209,000 rows 17.0 / 15.7; 600,011 mesh rows mixed, whole solve
// 8.20 / 7.39 ms.  (A product by itself is better off without: 1,000,003
// mesh rows 99.0 / 102.3 us a call.)
constexpr double kKeepBytes = 300e6;
static bool keep_matrix(const Mat& A, int fmt, int nd, bool mixed)
{
    const double vb = mixed ? 4.0 : 8.0, n = A.n;
    const double m = fmt == CEL_FMT_DIA   ? nd * vb * n
                     : fmt == CEL_FMT_JAD ? (4.0 + vb) * (double)A.jad_nnz
                                          : (4.0 + vb) * (double)A.nnz + 4.0 * n;
    // the vectors: FP64 x, r, p, v, b, Jacobi; mixed r, p, v, e, Jacobi and x
    return m + (mixed ? 28.0 : 48.0) * n <= kKeepBytes;
}

template <typename VT>
using K2Fn = void (*)(long long, VT*, const VT*, const VT*, const uint8_t*, VT*, double*, const double*, int,
                      const Ctrl*, Ctrl*, int*);
template <typename VT>
static K2Fn<VT> k2_kernel(bool cls, int stream)
{
    if (stream == kStreamAll)
        return cls ? k_pcg_update_r<VT, false, true, kStreamAll> : k_pcg_update_r<VT, false, false, kStreamAll>;
    return cls ? k_pcg_update_r<VT, false, true> : k_pcg_update_r<VT, false, false>;
}

template <typename VT>
using K3Fn = void (*)(long long, VT*, VT*, const VT*, const VT*, const uint8_t*, double*, const double*, int,
                      const Ctrl*, Ctrl*, Prm, int*);
template <typename VT>
static K3Fn<VT> k3_kernel(bool cls, int stream)
{
    constexpr bool M = sizeof(VT) == 4;
    switch (stream) {
    case kStreamAll:
        return cls ? k_pcg_update_xp<VT, M, true, kStreamAll> : k_pcg_update_xp<VT, M, false, kStreamAll>;
    case kStreamX:
        return cls ? k_pcg_update_xp<VT, M, true, kStreamX> : k_pcg_update_xp<VT, M, false, kStreamX>;
    default:
        return cls ? k_pcg_update_xp<VT, M, true, kStreamNone> : k_pcg_update_xp<VT, M, false, kStreamNone>;
    }
}

template <typename VT>
using StepFn = void (*)(MatView, const VT*, const VT*, VT*, VT*, double*, VT*, double*, ResArgs<VT>,
                        const double*, int, const Ctrl*, Ctrl*, Prm);

// (lines: DirectGroup)
static bool step_direct(int fmt, int n, bool mixed) { return fmt == CEL_FMT_CSR && n <= (mixed ? 120000 : 70000); }

template <typename VT>
static StepFn<VT> step_kernel(int fmt, int n)
{
    if (fmt == CEL_FMT_JAD) return k_pcg_step<VT, CEL_FMT_JAD>;
    if (step_direct(fmt, n, sizeof(VT) == 4)) return k_pcg_step<VT, CEL_FMT_CSR, true>;
    return fmt == CEL_FMT_DIA ? k_pcg_step<VT, CEL_FMT_DIA> : k_pcg_step<VT, CEL_FMT_CSR>;
}

// Whether a solve iterates with two kernels (k_pcg_step, K2) instead of
// three: small systems, whose iteration is launches and latency rather than
// bytes.  Measured per iteration on variable-coefficient 7-point cubes, two
// against three kernels, CSR: FP64 32^3 12.3 / 13.6 us, 64^3 17.4 / 18.6,
// 80^3 28.7 / 29.3, 100^3 43.0 / 39.8; mixed 32^3 12.6 / 14.4, 80^3 22.9 /
// 24.6, 100^3 32.7 / 33.6, 128^3 48.8 / 49.1 (DIA and JAD alike).  Long rows
// pay for the second gather at any size (30,011 mesh rows of 11 entries 19.3
// / 18.7 us, 200,003 rows 36.5 / 29.3 us).
static bool step_form(const Mat& A, int fmt, bool mixed)
{
    return A.n <= (mixed ? 1200000 : 300000) && !csr_long_rows(A) && !(fmt == CEL_FMT_JAD && A.jad_mmax > kGather);
}

// Whether a CSR solve runs on the K1 that loads the entries of long rows
// kGather at a time (and never on k_pcg_step, whose second gather they pay
// for one after another): matrices of short rows, most of them, and a few
// that one thread sums for longer than an iteration otherwise takes.
// Measured per iteration, rows of 5 entries and 30 longer ones, without / so:
// FP64 20,011 rows, longest of 26 17.6 / 17.0 us, of 74 42.6 / 22.5, of 522 239
// / 80; mixed 26 23.2 / 22.1, 522 228 / 107; FP64 600,011 rows 25 33.1 / 31.9,
// 521 276 / 102.  Loading them so in the kernels of every matrix costs those
// without long rows 2 to 6% (registers): FP64 32^3 11.3 / 11.7 us, mixed 40^3
// 12.2 / 12.8.
constexpr int kDeepRow = 24;
static bool deep_rows(const Mat& A) { return A.longest > kDeepRow && !csr_long_rows(A); }

// The set-up kernel of a solve in the CSR or JAD form.
template <typename OUT_T>
using ResFn = void (*)(MatView, ResArgs<OUT_T>, const Ctrl*, Ctrl*);

template <typename OUT_T>
static ResFn<OUT_T> res_kernel(int fmt, bool halo, bool lr)
{
    if (fmt == CEL_FMT_JAD) return k_residual<OUT_T, CEL_FMT_JAD, false, false>;
    if (fmt == kFmtClass) return k_residual<OUT_T, kFmtClass, false, false>;
    if constexpr (sizeof(OUT_T) == 8)
        if (halo)
            return lr ? k_residual<OUT_T, CEL_FMT_CSR, true, true> : k_residual<OUT_T, CEL_FMT_CSR, true, false>;
    return lr ? k_residual<OUT_T, CEL_FMT_CSR, false, true> : k_residual<OUT_T, CEL_FMT_CSR, false, false>;
}

// The allocation-free entry point's device memory: a file-scope array
// (one copy per GPU, resolved to a device address once per device), laid
// out as r, p, v (kNoAllocMaxRows doubles each), the three partial-sum
// arrays (kNoAllocMaxGrid, 2x and 3x that) and the five token slots.
constexpr size_t kNoAllocMaxRows = size_t(1) << 20;
constexpr size_t kNoAllocMaxGrid = 8192;
constexpr size_t kNoAllocDoubles = 3 * kNoAllocMaxRows + 6 * kNoAllocMaxGrid;
constexpr size_t kNoAllocBytes = kNoAllocDoubles * sizeof(double) + 5 * 128;
static_assert(sizeof(Ctrl) <= 128, "token slot");
static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];
constexpr int kMaxDevices = 64;
static void* g_scratch[kMaxDevices];

int pcg_noalloc_setup(int device)
{
    if (device < 0 || device >= kMaxDevices) return fail(CEL_ERR_ARG, "device index beyond the scratch table");
    if (g_scratch[device]) return CEL_OK;
    void* ptr = nullptr;
    // the name `scratch` is a host-side stand-in; kernels get this address
    CEL_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    g_scratch[device] = ptr;
    return CEL_OK;
}

// Device pointers of one solve's work vectors, partial sums and token.
struct WorkPtrs {
    double *r = nullptr, *p = nullptr, *v = nullptr, *part1 = nullptr, *part2 = nullptr,
           *rpart = nullptr;
    float *r32 = nullptr, *p32 = nullptr, *v32 = nullptr, *e32 = nullptr;
    Ctrl* ctrl = nullptr;
};

// One FP64 K1 of the solve on caller vectors (device pointers, n rows):
// y = A x in the CSR or DIA form, plus, with ghost, the halo products of
// the caller's ghost values (the halo records of the solve, built from
// them first), and dot = x.y summed over the K1's block partials in
// logical-block order, as the solve's K2 sums them.
int pcg_spmv_dot(Mat& A, int fmt, const double* x, const double* ghost, double* y, double* dot)
{
    CEL_TRY(ensure_init());
    const int n = A.n;
    if (fmt != CEL_FMT_CSR && fmt != CEL_FMT_DIA)
        return fail(CEL_ERR_ARG, "the fused product runs in the CSR or the DIA form");
    if (fmt == CEL_FMT_DIA && A.dia_nd == 0)
        return fail(CEL_ERR_STATE, "DIA requested but the matrix has no DIA form");
    if (A.ncols != n) return fail(CEL_ERR_ARG, "the fused product needs a square local block");
    const bool halo = ghost != nullptr;
    if (halo && A.halo.empty()) return fail(CEL_ERR_STATE, "ghost values given but no halo blocks");
    if (halo && (double)A.halo_nrows * 16.0 >= 2147483648.0 - 64.0)
        return fail(CEL_ERR_ARG, "the halo records need 31-bit offsets (< 2^27 halo rows)");
    if (fmt == CEL_FMT_DIA && (double)n * 8.0 >= 2147483648.0)
        return fail(CEL_ERR_ARG, "the DIA kernels address x with 32-bit byte offsets");
    if (dot) *dot = 0.0;
    if (n == 0) return CEL_OK;
    const int ntiles = (n + kTileRows - 1) / kTileRows;
    const int G1 = k1_grid(ntiles, false);
    Workspace& W = ws_of(A);
    CEL_TRY(W.part1.reserve((size_t)G1));
    CEL_TRY(W.ctrl.reserve(5));
    if (halo) {
        CEL_TRY(W.hrec.reserve(2 * (size_t)std::max(A.halo_nrows, 1)));
        // the CSR K1 finds the entries of rows with more than kHaloRec halo
        // entries through the per-tile compact row ranges
        CEL_TRY(build_hrow_tile(A, W, ntiles));
    }
    hipStream_t s = rt().stream;
    Ctrl c0{};
    c0.run = 1;
    CEL_HIP(hipMemcpyAsync(W.ctrl.p, &c0, sizeof(Ctrl), hipMemcpyHostToDevice, s));
    MatView V{};
    V.n = n;
    V.xadj = A.xadj.p;
    V.cols = A.cols.p;
    V.vals = A.vals.p;
    V.dvals = A.dia_vals.p;
    V.dmask = A.dia_mask.p;
    V.dmask8 = A.dia_mask8.p;
    V.nd = A.dia_nd;
    V.dzero = -1;
    for (int d = 0; d < A.dia_nd; ++d) {
        V.doff[d] = A.dia_off[d];
        if (A.dia_off[d] == 0) V.dzero = d;
    }
    if (halo) {
        V.hrow_tile = W.hrow_tile.p;
        V.hrows = A.halo_rows.p;
        V.hptr = A.halo_ptr.p;
        V.hcols = A.halo_cols.p;
        V.hvals = A.halo_vals.p;
        V.ghost = ghost;
        V.hrec = W.hrec.p;
        V.hrowq = A.halo_rowq.p;
        V.hflag = A.halo_flag.p;
        V.hwq = A.halo_wq.p;
        V.hnq = A.halo_nrows;
        if (A.halo_nrows > 0)
            hipLaunchKernelGGL(k_halo_rec, dim3((A.halo_nrows + kBlock - 1) / kBlock), dim3(kBlock), 0, s,
                               A.halo_nrows, A.halo_ptr.p, A.halo_cols.p, A.halo_vals.p, ghost, W.hrec.p,
                               W.ctrl.p);
    }
    const Prm P{};
    hipLaunchKernelGGL(k1_kernel<double>(fmt, halo, csr_long_rows(A)), dim3(G1), dim3(kBlock), 0, s, V,
                       x, y, W.part1.p, ResArgs<double>{}, W.ctrl.p, W.ctrl.p + 1, P);
    CEL_HIP(hipGetLastError());
    std::vector<double> part((size_t)G1);
    CEL_HIP(hipMemcpyAsync(part.data(), W.part1.p, sizeof(double) * G1, hipMemcpyDeviceToHost, s));
    CEL_HIP(hipStreamSynchronize(s));
    double acc = 0.0;
    for (int b = 0; b < G1; ++b) acc = acc + part[(size_t)b];
    if (dot) *dot = acc;
    return CEL_OK;
}

// The walks of a wide K1's blocks: the walks whose groups start in the
// same eighth of the matrix's period (its farthest diagonal) go to one XCD,
// so the rows a tile gathers from the planes beside it, and all but the
// outermost of its own plane's neighbours, are in that XCD's L2.  Each block
// keeps its walk's slot, so the partials are the same.  Measured per
// iteration: mixed 100^3 27.0 -> 24.3 us, 200^3 82.0 -> 80.2; FP64 256^3
// 357 -> 351; symmetric diagonals FP64 200^3 198 -> 192.
static int wide_walk(MatView& V, Workspace& W, int G)
{
    const int far = std::max(std::abs(V.doff[0]), std::abs(V.doff[V.nd - 1]));
    const int period = std::max(1, (far + kTileGroup * kTileRows / 2) / (kTileGroup * kTileRows));
    if (G % kXcds || period < 2 * kXcds) return CEL_OK;
    std::vector<int> order(G), w(G);
    for (int b = 0; b < G; ++b) order[b] = b;
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
        return (long long)(a % period) * kXcds / period < (long long)(b % period) * kXcds / period;
    });
    for (int h = 0; h < G; ++h) w[h] = order[(h % kXcds) * (G / kXcds) + h / kXcds];
    CEL_TRY(W.walk.reserve(G));
    CEL_HIP(hipMemcpyAsync(W.walk.p, w.data(), sizeof(int) * G, hipMemcpyHostToDevice, rt().stream));
    CEL_HIP(hipStreamSynchronize(rt().stream));
    V.walk = W.walk.p;
    return CEL_OK;
}

int pcg_solve(Mat& A, const double* b, double* x, const cel_pcg_params& prm, cel_pcg_stats& stats,
              double* hist, bool noalloc)
{
    CEL_TRY(ensure_init());
    hipStream_t s = rt().stream;
    const int n = A.n;
    const bool mixed = prm.precision == CEL_PREC_MIXED;
    // COO (cel_fop_mv_module.f90:357-403) walks the block's row-sorted
    // entries with the CSR kernels, adding each product to v in entry order
    const bool coo = prm.format == CEL_FMT_COO;
    const int fmt = coo ? CEL_FMT_CSR : prm.format;
    const bool halo = prm.use_halo != 0;
    if (fmt != CEL_FMT_CSR && fmt != CEL_FMT_JAD && fmt != CEL_FMT_DIA)
        return fail(CEL_ERR_ARG, "format must be CSR, COO, JAD or DIA");
    if (fmt == CEL_FMT_JAD && (A.jad_mode < 0 || A.jad_ndef != A.jad_mmax))
        return fail(CEL_ERR_STATE, "JAD requested but the matrix has no complete JAD arrays");
    if (fmt == CEL_FMT_DIA && A.dia_nd == 0)
        return fail(CEL_ERR_STATE, "DIA requested but the matrix has no DIA form");
    if (halo && (mixed || fmt == CEL_FMT_JAD))
        return fail(CEL_ERR_ARG, "halo blocks are applied by the FP64 CSR and DIA forms only");
    if (halo && (double)A.halo_nrows * 16.0 >= 2147483648.0 - 64.0)
        return fail(CEL_ERR_ARG, "halo solve: the halo records need 31-bit offsets (< 2^27 halo rows)");
    if (!A.has_jac) return fail(CEL_ERR_STATE, "cel_gpu_mat_set_jacobi has not been called");
    if (A.ncols != n) return fail(CEL_ERR_ARG, "PCG needs a square local block");
    if (prm.iter_max < 0) return fail(CEL_ERR_ARG, "iter_max < 0");
    if (noalloc) {
        if (mixed || halo || fmt == CEL_FMT_JAD)
            return fail(CEL_ERR_ARG, "the allocation-free solve runs FP64 in the CSR, COO or DIA form, "
                                     "without halo blocks");
        if (prm.memspace != CEL_MEM_DEVICE)
            return fail(CEL_ERR_ARG, "the allocation-free solve takes device pointers");
        if (hist) return fail(CEL_ERR_ARG, "the allocation-free solve records no history");
        if ((size_t)n > kNoAllocMaxRows)
            return fail(CEL_ERR_ARG, "the allocation-free solve holds at most " +
                                         std::to_string(kNoAllocMaxRows) + " rows");
        if (rt().device < 0 || rt().device >= kMaxDevices || !g_scratch[rt().device])
            return fail(CEL_ERR_STATE, "no scratch address for this device (cel_gpu_init)");
    }
    if (n == 0) {  // nothing to solve (the kernels assume at least one row)
        stats = cel_pcg_stats{};
        stats.status = CEL_OK;
        return CEL_OK;
    }

    // a JAD solve runs in the permuted row order (vectors gathered on entry,
    // x scattered back on exit), with the columns renumbered into it
    const bool jadp = fmt == CEL_FMT_JAD;
    if (jadp) {
        // the JAD K1 addresses the entries with unsigned 32-bit byte offsets
        const double lim = 4294967296.0 - 64.0;
        if ((double)A.jad_nnz * (mixed ? 4.0 : 8.0) >= lim || (double)n * 8.0 >= lim)
            return fail(CEL_ERR_ARG, "JAD solve: entries beyond the 32-bit offsets of the JAD kernel");
        CEL_TRY(jad_prepare_permuted(A));
    }

    const int ntiles = std::max(1, (n + kTileRows - 1) / kTileRows);
    // grids: K1 variants that must agree share one grid, and so do the
    // residual kernels, and K2 and K3
    const int G1 = k1_grid(ntiles, mixed);
    const int Gr = fixed_grid(fmt == CEL_FMT_JAD ? kResBlocksPerCuJad : kResBlocksPerCu, ntiles);
    int Gv;
    // the residual kernels of a DIA solve use the CSR form
    const int rfmt = fmt == CEL_FMT_DIA ? CEL_FMT_CSR : fmt;
    const bool lr = csr_long_rows(A);
    {
        const long long units = ((long long)n + 2 * kBlock - 1) / (2 * kBlock);
        Gv = (int)std::min<long long>((long long)rt().num_cus * kVecBlocksPerCu,
                                      std::max<long long>(1, units));
        if (Gv >= kXcds) Gv = Gv / kXcds * kXcds;
    }

    if (noalloc && ((size_t)G1 > kNoAllocMaxGrid || (size_t)Gr > kNoAllocMaxGrid ||
                    (size_t)Gv > kNoAllocMaxGrid))
        return fail(CEL_ERR_ARG, "the allocation-free solve holds at most " +
                                     std::to_string(kNoAllocMaxGrid) + " blocks per kernel");

    // workspace: the matrix handle's buffers, or the scratch array
    const size_t nn = n > 0 ? n : 1;
    Workspace* Wp = noalloc ? nullptr : &ws_of(A);
    WorkPtrs w;
    if (noalloc) {
        double* base = static_cast<double*>(g_scratch[rt().device]);
        w.r = base;
        w.p = base + kNoAllocMaxRows;
        w.v = base + 2 * kNoAllocMaxRows;
        w.part1 = base + 3 * kNoAllocMaxRows;
        w.part2 = w.part1 + kNoAllocMaxGrid;
        w.rpart = w.part2 + 2 * kNoAllocMaxGrid;
        w.ctrl = reinterpret_cast<Ctrl*>(base + kNoAllocDoubles);
    } else {
        Workspace& W = *Wp;
        CEL_TRY(W.part1.reserve((size_t)G1));
        CEL_TRY(W.part2.reserve(2 * (size_t)Gv));
        CEL_TRY(W.rpart.reserve(3 * (size_t)Gr));
        CEL_TRY(W.ctrl.reserve(5));
        if (mixed) {
            CEL_TRY(W.r32.alloc(nn));
            CEL_TRY(W.p32.alloc(nn));
            CEL_TRY(W.v32.alloc(nn));
            CEL_TRY(W.e32.alloc(nn));
        } else {
            CEL_TRY(W.r.alloc(nn));
            CEL_TRY(W.p.alloc(nn));
            CEL_TRY(W.v.alloc(nn));
        }
        w.r = W.r.p;
        w.p = W.p.p;
        w.v = W.v.p;
        w.part1 = W.part1.p;
        w.part2 = W.part2.p;
        w.rpart = W.rpart.p;
        w.ctrl = W.ctrl.p;
        w.r32 = W.r32.p;
        w.p32 = W.p32.p;
        w.v32 = W.v32.p;
        w.e32 = W.e32.p;
    }
    const double* db = b;
    double* dx = x;
    if (prm.memspace == CEL_MEM_HOST) {
        Workspace& W = *Wp;
        CEL_TRY(W.b.alloc(nn));
        CEL_TRY(W.x.alloc(nn));
        CEL_HIP(hipMemcpyAsync(W.b.p, b, sizeof(double) * n, hipMemcpyHostToDevice, s));
        if (prm.x0_mode == CEL_X0_USER)
            CEL_HIP(hipMemcpyAsync(W.x.p, x, sizeof(double) * n, hipMemcpyHostToDevice, s));
        db = W.b.p;
        dx = W.x.p;
    }
    double* const dx_out = dx;
    const double* jac64 = A.jac.p;
    const float* jac32 = A.jac32.p;
    if (jadp) {
        Workspace& W = *Wp;
        CEL_TRY(W.bp.alloc(nn));
        CEL_TRY(W.xp.alloc(nn));
        CEL_TRY(W.jacp.alloc(nn));
        if (mixed) CEL_TRY(W.jacp32.alloc(nn));
        jac64 = W.jacp.p;
        jac32 = mixed ? W.jacp32.p : nullptr;
    }
    const int hist_cap = hist ? prm.iter_max + 1 : 0;
    if (hist_cap) CEL_TRY(Wp->hist.alloc(hist_cap));
    if (halo) {
        Workspace& W = *Wp;
        CEL_TRY(W.ghost.alloc(A.ghost_len > 0 ? A.ghost_len : 1));
        CEL_TRY(W.sendbuf.alloc(A.send_total > 0 ? A.send_total : 1));
        hipLaunchKernelGGL(k_fill, dim3(64), dim3(kBlock), 0, s, (long long)W.ghost.n, W.ghost.p, 0.0);
        CEL_TRY(W.hrec.reserve(2 * (size_t)std::max(A.halo_nrows, 1)));
        CEL_TRY(build_hrow_tile(A, W, ntiles));
    }

    // the form the K1s run on, and its residual's: the caller's, or a derived
    // one with the same bits (its grids are the caller's form's).  It is built
    // in what the solve's own memory, above, has left.
    int use = Derived::kNone;
    bool symmetric = false;
    DerivedUse reading;
    if (!noalloc && !halo && !coo && fmt != CEL_FMT_JAD) {
        reading.begin(A.derived);
        use = derived_prepare(A, fmt, mixed, prm.iter_max, &symmetric);
        if (use == Derived::kNone) reading.end();
    }
    const int kfmt = use == Derived::kClasses ? kFmtClass : use == Derived::kDiagonals ? CEL_FMT_DIA : fmt;
    const int kres = use == Derived::kClasses ? kFmtClass : rfmt;

    // matrix data for the mixed inner operator (once per matrix)
    if (mixed) {
        if (fmt == CEL_FMT_DIA && kfmt == CEL_FMT_DIA) CEL_TRY(dia_prepare_f32(A));
        // the DIA K1 reads dia_vals32 and the residual kernels the FP64 CSR
        // values, so only a CSR solve needs the FP32 CSR copy
        if (kfmt == CEL_FMT_CSR && !A.vals32.p) {
            CEL_TRY(A.vals32.alloc(A.nnz > 0 ? A.nnz : 1));
            CEL_TRY(launch_to_f32(A.vals.p, A.vals32.p, A.nnz));
        }
        if (fmt == CEL_FMT_JAD && !A.jad_vals32.p) {
            CEL_TRY(A.jad_vals32.alloc(A.jad_nnz > 0 ? A.jad_nnz : 1));
            CEL_TRY(launch_to_f32(A.jad_vals.p, A.jad_vals32.p, A.jad_nnz));
        }
    }

    const std::string err = last_error();  // (what is tried and not had below is no error of the solve)
    // the longest row: known from the start for matrices from host arrays and
    // of the generators, otherwise looked up once
    bool deep = false;
    if (kfmt == CEL_FMT_CSR && !lr && !halo && !noalloc) {
        if (A.longest < 0 && block_longest(A, A.longest) != CEL_OK) {
            A.longest = -1;
            set_error(err);
        }
        deep = deep_rows(A);
    }
    // two kernels per iteration on small systems; the halo blocks need a
    // stored direction before the product, profiling a product of its own (and
    // symmetric diagonals the wide walk, which a step does not have)
    bool step = !noalloc && !halo && !prm.profile && use == Derived::kNone && !symmetric && !deep &&
                step_form(A, fmt, mixed);
    double *pbuf[2] = {w.p, nullptr}, *zbuf = nullptr;
    float *pbuf32[2] = {w.p32, nullptr}, *zbuf32 = nullptr;
    if (step) {
        Workspace& W = *Wp;
        if (mixed) {
            step = W.p2_32.alloc(nn) == CEL_OK && W.z32.alloc(nn) == CEL_OK;
            pbuf32[1] = W.p2_32.p;
            zbuf32 = W.z32.p;
        } else {
            step = W.p2.alloc(nn) == CEL_OK && W.z.alloc(nn) == CEL_OK;
            pbuf[1] = W.p2.p;
            zbuf = W.z.p;
        }
        if (!step) set_error(err);  // no memory for them: three kernels
    }
    Prm P{};
    P.tol = prm.tol;
    P.tol_mode = prm.tol_mode;
    P.iter_max = prm.iter_max;
    P.small = 1.1 * 2.220446049250313e-16;  // cel_real_small (cel_types_module.f90:33)
    P.ru_delta = prm.ru_delta > 0 ? prm.ru_delta : 0.1;
    P.ru_restart = prm.ru_restart;
    P.alpha_stop = prm.alpha_stop;
    P.ru_max_inner = 1000;
    P.hist = hist_cap ? Wp->hist.p : nullptr;
    P.hist_cap = hist_cap;
    // every solve starts from a fresh token (the scratch array keeps the
    // last call's contents; everything else is written before it is read)
    hipLaunchKernelGGL(k_token, dim3(1), dim3(64), 0, s, w.ctrl);
    int* progress = nullptr;
    if (!noalloc) {
        CEL_TRY(Wp->host_alloc());
        Wp->host->progress = 0;
        progress = &Wp->host->progress;
    }
    // token slots: 0 -> K1 -> 1 -> K2 -> 2 -> K3 -> 0 (FP64);
    // (two-kernel form: 0 -> step -> 1 -> K2 -> 0)
    Ctrl* C0 = w.ctrl;
    Ctrl* C1 = w.ctrl + 1;
    Ctrl* C2 = w.ctrl + 2;
    Ctrl* C3 = w.ctrl + 3;

    MatView V{};
    V.n = n;
    V.coo = coo ? 1 : 0;
    V.mmax = A.jad_mmax;
    V.jnnz = A.jad_nnz;
    V.xadj = A.xadj.p;
    V.cols = A.cols.p;
    V.vals = A.vals.p;
    V.vals32 = A.vals32.p;
    V.jbegin = A.jad_begin.p;
    V.jcols = jadp ? A.jad_pcols.p : A.jad_cols.p;
    V.jperm = A.jad_perm.p;
    V.jvals = A.jad_vals.p;
    V.jvals32 = A.jad_vals32.p;
    V.dvals = A.dia_vals.p;
    V.dvals32 = A.dia_vals32.p;
    V.dmask = A.dia_mask.p;
    V.dmask8 = A.dia_mask8.p;
    V.nd = A.dia_nd;
    const int* doff = A.dia_off;
    if (use != Derived::kNone) {
        const Derived& D = A.derived;
        V.nd = D.nd;
        doff = D.off;
        V.cls = D.cls.p;
        V.ctab = D.classes();
        V.dvals = D.vals.p;
        V.dvals32 = D.vals32.p;
        V.dmask = nullptr;
        V.dmask8 = D.mask8.p;
    }
    V.dzero = -1;
    for (int d = 0; d < V.nd; ++d) {
        V.doff[d] = doff[d];
        if (doff[d] == 0) V.dzero = d;
    }
    const bool sym = kfmt == CEL_FMT_DIA && symmetric;
    V.dwide = sym;
    const int arrays = sym ? dia_bases(n, V.nd, V.doff, true, V.dbase) : V.nd;
    // (a symmetric block's values are read again a row, a line and a plane
    // later: 256^3 FP64 427 us per iteration marked as read once, 425 kept)
    const bool keep = sym || keep_matrix(A, kfmt, arrays, mixed);
    // long rows in a narrow band: the band is looked up once per matrix
    bool win = false;
    if (kfmt == CEL_FMT_CSR && lr && !mixed && !halo && !noalloc && n >= kWindowRows &&
        (A.band >= 0 || prm.iter_max >= 32)) {
        if (A.band < 0 && block_bandwidth(A, A.band) != CEL_OK) {  // without the window
            A.band = -1;
            set_error(err);
        }
        win = window_fits(A);
        V.band = A.band;
    }
    if ((use == Derived::kClasses || sym) && wide_walk(V, *Wp, G1) != CEL_OK) set_error(err);  // each block its own walk
    if (halo) {
        V.hrow_tile = Wp->hrow_tile.p;
        V.hrows = A.halo_rows.p;
        V.hrowq = A.halo_rowq.p;
        V.hptr = A.halo_ptr.p;
        V.hcols = A.halo_cols.p;
        V.hvals = A.halo_vals.p;
        V.ghost = Wp->ghost.p;
        V.hrec = Wp->hrec.p;
        V.hflag = A.halo_flag.p;
        V.hwq = A.halo_wq.p;
        V.hnq = A.halo_nrows;
    }

    // the allocation-free solve creates no events: it times with the host
    // clock around a synchronised stream
    StreamScope R(s);
    hipEvent_t e0 = nullptr, e1 = nullptr, e2 = nullptr;
    const auto t_host0 = std::chrono::steady_clock::now();
    if (!noalloc) {
        CEL_TRY(R.event(e0));
        CEL_TRY(R.event(e1));
        CEL_TRY(R.event(e2));
        CEL_HIP(hipEventRecord(e0, s));
    }
    if (jadp) {
        Workspace& W = *Wp;
        const int gp = std::max(1, std::min(Gv * 2, 4096));
        hipLaunchKernelGGL(k_perm_gather<double>, dim3(gp), dim3(kBlock), 0, s, (long long)n,
                           A.jad_perm.p, db, W.bp.p);
        hipLaunchKernelGGL(k_perm_gather<double>, dim3(gp), dim3(kBlock), 0, s, (long long)n,
                           A.jad_perm.p, A.jac.p, W.jacp.p);
        if (mixed)
            hipLaunchKernelGGL(k_perm_gather<float>, dim3(gp), dim3(kBlock), 0, s, (long long)n,
                               A.jad_perm.p, A.jac32.p, W.jacp32.p);
        if (prm.x0_mode == CEL_X0_USER)
            hipLaunchKernelGGL(k_perm_gather<double>, dim3(gp), dim3(kBlock), 0, s, (long long)n,
                               A.jad_perm.p, dx, W.xp.p);
        CEL_HIP(hipGetLastError());
        db = W.bp.p;
        dx = W.xp.p;
    }

    // x0 (cel_cgalg_module.f90:209 uses 1.0)
    if (prm.x0_mode != CEL_X0_USER)
        hipLaunchKernelGGL(k_fill, dim3(std::max(1, std::min(Gv * 2, 4096))), dim3(kBlock), 0, s,
                           (long long)n, dx, prm.x0_mode == CEL_X0_ONE ? 1.0 : 0.0);
    if (halo) CEL_TRY(launch_face_pack(A, dx, Wp->sendbuf.p));

    // r0, p0 and their partials; the first K1 folds them in.  The set-up
    // reads and writes token slot 0 (only block 0 writes, after its read).
    const ResArgs<double> R64{dx, db, jac64, nullptr, w.r, w.p, nullptr, w.rpart, Gr};
    const ResArgs<float> R32{dx, db, nullptr, jac32, w.r32, w.p32, w.e32, w.rpart, Gr};
    if (!mixed)
        hipLaunchKernelGGL(res_kernel<double>(kres, halo, lr), dim3(Gr), dim3(kBlock), 0, s, V, R64, C0, C0);
    else
        hipLaunchKernelGGL(res_kernel<float>(kres, false, lr), dim3(Gr), dim3(kBlock), 0, s, V, R32, C0, C0);
    CEL_HIP(hipGetLastError());
    if (!noalloc) CEL_HIP(hipEventRecord(e1, s));

    // profiling events around K1
    std::vector<hipEvent_t> pev;
    int pev_used = 0;
    auto prof_event = [&]() -> hipEvent_t {
        if (pev_used == (int)pev.size()) {
            hipEvent_t ev;
            if (R.event(ev) < 0) return nullptr;
            pev.push_back(ev);
        }
        return pev[pev_used++];
    };

    const long long n_ll = n;
    // the vector kernels' Jacobi values: the vector, or the classes' table
    const bool bycls = use == Derived::kClasses;
    const double* vjac64 = bycls ? V.ctab.jac64 : jac64;
    const float* vjac32 = bycls ? V.ctab.jac32 : jac32;
    const uint8_t *vcls = bycls ? V.cls : nullptr, *nocls = nullptr;
    const int stream = stream_level(n, mixed, bycls, sym ? arrays : 0);
    A.path = SolvePath{bycls                    ? "classes"
                       : kfmt == CEL_FMT_CSR ? (lr ? "csr-long" : "csr")
                       : kfmt == CEL_FMT_DIA ? "dia"
                                             : "jad",
                       step, step && step_direct(fmt, n, mixed), win, bycls || sym, deep, step || (keep && !halo && !bycls),
                       step ? 0 : stream};
    // One slot of the two-kernel form: the step finishes the iteration before
    // (its vectors and scalars) and forms the next product, K2 updates r.
    // The direction alternates between two buffers by slot.
    auto enqueue_step = [&](long long slot) -> int {
        const int in = (int)(slot & 1), out = in ^ 1;
        if (!mixed) {
            hipLaunchKernelGGL(step_kernel<double>(fmt, n), dim3(G1), dim3(kBlock), 0, s, V,
                               (const double*)pbuf[in], (const double*)zbuf, pbuf[out], dx, (double*)nullptr, w.v,
                               w.part1, R64, (const double*)w.part2, Gv, (const Ctrl*)C0, C1, P);
            hipLaunchKernelGGL((k_pcg_update_r<double, true, false>), dim3(Gv), dim3(kBlock), 0, s, n_ll, w.r, w.v,
                               jac64, nocls, zbuf, w.part2, w.part1, G1, C1, C0, progress);
        } else {
            ResArgs<float> R = R32;
            R.p = pbuf32[out];  // a restart's direction
            hipLaunchKernelGGL(step_kernel<float>(fmt, n), dim3(G1), dim3(kBlock), 0, s, V,
                               (const float*)pbuf32[in], (const float*)zbuf32, pbuf32[out], w.e32, dx, w.v32,
                               w.part1, R, (const double*)w.part2, Gv, (const Ctrl*)C0, C1, P);
            hipLaunchKernelGGL((k_pcg_update_r<float, true, false>), dim3(Gv), dim3(kBlock), 0, s, n_ll, w.r32, w.v32,
                               jac32, nocls, zbuf32, w.part2, w.part1, G1, C1, C0, progress);
        }
        CEL_HIP(hipGetLastError());
        return CEL_OK;
    };
    auto enqueue_iter = [&](bool profile, long long slot) -> int {
        if (step) return enqueue_step(slot);
        hipEvent_t ea = nullptr, eb = nullptr;
        if (halo) {
            CEL_TRY(launch_face_pack(A, w.p, Wp->sendbuf.p));
            // (a multi-GPU solve exchanges the faces here, then:)
            if (A.halo_nrows > 0)
                hipLaunchKernelGGL(k_halo_rec, dim3((A.halo_nrows + kBlock - 1) / kBlock), dim3(kBlock),
                                   0, s, A.halo_nrows, A.halo_ptr.p, A.halo_cols.p,
                                   A.halo_vals.p, Wp->ghost.p, Wp->hrec.p, C0);
        }
        if (profile) {
            ea = prof_event();
            eb = prof_event();
            if (!ea || !eb) return fail(CEL_ERR_HIP, "hipEventCreate failed");
            CEL_HIP(hipEventRecord(ea, s));
        }
        if (!mixed) {
            const auto k1 = !win ? k1_kernel<double>(kfmt, halo, lr, keep, deep)
                            : keep ? k_pcg_window<true> : k_pcg_window<false>;
            hipLaunchKernelGGL(k1, dim3(G1), dim3(kBlock), 0, s, V, w.p, w.v,
                               w.part1, R64, C0, C1, P);
            if (profile) CEL_HIP(hipEventRecord(eb, s));
            hipLaunchKernelGGL(k2_kernel<double>(bycls, stream), dim3(Gv), dim3(kBlock), 0, s, n_ll, w.r, w.v, vjac64,
                               vcls, (double*)nullptr, w.part2, w.part1, G1, C1, C2, (int*)nullptr);
            hipLaunchKernelGGL(k3_kernel<double>(bycls, stream), dim3(Gv), dim3(kBlock), 0, s, n_ll, dx, w.p, w.r,
                               vjac64, vcls, nullptr, w.part2, Gv, C2, C0, P, progress);
        } else {
            hipLaunchKernelGGL(k1_kernel<float>(kfmt, false, lr, keep, deep), dim3(G1), dim3(kBlock), 0, s, V, w.p32, w.v32,
                               w.part1, R32, C0, C1, P);
            if (profile) CEL_HIP(hipEventRecord(eb, s));
            hipLaunchKernelGGL(k2_kernel<float>(bycls, stream), dim3(Gv), dim3(kBlock), 0, s, n_ll, w.r32, w.v32,
                               vjac32, vcls, (float*)nullptr, w.part2, w.part1, G1, C1, C2, (int*)nullptr);
            hipLaunchKernelGGL(k3_kernel<float>(bycls, stream), dim3(Gv), dim3(kBlock), 0, s, n_ll, w.e32, w.p32,
                               w.r32, vjac32, vcls, dx, w.part2, Gv, C2, C0, P, progress);
        }
        CEL_HIP(hipGetLastError());
        return CEL_OK;
    };

    // iteration loop.  The loop needs at most iter_max iterations plus one
    // K1 that folds in the final partials.  The host runs a few slots ahead
    // of the progress word, so few launches find the solve stopped (a flag
    // copied back every 16 iterations, one chunk late, left 17 to 47 of them
    // and a copy a chunk: 1.78 against 1.51 ms for a 32^3 solve of 104
    // iterations); replayed graphs go chunk by chunk, one chunk ahead.  The
    // allocation-free solve, which has no host memory, reads the token after
    // every chunk.
    const bool use_graph = prm.use_graph && !prm.profile && !noalloc;
    long long chunk = prm.check_every > 0 ? prm.check_every : 16;
    const long long ahead = std::min(std::max(chunk, 2LL), 8LL);
    // a captured chunk of the two-kernel form starts at an even slot
    if (use_graph && step && (chunk & 1)) chunk *= 2;
    int hrun_sync = 1;

    int status = CEL_OK;
    // mixed: a replacement takes a slot, or two (the request of the two-kernel
    // form), and there is at most one per iteration
    const long long budget = (long long)(mixed ? (step ? 3 : 2) : 1) * ((long long)prm.iter_max + 1);
    long long enqueued = 0;
    while (enqueued < budget) {
        const int c = (int)std::min<long long>(use_graph || noalloc ? chunk : 1, budget - enqueued);
        if (use_graph && c == chunk) {
            if (!R.exec) {
                CEL_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
                for (int i = 0; i < c; ++i) {
                    int rc = enqueue_iter(false, i);
                    if (rc < 0) {
                        (void)hipStreamEndCapture(s, &R.graph);
                        return rc;
                    }
                }
                CEL_HIP(hipStreamEndCapture(s, &R.graph));
                CEL_HIP(hipGraphInstantiate(&R.exec, R.graph, nullptr, nullptr, 0));
            }
            CEL_HIP(hipGraphLaunch(R.exec, s));
        } else {
            for (int i = 0; i < c; ++i) {
                status = enqueue_iter(prm.profile != 0 && !noalloc, enqueued + i);
                if (status < 0) break;
            }
            if (status < 0) break;
        }
        enqueued += c;
        if (noalloc) {
            CEL_HIP(hipMemcpyAsync(&hrun_sync, &C0->run, sizeof(int), hipMemcpyDeviceToHost, s));
            CEL_HIP(hipStreamSynchronize(s));
            if (!hrun_sync) break;
            continue;
        }
        status = wait_progress(s, progress, enqueued - (use_graph ? chunk : ahead));
        if (status <= 0) break;
        status = CEL_OK;
    }
    if (mixed) {
        // a budget that ran out mid-way leaves a correction in e: fold it in
        hipLaunchKernelGGL(k_ru_flush, dim3(Gv), dim3(kBlock), 0, s, n_ll, dx, w.e32, C0, C3, 1);
    }
    if (jadp) {  // x back to the original row order
        hipLaunchKernelGGL(k_perm_scatter<double>, dim3(std::max(1, std::min(Gv * 2, 4096))),
                           dim3(kBlock), 0, s, n_ll, A.jad_perm.p, dx, dx_out);
        CEL_HIP(hipGetLastError());
    }
    if (!noalloc) CEL_HIP(hipEventRecord(e2, s));
    Ctrl out;
    if (noalloc) {
        CEL_HIP(hipStreamSynchronize(s));
        if (status < 0) return status;
        CEL_HIP(hipMemcpy(&out, C0, sizeof(Ctrl), hipMemcpyDeviceToHost));
    } else {
        CEL_HIP(hipMemcpyAsync(&Wp->host->ctrl, C0, sizeof(Ctrl), hipMemcpyDeviceToHost, s));
        CEL_HIP(hipStreamSynchronize(s));
        if (status < 0) return status;
        out = Wp->host->ctrl;
    }
    float ms_setup = 0, ms_all = 0;
    if (!noalloc) {
        CEL_HIP(hipEventElapsedTime(&ms_setup, e0, e1));
        CEL_HIP(hipEventElapsedTime(&ms_all, e0, e2));
    } else {
        ms_all = (float)std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() -
                                                                  t_host0)
                     .count();
    }
    double spmv_ms = 0;
    int spmv_n = 0;
    for (int i = 0; i + 1 < pev_used; i += 2) {
        float t = 0;
        if (hipEventElapsedTime(&t, pev[i], pev[i + 1]) == hipSuccess) {
            spmv_ms += t;
            ++spmv_n;
        }
    }

    if (prm.memspace == CEL_MEM_HOST)
        CEL_HIP(hipMemcpy(x, dx_out, sizeof(double) * n, hipMemcpyDeviceToHost));
    if (hist && hist_cap) {
        int cnt = std::min(out.iter + 1, hist_cap);
        CEL_HIP(hipMemcpy(hist, Wp->hist.p, sizeof(double) * cnt, hipMemcpyDeviceToHost));
    }

    stats.iters = out.iter;
    stats.outer_iters = out.outer;
    stats.norm0 = out.norm0;
    stats.final_norm = out.norm2;
    stats.eps_abs = out.eps;
    stats.alpha = out.alpha;
    stats.solve_ms = ms_all;
    stats.setup_ms = ms_setup;
    stats.spmv_ms = spmv_ms;
    stats.spmv_launches = spmv_n;
    const int prec = mixed ? CEL_PREC_MIXED : CEL_PREC_FP64;
    const double vb = mixed ? 4.0 : 8.0;
    stats.spmv_bytes = spmv_bytes(A, fmt, prec);
    if (jadp) stats.spmv_bytes -= 4.0 * n;  // the permuted-order K1 reads no permutation
    // a derived form: a class or mask byte per row, the diagonals' values, p and v
    if (use != Derived::kNone || sym) stats.spmv_bytes = (1.0 + (bycls ? 2.0 : 2.0 + arrays) * vb) * n;
    {
        // K1 matrix + p gather + v write ; K2 r,v,jac read + r write ;
        // K3 p,r,jac,x read + p,x write
        // (by classes: a byte for the Jacobi value in each)
        stats.iter_bytes = stats.spmv_bytes + vb * n * 4.0 + vb * n * 6.0 - (bycls ? 2.0 * (vb - 1.0) * n : 0.0) +
                           (halo ? 20.0 * A.send_total + 12.0 * A.ghost_len : 0.0);
    }
    if (out.status != 0) {
        stats.status = out.status;
        return fail(out.status, out.status == CEL_ERR_BREAKDOWN
                                    ? "PCG breakdown: p.Ap <= 0 or not finite"
                                    : "non-finite right-hand side");
    }
    const bool converged = out.norm2 <= out.eps;
    stats.status = converged ? CEL_OK : CEL_NOT_CONVERGED;
    if (!converged && out.iter < prm.iter_max && prm.alpha_stop && !(std::fabs(out.alpha) > P.small))
        stats.status = CEL_OK;  // stopped on |alpha| <= 1.1 eps (reference condition)
    return stats.status;
}

void pcg_release_workspace(Mat* A)
{
    delete A->ws;
    A->ws = nullptr;
}

}  // namespace cel

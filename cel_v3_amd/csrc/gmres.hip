// gmres.hip -- Jacobi-GMRES(m) in HBM, the element solver's default method.
//
// Replaces cel_gmresalg_2jacobi (src/fcgalg/cel_gmresalg_module.f90:570-851)
// with one rank.  The op sequence is the reference's:
//   x = 1 ; while iter <= iter_max and not converged:
//     iter += 1 ; r = b - A x ; beta = ||r||
//     up to m+1 cycles:
//       v1 = r * (1/beta) ; gamma1 = beta
//       for j = 1..m:  z_j = v_j * jac ; w = A z_j
//                      for i = 1..j: h_ij = v_i . w ; w = w - h_ij v_i
//                      h_j+1,j = ||w|| ; rotate column j (as the reference
//                      writes it, :722-727: both statements assign h_ij, so
//                      h_i+1,j is never rotated) ; new rotation ; gamma
//                      if |gamma_j+1| <= eps: x += sum alpha_i z_i, stop
//                      v_j+1 = w / h_j+1,j
//       if not stopped: x += sum alpha_i z_i (back substitution on m)
//       r = b - A x ; beta = ||r||
// Element-wise steps round every product before the add, as the reference's
// loops do.
//
// Everything stays on the device; the host only enqueues.  The scalars (the
// Hessenberg columns, rotations, gamma, residual norms, counters and stop
// flags) live in one state record in HBM.  Each vector kernel writes
// per-block partial sums over fixed contiguous chunks; the next kernel sums
// them in a fixed order, in every block, so the result depends on n only,
// never on timing.  In the CSR and DIA forms the products w = A z_j and r =
// b - A x form the partials of v_1 . w and r . r themselves, over the same
// chunks and in the same order as the separate dot kernels the JAD form runs
// after its product, so all three forms give the same bits.
//
// The small algebra has no launch of its own: the kernel that needs a norm
// (the one that forms v_j+1, or the cycle's x update) sums its partials and
// rotates the column in every block, in the reference's order, and block 0
// records the result.  Every state field a kernel writes is one that no
// other block of that kernel reads (raw and rotated columns, and gamma before
// and after its rotation, are kept apart), and the convergence flag names
// its column, so a block that starts late does not mistake it for an
// earlier one.  Partials alternate between two buffers.  On small systems the
// product that follows forms v_j and z_j itself (k_col); a cycle of
// GMRES(3) is then 11 launches, 14 otherwise.
//
// One outer iteration (its residual and m+1 cycles) is captured once as a
// hipGraph and replayed up to iter_max+1 times; after a replay the host
// reads the stop flag (one replay in flight).  Once the solve has converged
// every kernel of the rest of the graph returns at once: the kernels of
// later columns and cycles test `halt` (set at convergence), the cycle's
// closing residual and everything after it test `stop` (set after that
// residual).  v_m+1 is not formed (nothing reads it).
#include <cmath>
#include <string>
#include <utility>

#include "cel_internal.hpp"
#include "device_common.hpp"
#include "spmv_device.hpp"

namespace cel {
namespace {

constexpr int kThreads = 256;
constexpr int kMaxRestart = 32;
constexpr int kM1 = kMaxRestart + 2;  // 1-based index range of the small arrays
constexpr int kNoColumn = 1 << 20;    // halt without a converged column
constexpr int kWide = 1024;           // threads of the kernels of small systems
constexpr int kWideRows = 2048;       // rows of a chunk there

struct GmState {
    double H[kM1 * kM1];  // h(i, j) = H[i * kM1 + j], 1-based, as the Gram-Schmidt passes leave it
    double R[kM1 * kM1];  // the rotated columns
    double cs[kM1], sn[kM1];
    double gin[kM1], gam[kM1];  // gamma(j) as column j finds it, and after its rotation
    double residuum, norm0, eps;
    int iter, cycles, ncols;  // outer iterations, cycles, Arnoldi columns run
    int halt;                 // the column that converged (0: none): later columns and cycles do nothing
    int stop;                 // nothing runs any more
    int status;               // 0 or CEL_ERR_NONFINITE
    int pad[2];
};

// Sum over the first 256 threads of the block in block_sum's order, in every
// thread; red as block_sum_all.
__device__ __forceinline__ double sum256(double v, double* red)
{
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0 && wave < kWaves) red[wave] = v;
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) s = s + red[w];
    return s;
}

// The calling thread's part of a fold of the G partials; sum256 of the parts
// is their sum in a fixed order.
__device__ __forceinline__ double fold_part(const double* __restrict__ part, int G)
{
    return threadIdx.x < kBlock ? strided_sum(part, G) : 0.0;
}

// The terms f(i) of the block's chunk [c0, c1) summed into its partial: 256
// threads take rows 256 apart in ascending order, then block_sum's order.  A
// block of more threads evaluates the rows side by side and adds them from
// LDS in that same order.
template <int T, typename F>
__device__ __forceinline__ void chunk_partial(long long c0, long long c1, F&& f, double* __restrict__ part,
                                              double* red, double* terms /* chunk, T > 256 only */)
{
    double acc = 0.0;
    if constexpr (T == kBlock) {
        for (long long i = c0 + threadIdx.x; i < c1; i += T) acc = acc + f(i);
    } else {
        for (long long i = c0 + threadIdx.x; i < c1; i += T) terms[i - c0] = f(i);
        __syncthreads();
        if (threadIdx.x < kBlock)
            for (int i = threadIdx.x; i < (int)(c1 - c0); i += kBlock) acc = acc + terms[i];
    }
    const double s = sum256(acc, red);
    if (threadIdx.x == 0) part[blockIdx.x] = s;
}

#define CHUNK_BOUNDS                                                         \
    const long long c0 = (long long)blockIdx.x * chunk;                      \
    const long long c1 = c0 + chunk < n ? c0 + chunk : n;
#define CHUNK_LOOP(i)                                                        \
    CHUNK_BOUNDS                                                             \
    for (long long i = c0 + threadIdx.x; i < c1; i += blockDim.x)

__global__ void __launch_bounds__(kThreads)
k_fill(long long n, long long chunk, double* __restrict__ x, double v)
{
    CHUNK_LOOP(i) x[i] = v;
}

// Zeroes the state record (all threads of one block, 8 bytes each) and sets eps.
static_assert(sizeof(GmState) % 8 == 0, "GmState is cleared in 8-byte words");
__global__ void __launch_bounds__(kThreads) k_state_init(GmState* st, double eps)
{
    unsigned long long* w = reinterpret_cast<unsigned long long*>(st);
    for (int i = threadIdx.x; i < (int)(sizeof(GmState) / 8); i += kThreads) w[i] = 0ull;
    __syncthreads();
    if (threadIdx.x == 0) st->eps = eps;
}

// r = b - r ; partial r . r
__global__ void __launch_bounds__(kThreads)
k_resid(long long n, long long chunk, const double* __restrict__ b, double* __restrict__ r,
        double* __restrict__ part, const GmState* __restrict__ st)
{
    __shared__ double red[kWaves];
    if (st->stop) return;
    CHUNK_BOUNDS
    chunk_partial<kThreads>(c0, c1, [&](long long i) {
        const double ri = b[i] - r[i];
        r[i] = ri;
        const double p = ri * ri;
        return p;
    }, part, red, nullptr);
}

// After the closing residual of a cycle (CYCLE) or the first one of an outer
// iteration: residuum = ||r|| from its partials; returns it, or a negative
// number where nothing more runs.  A cycle that converged ends the solve.
// Every thread of the block; block 0 records.
__device__ __forceinline__ double residual_done(bool cycle, double folded, GmState* st, double* red)
{
    const int halt = st->halt;
    const double res = sqrt(sum256(folded, red));
    const bool end = cycle ? halt != 0 : !isfinite(res);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        st->residuum = res;
        if (cycle) {
            st->cycles = st->cycles + 1;
        } else {
            st->iter = st->iter + 1;
            if (st->iter == 1) st->norm0 = res;
            if (end) {
                st->status = CEL_ERR_NONFINITE;
                st->halt = kNoColumn;
            }
        }
        if (end) st->stop = 1;
    }
    return end ? -1.0 : res;
}

// End of the last cycle of an outer iteration (one block).
__global__ void __launch_bounds__(kThreads)
k_cycle_end(const double* __restrict__ part, int G, GmState* st)
{
    __shared__ double red[kWaves];
    const double f = fold_part(part, G);
    if (st->stop) return;
    (void)residual_done(true, f, st, red);
}

// v1 = r * (1/beta) ; z1 = v1 * jac ; gamma1 = beta
__global__ void __launch_bounds__(kThreads)
k_scale_jac(long long n, long long chunk, int cycle, const double* __restrict__ part, int G,
            const double* __restrict__ r, const double* __restrict__ jac, double* __restrict__ v,
            double* __restrict__ z, GmState* st)
{
    __shared__ double red[kWaves];
    const double f = fold_part(part, G);  // (the loads do not wait for the flag)
    if (st->stop) return;
    const double beta = residual_done(cycle, f, st, red);
    if (beta < 0.0) return;  // uniform
    const double tmp = 1.0 / beta;
    CHUNK_LOOP(i) {
        const double vi = r[i] * tmp;
        v[i] = vi;
        z[i] = vi * jac[i];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) st->gin[1] = beta;
}

// partial a . b
__global__ void __launch_bounds__(kThreads)
k_dot(long long n, long long chunk, const double* __restrict__ a, const double* __restrict__ b,
      double* __restrict__ part, const GmState* __restrict__ st)
{
    __shared__ double red[kWaves];
    if (st->halt) return;
    CHUNK_BOUNDS
    chunk_partial<kThreads>(c0, c1, [&](long long i) {
        const double p = a[i] * b[i];
        return p;
    }, part, red, nullptr);
}

// h_ii,jj = sum(prev partials) ; w = w - h vi ; partial (next ? next . w : w . w)
template <int T>
__global__ void __launch_bounds__(T)
k_mgs(long long n, long long chunk, int ii, int jj, const double* __restrict__ prev, int G,
      const double* __restrict__ vi, double* __restrict__ w, const double* __restrict__ next,
      double* __restrict__ part, GmState* st)
{
    __shared__ double red[2 * kWaves];
    __shared__ double terms[T == kThreads ? 1 : kWideRows];
    const double f = fold_part(prev, G);
    if (st->halt) return;
    const double h = sum256(f, red + kWaves);
    if (blockIdx.x == 0 && threadIdx.x == 0) st->H[ii * kM1 + jj] = h;
    CHUNK_BOUNDS
    chunk_partial<T>(c0, c1, [&](long long i) {
        const double t = h * vi[i];
        const double wi = w[i] - t;
        w[i] = wi;
        const double p = (next ? next[i] : wi) * wi;
        return p;
    }, part, red, terms);
}

// What a block knows after a column (LDS).
struct Column {
    double h[kM1], cs[kM1], sn[kM1], gam[kM1], alp[kM1];
    double R[kMaxRestart * (kMaxRestart + 1) / 2];  // the rotated columns before it, packed
    int k;  // coefficients of the x update in alp (0: none)
};

// After the last Gram-Schmidt pass of column jj: h_jj+1,jj = sqrt(sum of its
// partials) ; the column's rotations as the reference writes them ; new
// rotation ; gamma ; convergence test ; the back-substitution coefficients
// (cel_gmresalg_module.f90:760-772 order) when the column converged or is
// the cycle's last.  Every thread of the block; the algebra runs in one
// thread over LDS, block 0 records it.
__device__ __forceinline__ void column_done(int jj, int m, double folded, GmState* st, Column& c,
                                            double* red)
{
    const int tid = threadIdx.x;
    if (tid <= jj && tid > 0) c.h[tid] = st->H[tid * kM1 + jj];
    if (tid < jj && tid > 0) {
        c.cs[tid] = st->cs[tid];
        c.sn[tid] = st->sn[tid];
        c.gam[tid] = st->gam[tid];
    }
    if (tid == 0) c.gam[jj] = st->gin[jj];
    for (int q = tid; q < jj * (jj - 1) / 2; q += blockDim.x) {
        int k = 1, at = q;  // entry (i, k), i <= k < jj
        while (at >= k) at -= k++;
        c.R[q] = st->R[(at + 1) * kM1 + k];
    }
    const double s = sum256(folded, red);  // (synchronises)
    if (tid == 0) {
        c.h[jj + 1] = sqrt(s);
        for (int ii = 1; ii <= jj - 1; ++ii) {  // both statements assign h(ii,jj) (:722-727)
            double a = c.h[ii] * c.cs[ii];
            double d = c.h[ii + 1] * c.sn[ii];
            c.h[ii] = a + d;
            a = -c.h[ii] * c.sn[ii];
            d = c.h[ii + 1] * c.cs[ii];
            c.h[ii] = a + d;
        }
        const double a = c.h[jj] * c.h[jj];
        const double d = c.h[jj + 1] * c.h[jj + 1];
        const double betta = sqrt(a + d);
        const double sn = c.h[jj + 1] / betta, cs = c.h[jj] / betta;
        const double gnext = -sn * c.gam[jj];
        c.h[jj] = betta;
        c.gam[jj] = cs * c.gam[jj];
        const bool conv = fabs(gnext) <= st->eps;
        c.k = conv || jj == m ? jj : 0;
        for (int ii = c.k; ii >= 1; --ii) {
            double sum = 0.0;
            for (int kk = ii + 1; kk <= c.k; ++kk) {
                const double hik = kk == jj ? c.h[ii] : c.R[kk * (kk - 1) / 2 + ii - 1];
                const double t = hik * c.alp[kk];
                sum = sum + t;
            }
            const double hii = ii == jj ? betta : c.R[ii * (ii - 1) / 2 + ii - 1];
            const double inv = 1.0 / hii;
            c.alp[ii] = inv * (c.gam[ii] - sum);
        }
        if (blockIdx.x == 0) {
            for (int ii = 1; ii <= jj; ++ii) st->R[ii * kM1 + jj] = c.h[ii];
            st->cs[jj] = cs;
            st->sn[jj] = sn;
            st->gin[jj + 1] = gnext;
            st->gam[jj] = c.gam[jj];
            st->ncols = st->ncols + 1;
            if (conv) st->halt = jj;
        }
    }
    __syncthreads();
}

// column_done for the first columns (JJ <= kShort): the algebra in registers,
// in every thread, its operands loaded side by side with the partials.  In
// one thread over LDS each operand waited for the one before it, about 6 us
// of a launch (GMRES(3), 48^3: the last column's kernel 10.1 -> 5.5 us, with
// the loads ahead of it in k_last_small).
constexpr int kShort = 4;
template <int JJ>
__device__ __forceinline__ void column_short(int m, double folded, GmState* st, Column& c, double* red)
{
    double h[JJ + 2], cs[JJ + 1], sn[JJ + 1], gam[JJ + 1], alp[JJ + 1], R[JJ + 1][JJ + 1];
#pragma unroll
    for (int i = 1; i <= JJ; ++i) h[i] = st->H[i * kM1 + JJ];
#pragma unroll
    for (int i = 1; i < JJ; ++i) {
        cs[i] = st->cs[i];
        sn[i] = st->sn[i];
        gam[i] = st->gam[i];
#pragma unroll
        for (int k = i; k < JJ; ++k) R[i][k] = st->R[i * kM1 + k];
    }
    gam[JJ] = st->gin[JJ];
    const double eps = st->eps;
    const double s = sum256(folded, red);
    h[JJ + 1] = sqrt(s);
#pragma unroll
    for (int i = 1; i < JJ; ++i) {  // both statements assign h(ii,jj) (:722-727)
        double a = h[i] * cs[i];
        double d = h[i + 1] * sn[i];
        h[i] = a + d;
        a = -h[i] * sn[i];
        d = h[i + 1] * cs[i];
        h[i] = a + d;
    }
    const double a = h[JJ] * h[JJ];
    const double d = h[JJ + 1] * h[JJ + 1];
    const double betta = sqrt(a + d);
    const double sj = h[JJ + 1] / betta, cj = h[JJ] / betta;
    const double gnext = -sj * gam[JJ];
    gam[JJ] = cj * gam[JJ];
    const bool conv = fabs(gnext) <= eps;
    const int k = conv || JJ == m ? JJ : 0;
    h[JJ] = betta;
#pragma unroll
    for (int i = 1; i <= JJ; ++i) R[i][JJ] = h[i];
    if (k) {  // uniform
#pragma unroll
        for (int i = JJ; i >= 1; --i) {
            double sum = 0.0;
#pragma unroll
            for (int kk = i + 1; kk <= JJ; ++kk) {
                const double t = R[i][kk] * alp[kk];
                sum = sum + t;
            }
            const double inv = 1.0 / R[i][i];
            alp[i] = inv * (gam[i] - sum);
        }
    }
    if (threadIdx.x == 0) {
        c.k = k;
        c.h[JJ + 1] = h[JJ + 1];
        if (k) {
#pragma unroll
            for (int i = 1; i <= JJ; ++i) c.alp[i] = alp[i];
        }
        if (blockIdx.x == 0) {
#pragma unroll
            for (int i = 1; i <= JJ; ++i) st->R[i * kM1 + JJ] = h[i];
            st->cs[JJ] = cj;
            st->sn[JJ] = sj;
            st->gin[JJ + 1] = gnext;
            st->gam[JJ] = gam[JJ];
            st->ncols = st->ncols + 1;
            if (conv) st->halt = JJ;
        }
    }
    __syncthreads();
}

// MOST: the last column that runs in registers (those of k_col hold its loads).
template <int MOST>
__device__ __forceinline__ void column_end(int jj, int m, double folded, GmState* st, Column& c, double* red)
{
    static_assert(MOST <= kShort, "a case each");
    if (jj == 1) column_short<1>(m, folded, st, c, red);  // (jj is uniform)
    else if (MOST >= 2 && jj == 2) column_short<2>(m, folded, st, c, red);
    else if (MOST >= 3 && jj == 3) column_short<3>(m, folded, st, c, red);
    else if (MOST >= 4 && jj == 4) column_short<4>(m, folded, st, c, red);
    else column_done(jj, m, folded, st, c, red);
}

// x = x + a_1 z_1 + ... + a_k z_k, added in that order
__device__ __forceinline__ double x_updated(double xi, const Column& c, const double* __restrict__ Z,
                                            long long n, long long i)
{
    for (int j = 0; j < c.k; ++j) {
        const double t = c.alp[j + 1] * Z[(long long)j * n + i];
        xi = xi + t;
    }
    return xi;
}

// After column jj: with coefficients (the column converged or is the
// cycle's last) the x update; else v_jj+1 = w / h_jj+1,jj and z_jj+1 =
// v_jj+1 * jac.
__global__ void __launch_bounds__(kThreads)
k_next(long long n, long long chunk, int jj, int m, const double* __restrict__ part, int G,
       const double* __restrict__ w, const double* __restrict__ jac, double* __restrict__ V,
       double* __restrict__ Z, double* __restrict__ x, GmState* st)
{
    __shared__ double red[kWaves];
    __shared__ Column c;
    const double f = fold_part(part, G);
    // (a flag of this column is this launch's own)
    if (st->stop || (st->halt && st->halt != jj)) return;
    column_end<kShort>(jj, m, f, st, c, red);
    if (c.k > 0) {
        CHUNK_LOOP(i) x[i] = x_updated(x[i], c, Z, n, i);
        return;
    }
    const double h = c.h[jj + 1];
    double* v = V + (long long)jj * n;  // v_jj+1
    double* z = Z + (long long)jj * n;  // z_jj+1
    CHUNK_LOOP(i) {
        const double vi = w[i] / h;
        v[i] = vi;
        z[i] = vi * jac[i];
    }
}

// ------------------------------------------------------------------ small systems
// w / h for many w: y = 1/h and two residual corrections, which give the
// correctly rounded quotient (Markstein's theorem: the first correction is
// within an ulp, the second rounds it; checked against w / h on 2.6e8 pairs)
// away from the ends of the exponent range, where w / h itself is taken.
struct Quotient {
    double h, y;
    bool mid;
    __device__ explicit Quotient(double d) : h(d), y(1.0 / d), mid(fabs(d) > 1e-100 && fabs(d) < 1e100) {}
    __device__ __forceinline__ double operator()(double w) const
    {
        const double q0 = w * y;
        const double q1 = __builtin_fma(__builtin_fma(-h, q0, w), y, q0);
        const double q2 = __builtin_fma(__builtin_fma(-h, q1, w), y, q1);
        const double a = fabs(w);
        return mid && a > 1e-150 && a < 1e150 ? q2 : w / h;
    }
};

// z_j where a product gathers it: (r * (1/beta)) * jac for the first column
// of a cycle, (w / h) * jac for the others.
template <bool FIRST>
struct XKrylov {
    struct Raw {
        double a, j;
    };
    struct Buf {
        __amdgpu_buffer_rsrc_t a, j;
    };
    const double *a, *jac;
    double s;  // 1/beta
    Quotient q;
    __device__ __forceinline__ Raw load(int i) const { return Raw{a[i], jac[i]}; }
    __device__ __forceinline__ double v(const Raw& r) const
    {
        if constexpr (FIRST) return r.a * s;
        else return q(r.a);
    }
    __device__ __forceinline__ double value(const Raw& r) const { return v(r) * r.j; }
    __device__ __forceinline__ Buf buf(unsigned bytes) const
    {
        return Buf{tile_rsrc(a, (int)bytes), tile_rsrc(jac, (int)bytes)};
    }
    __device__ __forceinline__ Raw load(const Buf& b, int off) const
    {
        return Raw{buf_load<double>(b.a, off), buf_load<double>(b.j, off)};
    }
};

struct GmMat {
    int n;
    const int *xadj, *cols;
    const double *vals, *dvals;
    const uint32_t* mask;
    const uint8_t* mask8;
    int nd, off[32];
};

// Row sums of rows r[0..2) (r[k] >= n: not used) in CSR column order.
template <int FMT, typename X>
__device__ __forceinline__ void two_rows(const GmMat& A, const int (&r)[2], const X& x, double (&s)[2])
{
    if constexpr (FMT == CEL_FMT_DIA) {
        if (r[0] < A.n) dia_rows<double, 2, 4, true>(A.n, A.nd, A.off, A.dvals, A.mask8, A.mask, r, x, s);
    } else {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            s[k] = 0.0;
            const int lo = r[k] < A.n ? A.xadj[r[k]] : 0, hi = r[k] < A.n ? A.xadj[r[k] + 1] : 0;
            for (int j0 = lo; j0 < hi; j0 += kGather) {
                typename X::Raw xv[kGather];
                double a[kGather];
#pragma unroll
                for (int i = 0; i < kGather; ++i) {
                    const bool on = j0 + i < hi;
                    const int c = A.cols[on ? j0 + i : lo];
                    a[i] = A.vals[on ? j0 + i : lo];
                    xv[i] = x.load(c);
                }
#pragma unroll
                for (int i = 0; i < kGather; ++i) {
                    const double t = a[i] * x.value(xv[i]);
                    const double u = s[k] + t;
                    s[k] = j0 + i < hi ? u : s[k];
                }
            }
        }
    }
}

// Column j of a small system's cycle in one launch: the scalars that end the
// column before it (FIRST: the residual), v_j and z_j, w_j = A z_j and the
// partials of v_1 . w_j.  Every gather forms z_j itself from r or the last
// w and jac, so no launch stands between a norm and the product; w
// alternates between two buffers.  With coefficients after the column
// before it (it converged), the x update instead.  One block of 1,024
// threads per chunk, two rows each.
template <int FMT, bool FIRST>
__global__ void __launch_bounds__(kWide)
k_col(GmMat A, long long chunk, int j, int m, int cycle, const double* __restrict__ prev, int G,
      const double* __restrict__ src, const double* __restrict__ jac, double* __restrict__ V,
      double* __restrict__ Z, double* __restrict__ w, double* __restrict__ x,
      double* __restrict__ part, GmState* st)
{
    __shared__ double red[2 * kWaves];
    __shared__ double terms[kWideRows];
    __shared__ Column c;
    const long long n = A.n;
    double beta = 1.0;
    const double f = fold_part(prev, G);
    if (st->stop) return;
    if constexpr (FIRST) {
        beta = residual_done(cycle, f, st, red + kWaves);
        if (beta < 0.0) return;  // uniform
        if (blockIdx.x == 0 && threadIdx.x == 0) st->gin[1] = beta;
    } else {
        if (st->halt && st->halt != j - 1) return;
        column_end<2>(j - 1, m, f, st, c, red + kWaves);
        if (c.k > 0) {
            CHUNK_LOOP(i) x[i] = x_updated(x[i], c, Z, n, i);
            return;
        }
    }
    const XKrylov<FIRST> X{src, jac, 1.0 / beta, Quotient(FIRST ? 1.0 : c.h[j])};
    double* v = V + (long long)(j - 1) * n;
    double* z = Z + (long long)(j - 1) * n;
    CHUNK_BOUNDS
    int r[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const long long i = c0 + threadIdx.x + (long long)k * kWide;
        r[k] = i < c1 ? (int)i : A.n;
    }
    double s[2] = {0.0, 0.0};
    two_rows<FMT>(A, r, X, s);
#pragma unroll
    for (int k = 0; k < 2; ++k)
        if (r[k] < A.n) {
            const auto raw = X.load(r[k]);
            const double vi = X.v(raw), wi = 0.0 + s[k];
            v[r[k]] = vi;
            z[r[k]] = vi * raw.j;
            w[r[k]] = wi;
            const double p = (FIRST ? vi : V[r[k]]) * wi;
            terms[r[k] - c0] = p;
        }
    __syncthreads();
    double acc = 0.0;
    if (threadIdx.x < kBlock)
        for (int i = threadIdx.x; i < (int)(c1 - c0); i += kBlock) acc = acc + terms[i];
    const double t = sum256(acc, red);
    if (threadIdx.x == 0) part[blockIdx.x] = t;
}

// r = b - A x and the partials of r . r
template <int FMT>
__global__ void __launch_bounds__(kWide)
k_resid_small(GmMat A, long long chunk, const double* __restrict__ x, const double* __restrict__ b,
              double* __restrict__ rr, double* __restrict__ part, const GmState* __restrict__ st)
{
    __shared__ double red[kWaves];
    __shared__ double terms[kWideRows];
    if (st->stop) return;
    const long long n = A.n;
    CHUNK_BOUNDS
    int r[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const long long i = c0 + threadIdx.x + (long long)k * kWide;
        r[k] = i < c1 ? (int)i : A.n;
    }
    double s[2] = {0.0, 0.0};
    two_rows<FMT>(A, r, XPlain<double>{x}, s);
#pragma unroll
    for (int k = 0; k < 2; ++k)
        if (r[k] < A.n) {
            const double ri = b[r[k]] - (0.0 + s[k]);
            rr[r[k]] = ri;
            const double p = ri * ri;
            terms[r[k] - c0] = p;
        }
    __syncthreads();
    double acc = 0.0;
    if (threadIdx.x < kBlock)
        for (int i = threadIdx.x; i < (int)(c1 - c0); i += kBlock) acc = acc + terms[i];
    const double t = sum256(acc, red);
    if (threadIdx.x == 0) part[blockIdx.x] = t;
}

// k_next of a small system's last column: the x update, on the blocks of its
// other kernels, two rows per thread.
__global__ void __launch_bounds__(kWide)
k_last_small(long long n, long long chunk, int m, const double* __restrict__ part, int G,
             const double* __restrict__ Z, double* __restrict__ x, GmState* st)
{
    __shared__ double red[kWaves];
    __shared__ Column c;
    const double f = fold_part(part, G);
    CHUNK_BOUNDS
    int r[2];
    double xi[2], z[2][kShort];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const long long i = c0 + threadIdx.x + (long long)k * kWide;
        r[k] = i < c1 ? (int)i : (int)n;
        const int rc = r[k] < n ? r[k] : 0;
        xi[k] = x[rc];
#pragma unroll
        for (int j = 0; j < kShort; ++j) z[k][j] = Z[(long long)(j < m ? j : 0) * n + rc];
    }
    if (st->stop || (st->halt && st->halt != m)) return;
    column_end<kShort>(m, m, f, st, c, red);
#pragma unroll
    for (int k = 0; k < 2; ++k)
        if (r[k] < n) {
            double s = xi[k];
#pragma unroll
            for (int j = 0; j < kShort; ++j) {
                if (j < c.k) {
                    const double t = c.alp[j + 1] * z[k][j];
                    s = s + t;
                }
            }
            for (int j = kShort; j < c.k; ++j) {
                const double t = c.alp[j + 1] * Z[(long long)j * n + r[k]];
                s = s + t;
            }
            x[r[k]] = s;
        }
}

// DIA rows of a small system's chunk with the vector's values in LDS.  The
// gathers of 2,048 rows on one CU, and a quotient for each of them, are what
// a column's launch consists of (54 blocks at 48^3); so a block forms each
// value of its chunk once, kNear rows on either side with it, and a row
// takes the inner diagonals from there and forms the two outer ones itself:
// 3.1 values per row instead of 7.  All loads are issued before the scalars
// are there.  k_col 12.1 -> 10.7 us, the first column's 10.1 -> 8.5; a cycle
// of GMRES(3) with column_short and k_last_small 77.3 -> 67.4 us (CSR, without
// the window, 93.6 -> 87.8), 16^3 69.8 -> 62.3, 80^3 97.6 -> 96.3.  The
// Gram-Schmidt launches, 4.1 us each, are near an empty one's 3.  (512-row
// chunks would fill the chip but group the sums anew, and the reference's
// rotation answers rounding with other iteration counts.)  A rule on the
// offsets (window()): all diagonals but the first and the last within kNear
// of the main one.
constexpr int kNear = 1024;
struct Window {
    double val[kWideRows + 2 * kNear];  // [kNear + i - c0]
};
template <typename X>
struct WindowRows {
    typename X::Raw own[2], first[2], last[2], side[2];
    double a[2][kGather];
    unsigned m[2];
    int r[2], at[2];  // rows (n: none) and the rows beside the chunk

    __device__ __forceinline__ void load(const GmMat& A, long long c0, long long c1, const X& x)
    {
        const auto rx = x.buf((unsigned)A.n * 8u);
        const int far0 = A.off[0], far1 = A.off[A.nd - 1];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const long long i = c0 + threadIdx.x + (long long)k * kWide;
            r[k] = i < c1 ? (int)i : A.n;
            const int rc = r[k] < A.n ? r[k] : 0;
            own[k] = x.load(rc);
            // (an absent entry's column may lie outside [0, n): as dia_rows)
            first[k] = x.load(rx, (int)((unsigned)(rc + far0) * 8u));
            last[k] = x.load(rx, (int)((unsigned)(rc + far1) * 8u));
            m[k] = A.mask8[rc];
#pragma unroll
            for (int d = 0; d < kGather; ++d) a[k][d] = d < A.nd ? A.dvals[(long long)d * A.n + rc] : 0.0;
        }
        // kNear = kWide rows before the chunk and after it
        at[0] = (int)(c0 - kNear + threadIdx.x);
        at[1] = (int)(c1 + threadIdx.x);
#pragma unroll
        for (int k = 0; k < 2; ++k) side[k] = x.load(rx, (int)((unsigned)at[k] * 8u));
    }
    // every thread of the block; it synchronises
    __device__ __forceinline__ void stage(const GmMat& A, long long c0, const X& x, Window& w) const
    {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            if (r[k] < A.n) w.val[kNear + r[k] - c0] = x.value(own[k]);
            w.val[kNear + at[k] - c0] = x.value(side[k]);
        }
        __syncthreads();
    }
    __device__ __forceinline__ double sum(int k, const GmMat& A, long long c0, const X& x, const Window& w) const
    {
        double s = 0.0;
        const double* near = w.val + (kNear + r[k] - c0);
#pragma unroll
        for (int d = 0; d < kGather; ++d)
            if (d < A.nd) {
                const double z = d == 0 ? x.value(first[k]) : d == A.nd - 1 ? x.value(last[k]) : near[A.off[d]];
                const double t = a[k][d] * z;
                const double u = s + t;
                s = (m[k] >> d) & 1u ? u : s;
            }
        return s;
    }
};
static_assert(kNear == kWide, "one row beside the chunk per thread and side");

// k_col and k_resid_small by the window
template <bool FIRST>
__global__ void __launch_bounds__(kWide)
k_col_window(GmMat A, long long chunk, int j, int m, int cycle, const double* __restrict__ prev, int G,
             const double* __restrict__ src, const double* __restrict__ jac, double* __restrict__ V,
             double* __restrict__ Z, double* __restrict__ w, double* __restrict__ x,
             double* __restrict__ part, GmState* st)
{
    __shared__ double red[2 * kWaves];
    __shared__ double terms[kWideRows];
    __shared__ Window win;
    __shared__ Column c;
    const long long n = A.n;
    const double f = fold_part(prev, G);
    using X = XKrylov<FIRST>;
    CHUNK_BOUNDS
    WindowRows<X> rows;
    rows.load(A, c0, c1, X{src, jac, 1.0, Quotient(1.0)});
    double v1[2];
#pragma unroll
    for (int k = 0; k < 2; ++k)
        if constexpr (!FIRST) v1[k] = V[rows.r[k] < A.n ? rows.r[k] : 0];
    double beta = 1.0;
    if (st->stop) return;
    if constexpr (FIRST) {
        beta = residual_done(cycle, f, st, red + kWaves);
        if (beta < 0.0) return;  // uniform
        if (blockIdx.x == 0 && threadIdx.x == 0) st->gin[1] = beta;
    } else {
        if (st->halt && st->halt != j - 1) return;
        column_end<2>(j - 1, m, f, st, c, red + kWaves);
        if (c.k > 0) {
            for (long long i = c0 + threadIdx.x; i < c1; i += kWide) x[i] = x_updated(x[i], c, Z, n, i);
            return;
        }
    }
    const X kx{src, jac, 1.0 / beta, Quotient(FIRST ? 1.0 : c.h[j])};
    double* v = V + (long long)(j - 1) * n;
    double* z = Z + (long long)(j - 1) * n;
    rows.stage(A, c0, kx, win);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int r = rows.r[k];
        if (r < A.n) {
            const double vi = kx.v(rows.own[k]), wi = 0.0 + rows.sum(k, A, c0, kx, win);
            v[r] = vi;
            z[r] = vi * rows.own[k].j;
            w[r] = wi;
            const double p = (FIRST ? vi : v1[k]) * wi;
            terms[r - c0] = p;
        }
    }
    __syncthreads();
    double acc = 0.0;
    if (threadIdx.x < kBlock)
        for (int i = threadIdx.x; i < (int)(c1 - c0); i += kBlock) acc = acc + terms[i];
    const double t = sum256(acc, red);
    if (threadIdx.x == 0) part[blockIdx.x] = t;
}

__global__ void __launch_bounds__(kWide)
k_resid_window(GmMat A, long long chunk, const double* __restrict__ x, const double* __restrict__ b,
               double* __restrict__ rr, double* __restrict__ part, const GmState* __restrict__ st)
{
    __shared__ double red[kWaves];
    __shared__ double terms[kWideRows];
    __shared__ Window win;
    const long long n = A.n;
    CHUNK_BOUNDS
    const XPlain<double> X{x};
    WindowRows<XPlain<double>> rows;
    rows.load(A, c0, c1, X);
    double bi[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) bi[k] = b[rows.r[k] < A.n ? rows.r[k] : 0];
    if (st->stop) return;
    rows.stage(A, c0, X, win);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int r = rows.r[k];
        if (r < A.n) {
            const double ri = bi[k] - (0.0 + rows.sum(k, A, c0, X, win));
            rr[r] = ri;
            const double p = ri * ri;
            terms[r - c0] = p;
        }
    }
    __syncthreads();
    double acc = 0.0;
    if (threadIdx.x < kBlock)
        for (int i = threadIdx.x; i < (int)(c1 - c0); i += kBlock) acc = acc + terms[i];
    const double t = sum256(acc, red);
    if (threadIdx.x == 0) part[blockIdx.x] = t;
}

struct Gmres {
    const Mat& A;
    int format;
    long long n, chunk;
    int G;
    hipStream_t st;

    Gmres(const Mat& M, int fmt) : A(M), format(fmt), n(M.n), st(rt().stream)
    {
        // fixed chunks of a multiple of the workgroup size: the grouping of
        // every dot product depends on n only (2048 rows per chunk up to
        // 1024 chunks: one 8-row step per thread of the fused DIA product)
        long long g = (n + 2047) / 2048;
        G = (int)(g < 1 ? 1 : g > 1024 ? 1024 : g);
        chunk = ((n + G - 1) / G + kThreads - 1) / kThreads * kThreads;
        if (chunk < kThreads) chunk = kThreads;
    }
    // Whether a column is one launch (k_col) plus its Gram-Schmidt passes.
    // Measured per cycle of GMRES(3), 7-point cubes, k_col / separate
    // launches: 16^3 DIA 76.0 / 83.2 us, CSR 88.8 / 105; 48^3 84.8 / 92.1, 101
    // / 119; 80^3 112 / 129, 121 / 155; 100^3 183 / 175, 196 / 198; 128^3 338 /
    // 283, 420 / 328 (the second gathered array and the quotients cost more
    // than the launches).  Long rows gather too much at any size (30,011 mesh
    // rows of 11 entries 185 / 169).
    bool small() const { return format != CEL_FMT_JAD && n <= 600000 && !csr_long_rows(A); }
    bool window() const
    {
        if (format != CEL_FMT_DIA || A.dia_nd > kGather) return false;
        for (int d = 1; d + 1 < A.dia_nd; ++d)
            if (A.dia_off[d] < -kNear || A.dia_off[d] > kNear) return false;
        return true;
    }
    GmMat mat() const
    {
        GmMat M{};
        M.n = A.n;
        M.xadj = A.xadj.p;
        M.cols = A.cols.p;
        M.vals = A.vals.p;
        M.dvals = A.dia_vals.p;
        M.mask = A.dia_mask.p;
        M.mask8 = A.dia_mask8.p;
        M.nd = A.dia_nd;
        for (int d = 0; d < A.dia_nd; ++d) M.off[d] = A.dia_off[d];
        return M;
    }
    // w = A z with the partials of v1 . w (skipped once halt is set)
    int spmv_dot(const double* z, double* w, const double* v1, double* part, GmState* gs)
    {
        const int* skip = &gs->halt;
        if (format == CEL_FMT_DIA)
            return launch_dia_spmv_fused(A, kFuseDot, chunk, G, z, w, v1, part, skip);
        if (format == CEL_FMT_CSR)
            return launch_csr_spmv_fused(A, kFuseDot, chunk, G, z, w, v1, part, skip);
        CEL_TRY(launch_jad_spmv(A, z, w, 0, skip));
        k_dot<<<G, kThreads, 0, st>>>(n, chunk, v1, w, part, gs);
        return CEL_OK;
    }
    // r = b - A x with the partials of r . r (skipped once stop is set)
    int spmv_resid(const double* x, double* r, const double* b, double* part, GmState* gs)
    {
        const int* skip = &gs->stop;
        if (format == CEL_FMT_DIA)
            return launch_dia_spmv_fused(A, kFuseResid, chunk, G, x, r, b, part, skip);
        if (format == CEL_FMT_CSR)
            return launch_csr_spmv_fused(A, kFuseResid, chunk, G, x, r, b, part, skip);
        CEL_TRY(launch_jad_spmv(A, x, r, 0, skip));
        k_resid<<<G, kThreads, 0, st>>>(n, chunk, b, r, part, gs);
        return CEL_OK;
    }
};

}  // namespace

int gmres_solve(Mat& A, const double* b_in, double* x_out, const cel_gmres_params& prm,
                cel_pcg_stats& stats)
{
    const int m = prm.restart;
    if (m < 1 || m > kMaxRestart) return fail(CEL_ERR_ARG, "restart must be 1..32");
    if (prm.iter_max < 0) return fail(CEL_ERR_ARG, "iter_max must be >= 0");
    if (!A.has_jac) return fail(CEL_ERR_STATE, "cel_gpu_mat_set_jacobi has not been called");
    if (prm.format == CEL_FMT_JAD && A.jad_mode < 0)
        return fail(CEL_ERR_STATE, "JAD requested before cel_gpu_mat_to_jad");
    if (prm.format == CEL_FMT_JAD && A.jad_ndef < A.jad_mmax)
        return fail(CEL_ERR_REF_UNDEFINED, "the JAD form of this matrix is undefined in the reference");
    if (prm.format == CEL_FMT_DIA && A.dia_nd == 0)
        return fail(CEL_ERR_STATE, "DIA requested before cel_gpu_mat_to_dia");
    if (A.n != A.ncols) return fail(CEL_ERR_ARG, "GMRES needs a square local block");
    const long long n = A.n;
    stats = cel_pcg_stats{};
    if (n == 0) return CEL_OK;
    Gmres S(A, prm.format);
    hipStream_t st = S.st;
    const int G = S.G;
    const long long ck = S.chunk;
    DevBuf<double> xb, bb, r, w, V, Z, partA, partB;
    DevBuf<GmState> state;
    CEL_TRY(r.alloc(n));
    CEL_TRY(w.alloc(n));
    CEL_TRY(V.alloc((size_t)n * m));
    CEL_TRY(Z.alloc((size_t)n * m));
    CEL_TRY(partA.alloc(G));
    CEL_TRY(partB.alloc(G));
    CEL_TRY(state.alloc(1));
    const double* b = b_in;
    double* x = x_out;
    if (prm.memspace == CEL_MEM_HOST) {
        CEL_TRY(bb.alloc(n));
        CEL_TRY(xb.alloc(n));
        CEL_HIP(hipMemcpyAsync(bb.p, b_in, sizeof(double) * n, hipMemcpyHostToDevice, st));
        if (prm.x0_mode == CEL_X0_USER)
            CEL_HIP(hipMemcpyAsync(xb.p, x_out, sizeof(double) * n, hipMemcpyHostToDevice, st));
        b = bb.p;
        x = xb.p;
    }
    GmState* gs = state.p;
    const int* stop = &gs->stop;
    auto vv = [&](int k) { return V.p + (size_t)(k - 1) * n; };  // v_k, 1-based
    auto zz = [&](int k) { return Z.p + (size_t)(k - 1) * n; };

    const bool small = S.small();
    DevBuf<double> w2;
    if (small) CEL_TRY(w2.alloc(n));
    const GmMat GM = S.mat();
    const bool dia = prm.format == CEL_FMT_DIA, win = S.window();
    A.path = SolvePath{"gmres", small, false, small && win};
    // the same on a small system: k_col in place of k_scale_jac / k_next and
    // the product
    auto enqueue_small = [&]() -> int {
        auto resid = [&]() {
            if (win) k_resid_window<<<G, kWide, 0, st>>>(GM, ck, x, b, r.p, partA.p, gs);
            else if (dia) k_resid_small<CEL_FMT_DIA><<<G, kWide, 0, st>>>(GM, ck, x, b, r.p, partA.p, gs);
            else k_resid_small<CEL_FMT_CSR><<<G, kWide, 0, st>>>(GM, ck, x, b, r.p, partA.p, gs);
        };
        auto col = [&](auto kernel, int j, int cycle, const double* prev, const double* src, double* out, double* part) {
            kernel<<<G, kWide, 0, st>>>(GM, ck, j, m, cycle, prev, G, src, A.jac.p, V.p, Z.p, out, x, part, gs);
        };
        resid();
        for (int c = 0; c <= m; ++c) {
            double *cur = partA.p, *nxt = partB.p, *wi = w.p, *wo = w2.p;
            for (int jj = 1; jj <= m; ++jj) {
                if (jj == 1) col(win ? k_col_window<true> : dia ? k_col<CEL_FMT_DIA, true> : k_col<CEL_FMT_CSR, true>, jj, c > 0, cur, r.p, wo, nxt);
                else col(win ? k_col_window<false> : dia ? k_col<CEL_FMT_DIA, false> : k_col<CEL_FMT_CSR, false>, jj, 0, cur, wi, wo, nxt);
                std::swap(cur, nxt);
                std::swap(wi, wo);
                for (int ii = 1; ii <= jj; ++ii) {
                    const double* next = ii < jj ? vv(ii + 1) : nullptr;
                    k_mgs<kWide><<<G, kWide, 0, st>>>(n, ck, ii, jj, cur, G, vv(ii), wi, next, nxt, gs);
                    std::swap(cur, nxt);
                }
            }
            k_last_small<<<G, kWide, 0, st>>>(n, ck, m, cur, G, Z.p, x, gs);
            resid();
        }
        k_cycle_end<<<1, kThreads, 0, st>>>(partA.p, G, gs);
        CEL_HIP(hipGetLastError());
        return CEL_OK;
    };
    // one outer iteration: r = b - A x, then up to m+1 cycles
    auto enqueue_outer = [&]() -> int {
        if (small) return enqueue_small();
        CEL_TRY(S.spmv_resid(x, r.p, b, partA.p, gs));
        for (int c = 0; c <= m; ++c) {
            k_scale_jac<<<G, kThreads, 0, st>>>(n, ck, c > 0, partA.p, G, r.p, A.jac.p, vv(1), zz(1), gs);
            for (int jj = 1; jj <= m; ++jj) {
                double* cur = partB.p;
                double* nxt = partA.p;
                CEL_TRY(S.spmv_dot(zz(jj), w.p, vv(1), cur, gs));
                for (int ii = 1; ii <= jj; ++ii) {
                    const double* next = ii < jj ? vv(ii + 1) : nullptr;
                    k_mgs<kThreads><<<G, kThreads, 0, st>>>(n, ck, ii, jj, cur, G, vv(ii), w.p, next, nxt, gs);
                    std::swap(cur, nxt);
                }
                k_next<<<G, kThreads, 0, st>>>(n, ck, jj, m, cur, G, w.p, A.jac.p, V.p, Z.p, x, gs);
            }
            CEL_TRY(S.spmv_resid(x, r.p, b, partA.p, gs));
        }
        k_cycle_end<<<1, kThreads, 0, st>>>(partA.p, G, gs);
        CEL_HIP(hipGetLastError());
        return CEL_OK;
    };

    StreamScope R(st);
    hipEvent_t e0, e1, cev[2];
    CEL_TRY(R.event(e0));
    CEL_TRY(R.event(e1));
    CEL_TRY(R.event(cev[0], hipEventDisableTiming));
    CEL_TRY(R.event(cev[1], hipEventDisableTiming));
    int* hstop = nullptr;
    CEL_TRY(R.host_alloc(hstop, 2));
    hstop[0] = hstop[1] = 0;

    CEL_HIP(hipEventRecord(e0, st));
    k_state_init<<<1, kThreads, 0, st>>>(gs, prm.eps);
    if (prm.x0_mode == CEL_X0_ONE || prm.x0_mode == CEL_X0_ZERO)
        k_fill<<<G, kThreads, 0, st>>>(n, ck, x, prm.x0_mode == CEL_X0_ONE ? 1.0 : 0.0);
    CEL_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
    {
        const int rc = enqueue_outer();
        const hipError_t ec = hipStreamEndCapture(st, &R.graph);
        if (rc < 0) return rc;
        CEL_HIP(ec);
    }
    CEL_HIP(hipGraphInstantiate(&R.exec, R.graph, nullptr, nullptr, 0));
    // outer iterations: the reference runs them while iter <= iter_max
    // (iter counted from 1), so at most iter_max + 1
    const long long budget = (long long)prm.iter_max + 1;
    for (long long k = 0; k < budget; ++k) {
        CEL_HIP(hipGraphLaunch(R.exec, st));
        CEL_HIP(hipMemcpyAsync(&hstop[k & 1], stop, sizeof(int), hipMemcpyDeviceToHost, st));
        CEL_HIP(hipEventRecord(cev[k & 1], st));
        if (k > 0) {
            CEL_HIP(hipEventSynchronize(cev[(k - 1) & 1]));
            if (hstop[(k - 1) & 1]) break;
        }
    }
    CEL_HIP(hipEventRecord(e1, st));
    if (prm.memspace == CEL_MEM_HOST)
        CEL_HIP(hipMemcpyAsync(x_out, x, sizeof(double) * n, hipMemcpyDeviceToHost, st));
    CEL_HIP(hipStreamSynchronize(st));
    GmState out{};
    CEL_HIP(hipMemcpy(&out, gs, sizeof(GmState), hipMemcpyDeviceToHost));
    float ms = 0.f;
    CEL_HIP(hipEventElapsedTime(&ms, e0, e1));

    stats.iters = out.iter;
    stats.outer_iters = out.cycles;
    stats.norm0 = out.norm0;
    stats.final_norm = out.residuum;
    stats.eps_abs = prm.eps;
    stats.solve_ms = ms;
    // products run: one per outer residual, per cycle residual, per column
    stats.spmv_launches = out.iter + out.cycles + out.ncols;
    if (out.status != 0) {
        stats.status = out.status;
        return fail(out.status, "the residual is not finite");
    }
    stats.status = out.halt ? CEL_OK : CEL_NOT_CONVERGED;
    return stats.status;
}

}  // namespace cel

using namespace cel;

extern "C" void cel_gpu_gmres_params_default(cel_gmres_params* p)
{
    if (!p) return;
    // the element solver's settings (src/felmsolver/cel_elmsolver_module.f90:140-151)
    p->eps = 0.1e-07;
    p->iter_max = 5000;
    p->restart = 4 - 1;
    p->x0_mode = CEL_X0_ONE;
    p->memspace = CEL_MEM_HOST;
    p->format = CEL_FMT_CSR;
}

extern "C" int cel_gpu_gmres_solve(cel_gpu_mat* A, const double* b, double* x,
                                   const cel_gmres_params* params, cel_pcg_stats* stats)
{
    CEL_TRY(ensure_init());
    if (!A || !b || !x) return fail(CEL_ERR_ARG, "null argument to cel_gpu_gmres_solve");
    cel_gmres_params p;
    if (params) p = *params;
    else cel_gpu_gmres_params_default(&p);
    if ((p.memspace != CEL_MEM_HOST && p.memspace != CEL_MEM_DEVICE) ||
        (p.format != CEL_FMT_CSR && p.format != CEL_FMT_JAD && p.format != CEL_FMT_DIA) ||
        (p.x0_mode != CEL_X0_ONE && p.x0_mode != CEL_X0_ZERO && p.x0_mode != CEL_X0_USER) ||
        !(p.eps >= 0.0))
        return fail(CEL_ERR_ARG, "bad cel_gmres_params");
    cel_pcg_stats s{};
    int rc = gmres_solve(A->m, b, x, p, s);
    if (stats) *stats = s;
    return rc;
}

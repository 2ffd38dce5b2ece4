// dia.hip -- DIA form of a CSR block and its SpMV (no reference counterpart).
//
// A block whose entries lie on a few diagonals (structured-grid stencils)
// is stored per diagonal: vals[d * n + i] is the entry of row i in column
// i + off[d] (0 where absent), bit d of mask[i] tells whether it exists.
// Offsets ascend, so a row sum over d visits the row's entries in the CSR
// column order; absent entries are skipped (not added as zeros: 0 * x is
// not +0 for every x), so the product is bit-identical to the CSR one,
// without column indices and with x read contiguously per diagonal.  The
// mask is one byte per row when there are at most 8 diagonals.
#include <algorithm>
#include <vector>

#include "cel_internal.hpp"
#include "spmv_device.hpp"

namespace cel {

constexpr int kMaxDiag = 32;

namespace {

int grid_of(long long n)
{
    long long g = (n + kBlock - 1) / kBlock;
    long long cap = (long long)rt().num_cus * 16;
    return (int)(g < 1 ? 1 : g > cap ? cap : g);
}

// The distinct offsets col - row of a block, at most kMaxDiag of them.
struct OffsetSet {
    int slot[2 * kMaxDiag];  // open addressing; kNoOffset: free
    int count;
    int over;                // more than `most` offsets
    int bad;                 // a row whose columns do not strictly ascend
};
constexpr int kNoOffset = -2147483647 - 1;  // no column lies 2^31 left of its row
constexpr int kRowAhead = 8;                // columns a thread loads at once

__device__ __forceinline__ int offset_hash(int o)
{
    return (int)(((unsigned)o * 2654435761u) >> 26);  // 0..63
}

// true: o is in the set (put there if it was missing); *added: it was missing
__device__ __forceinline__ bool offset_put(int* slot, int o, bool& added)
{
    added = false;
    int at = offset_hash(o);
    for (int k = 0; k < 2 * kMaxDiag; ++k, at = (at + 1) & (2 * kMaxDiag - 1)) {
        int v = slot[at];
        if (v == kNoOffset) {
            v = atomicCAS(&slot[at], kNoOffset, o);
            if (v == kNoOffset) {
                added = true;
                return true;
            }
        }
        if (v == o) return true;
    }
    return false;
}

__global__ void __launch_bounds__(kBlock) k_offset_clear(OffsetSet* sets)
{
    OffsetSet* g = sets + blockIdx.x;
    if (threadIdx.x < 2 * kMaxDiag) g->slot[threadIdx.x] = kNoOffset;
    if (threadIdx.x == 0) g->count = g->over = g->bad = 0;
}

// One thread per row; a block keeps the offsets it has met in LDS and adds
// them to the set of the grid at its end.  Bound by reading the columns
// once; a block that meets too many offsets, or sees that another one did,
// stops.  (Sorting the offsets of every entry and encoding the runs took
// 0.95 ms of kernels on a 128^3 block and four arrays of nnz integers.)
__global__ void __launch_bounds__(kBlock)
k_offset_scan(int n, const int* __restrict__ xadj, const int* __restrict__ cols, int most,
              OffsetSet* g)
{
    __shared__ int slot[2 * kMaxDiag];
    __shared__ int count, over, bad, stop;
    if (threadIdx.x < 2 * kMaxDiag) slot[threadIdx.x] = kNoOffset;
    if (threadIdx.x == 0) count = over = bad = 0;
    __syncthreads();
    for (long long i0 = (long long)blockIdx.x * kBlock; i0 < n; i0 += (long long)gridDim.x * kBlock) {
        const long long i = i0 + threadIdx.x;
        const int lo = i < n ? xadj[i] : 0, hi = i < n ? xadj[i + 1] : 0;
        int prev = -1;
        for (int j0 = lo; j0 < hi; j0 += kRowAhead) {
            int c[kRowAhead];
#pragma unroll
            for (int k = 0; k < kRowAhead; ++k) c[k] = cols[j0 + k < hi ? j0 + k : lo];
#pragma unroll
            for (int k = 0; k < kRowAhead; ++k) {
                if (j0 + k >= hi) break;
                if (c[k] <= prev) bad = 1;
                prev = c[k];
                bool added;
                if (!offset_put(slot, c[k] - (int)i, added) || (added && atomicAdd(&count, 1) >= most)) over = 1;
            }
            if (over) break;
        }
        __syncthreads();
        if (threadIdx.x == 0) stop = over | *(volatile int*)&g->over;
        __syncthreads();
        if (stop) break;  // uniform; this block's set is incomplete, but the result is `over`
    }
    __syncthreads();
    if (threadIdx.x < 2 * kMaxDiag && slot[threadIdx.x] != kNoOffset) {
        bool added;
        if (!offset_put(g->slot, slot[threadIdx.x], added) || (added && atomicAdd(&g->count, 1) >= most))
            atomicOr(&g->over, 1);
    }
    if (threadIdx.x == 0) {
        if (over) atomicOr(&g->over, 1);
        if (bad) atomicOr(&g->bad, 1);
    }
}

// For the refusal of a block with too many diagonals: which offsets it has, as
// bits (offset + n - 1), and whether a row's columns do not strictly ascend
// (k_offset_scan stops before it has seen every row).
__global__ void __launch_bounds__(kBlock)
k_offset_bits(int n, const int* __restrict__ xadj, const int* __restrict__ cols, unsigned* bits, int* bad)
{
    for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long long)gridDim.x * kBlock) {
        int prev = -1;
        for (int j = xadj[i]; j < xadj[i + 1]; ++j) {
            const int c = cols[j];
            if (c <= prev) *(volatile int*)bad = 1;
            prev = c;
            const long long at = c - i + n - 1;
            if (at < 0 || at >= 2LL * n - 1) continue;
            const unsigned bit = 1u << (at & 31);
            if (!(*(volatile unsigned*)&bits[at >> 5] & bit)) atomicOr(&bits[at >> 5], bit);
        }
    }
}
__global__ void __launch_bounds__(kBlock) k_count_bits(long long words, const unsigned* __restrict__ bits, int* sum)
{
    int c = 0;
    for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < words; i += (long long)gridDim.x * kBlock)
        c += __popc(bits[i]);
    if (c) atomicAdd(sum, c);
}

struct Offsets {
    int nd;
    int off[kMaxDiag];
};

// SHORT (at most 8 diagonals, so rows of at most 8 entries): a row's entries
// are loaded at once and every slot is written, absent ones with 0 (one
// entry after another, over zeroed slots: 128^3 block 155 us and a memset,
// 85 us so).
template <typename VT, bool SHORT>
__global__ void __launch_bounds__(kBlock)
k_dia_fill(int n, const int* __restrict__ xadj, const int* __restrict__ cols,
           const double* __restrict__ vals, Offsets O, VT* __restrict__ dv,
           uint32_t* __restrict__ mask, uint8_t* __restrict__ mask8)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x) {
        unsigned m = 0;
        const int lo = xadj[i], len = xadj[i + 1] - lo;
        if constexpr (SHORT) {
            int c[8];
            double a[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                c[k] = k < len ? cols[lo + k] - (int)i : 0;
                a[k] = k < len ? vals[lo + k] : 0.0;
            }
#pragma unroll
            for (int d = 0; d < 8; ++d)
                if (d < O.nd) {
                    double v = 0.0;
#pragma unroll
                    for (int k = 0; k < 8; ++k)
                        if (k < len && c[k] == O.off[d]) {
                            v = a[k];
                            m |= 1u << d;
                        }
                    dv[(size_t)d * n + i] = (VT)v;
                }
        } else {
            for (int j = lo; j < lo + len; ++j) {
                const int o = cols[j] - (int)i;
                int d = 0;
                while (d < O.nd - 1 && O.off[d] != o) ++d;
                dv[(size_t)d * n + i] = (VT)vals[j];
                m |= 1u << d;
            }
        }
        if (mask8) mask8[i] = (uint8_t)m;
        else mask[i] = m;
    }
}

Offsets offsets_of(const Mat& A)
{
    Offsets O{};
    O.nd = A.dia_nd;
    for (int d = 0; d < A.dia_nd; ++d) O.off[d] = A.dia_off[d];
    return O;
}

// y = A x (accumulate: y += A x); for every group T of R 256-row tiles it
// owns (T = block, block + G, ...), each thread sums rows T*R*256 + tid +
// 256k, k < R, loading GD diagonals of all R rows at a time.
template <typename VT, int R, int GD>
__global__ void __launch_bounds__(kBlock)
k_dia_spmv(int n, Offsets O, const VT* __restrict__ dv, const uint32_t* __restrict__ mask,
           const uint8_t* __restrict__ mask8, const VT* __restrict__ x, VT* __restrict__ y,
           int accumulate, const int* __restrict__ skip)
{
    if (skip && *skip) return;
    const long long groups = ((long long)n + R * kBlock - 1) / (R * kBlock);
    for (long long T = blockIdx.x; T < groups; T += gridDim.x) {
        int r[R];
#pragma unroll
        for (int k = 0; k < R; ++k) r[k] = (int)(T * R * kBlock) + threadIdx.x + k * kBlock;
        if (r[0] >= n) continue;
        VT s[R];
        dia_rows<VT, R, GD>(n, O.nd, O.off, dv, mask8, mask, r, XPlain<VT>{x}, s);
#pragma unroll
        for (int k = 0; k < R; ++k)
            if (r[k] < n) y[r[k]] = accumulate ? y[r[k]] + s[k] : s[k];
    }
}

// Launch shapes of the plain product, measured on the 256^3 7-point block
// (20 back-to-back launches): FP32 4 rows per thread at 2 blocks per CU
// (100 us against 106-113 us for 2 rows per thread at 2-8 blocks per CU);
// FP64 8 rows per thread, 4 diagonals per load group, at 8 blocks per CU
// (225 us against 231 us).
template <typename VT>
struct DiaShape;
template <>
struct DiaShape<float> {
    static constexpr int R = 4, GD = 8, per_cu = 2;
};
template <>
struct DiaShape<double> {
    static constexpr int R = 8, GD = 4, per_cu = 8;
};

template <typename VT>
int launch_dia(const Mat& A, const VT* vals, const VT* x, VT* y, int accumulate, const int* skip)
{
    using S = DiaShape<VT>;
    const long long groups = ((long long)A.n + S::R * kBlock - 1) / (S::R * kBlock);
    const int G = (int)std::min<long long>(groups, (long long)rt().num_cus * S::per_cu);
    hipLaunchKernelGGL((k_dia_spmv<VT, S::R, S::GD>), dim3(G), dim3(kBlock), 0, rt().stream, A.n,
                       offsets_of(A), vals, A.dia_mask.p, A.dia_mask8.p, x, y, accumulate, skip);
    CEL_HIP(hipGetLastError());
    return CEL_OK;
}

// FP64 product fused with the next dot product (kFuseDot / kFuseResid,
// cel_internal.hpp): block b covers the rows of its chunk [b*chunk,
// b*chunk + chunk) in steps of R*256 rows, R rows 256 apart per thread (the
// plain FP64 shape), so each thread meets its rows in ascending order.
template <int FUSE>
__global__ void __launch_bounds__(kBlock)
k_dia_spmv_fused(int n, long long chunk, Offsets O, const double* __restrict__ dv,
                 const uint32_t* __restrict__ mask, const uint8_t* __restrict__ mask8,
                 const double* __restrict__ x, double* __restrict__ y,
                 const double* __restrict__ aux, double* __restrict__ part,
                 const int* __restrict__ skip)
{
    if (skip && *skip) return;  // uniform across the grid
    __shared__ double red[kWaves];
    constexpr int R = DiaShape<double>::R, GD = DiaShape<double>::GD;
    const long long c0 = (long long)blockIdx.x * chunk;
    const long long c1 = c0 + chunk < n ? c0 + chunk : n;
    double acc = 0.0;
    for (long long s0 = c0; s0 < c1; s0 += (long long)R * kBlock) {
        int r[R];
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const long long rk = s0 + threadIdx.x + (long long)k * kBlock;
            r[k] = rk < c1 ? (int)rk : n;  // rows past the chunk are not used
        }
        if (r[0] >= n) continue;  // no barrier in this loop
        double s[R];
        dia_rows<double, R, GD>(n, O.nd, O.off, dv, mask8, mask, r, XPlain<double>{x}, s);
#pragma unroll
        for (int k = 0; k < R; ++k)
            if (r[k] < n) acc = acc + fuse_row<FUSE>(s[k], r[k], aux, y);
    }
    const double bs = block_sum(acc, red);
    if (threadIdx.x == 0) part[blockIdx.x] = bs;
}


}  // namespace

int launch_dia_spmv(const Mat& A, const double* x, double* y, int accumulate, const int* skip)
{
    if (A.n == 0) return CEL_OK;
    return launch_dia<double>(A, A.dia_vals.p, x, y, accumulate, skip);
}

int launch_dia_spmv_fused(const Mat& A, int fuse, long long chunk, int G, const double* x,
                          double* y, const double* aux, double* part, const int* skip)
{
    if (A.n == 0 || A.dia_nd == 0 || A.n != A.ncols)
        return fail(CEL_ERR_ARG, "fused product: a square block with a DIA form");
    if (chunk <= 0 || chunk % kBlock != 0 || (long long)G * chunk < A.n)
        return fail(CEL_ERR_ARG, "fused product: chunks must be whole tiles covering every row");
    if (fuse == kFuseDot)
        hipLaunchKernelGGL(k_dia_spmv_fused<kFuseDot>, dim3(G), dim3(kBlock), 0, rt().stream, A.n,
                           chunk, offsets_of(A), A.dia_vals.p, A.dia_mask.p, A.dia_mask8.p, x, y,
                           aux, part, skip);
    else if (fuse == kFuseResid)
        hipLaunchKernelGGL(k_dia_spmv_fused<kFuseResid>, dim3(G), dim3(kBlock), 0, rt().stream, A.n,
                           chunk, offsets_of(A), A.dia_vals.p, A.dia_mask.p, A.dia_mask8.p, x, y,
                           aux, part, skip);
    else
        return fail(CEL_ERR_ARG, "fused product: unknown epilogue");
    CEL_HIP(hipGetLastError());
    return CEL_OK;
}

int dia_offsets_all(const std::vector<Mat*>& mats, int most, std::vector<DiagonalSet>& out)
{
    const size_t k = mats.size();
    out.assign(k, DiagonalSet{});
    if (k == 0) return CEL_OK;
    hipStream_t st = rt().stream;
    DevBuf<OffsetSet> g;
    CEL_TRY(g.alloc(k));
    hipLaunchKernelGGL(k_offset_clear, dim3((unsigned)k), dim3(kBlock), 0, st, g.p);
    for (size_t q = 0; q < k; ++q)
        hipLaunchKernelGGL(k_offset_scan, dim3(grid_of(mats[q]->n)), dim3(kBlock), 0, st, mats[q]->n, mats[q]->xadj.p,
                           mats[q]->cols.p, most, g.p + q);
    CEL_HIP(hipGetLastError());
    std::vector<OffsetSet> h(k);
    CEL_HIP(hipMemcpyAsync(h.data(), g.p, sizeof(OffsetSet) * k, hipMemcpyDeviceToHost, st));
    CEL_HIP(hipStreamSynchronize(st));
    for (size_t q = 0; q < k; ++q) {
        DiagonalSet& d = out[q];
        d.ascending = !h[q].bad;
        d.nd = most + 1;
        if (h[q].over || h[q].count > most) continue;
        d.nd = 0;
        for (int v : h[q].slot)
            if (v != kNoOffset) d.off[d.nd++] = v;
        std::sort(d.off, d.off + d.nd);
    }
    return CEL_OK;
}

int dia_offsets(const Mat& A, int most, int* nd, int* off, bool* ascending)
{
    std::vector<DiagonalSet> d;
    CEL_TRY(dia_offsets_all({const_cast<Mat*>(&A)}, most, d));
    *ascending = d[0].ascending;
    *nd = d[0].nd;
    if (d[0].nd <= most) std::copy(d[0].off, d[0].off + d[0].nd, off);
    return CEL_OK;
}

// The number of distinct offsets of a block, and whether every row's columns
// strictly ascend.
static int offset_count(const Mat& A, int* nd, bool* ascending)
{
    hipStream_t st = rt().stream;
    const long long words = (2LL * A.n + 30) / 32;
    DevBuf<unsigned> bits;
    DevBuf<int> out;
    CEL_TRY(bits.alloc((size_t)words));
    CEL_TRY(out.alloc(2));
    CEL_HIP(hipMemsetAsync(bits.p, 0, sizeof(unsigned) * (size_t)words, st));
    CEL_HIP(hipMemsetAsync(out.p, 0, sizeof(int) * 2, st));
    hipLaunchKernelGGL(k_offset_bits, dim3(grid_of(A.n)), dim3(kBlock), 0, st, A.n, A.xadj.p, A.cols.p, bits.p, out.p);
    hipLaunchKernelGGL(k_count_bits, dim3(grid_of(words)), dim3(kBlock), 0, st, words, bits.p, out.p + 1);
    CEL_HIP(hipGetLastError());
    int h[2];
    CEL_HIP(hipMemcpyAsync(h, out.p, sizeof(h), hipMemcpyDeviceToHost, st));
    CEL_HIP(hipStreamSynchronize(st));
    *ascending = !h[0];
    *nd = h[1];
    return CEL_OK;
}

int dia_fill(const Mat& A, int nd, const int* off, double* v64, float* v32, uint8_t* mask8)
{
    Offsets O{};
    O.nd = nd;
    for (int d = 0; d < nd; ++d) O.off[d] = off[d];
    if (v64)
        hipLaunchKernelGGL((k_dia_fill<double, true>), dim3(grid_of(A.n)), dim3(kBlock), 0, rt().stream, A.n, A.xadj.p,
                           A.cols.p, A.vals.p, O, v64, (uint32_t*)nullptr, mask8);
    else
        hipLaunchKernelGGL((k_dia_fill<float, true>), dim3(grid_of(A.n)), dim3(kBlock), 0, rt().stream, A.n, A.xadj.p,
                           A.cols.p, A.vals.p, O, v32, (uint32_t*)nullptr, mask8);
    CEL_HIP(hipGetLastError());
    return CEL_OK;
}

int dia_prepare_f32(Mat& A)
{
    if (A.dia_vals32.p || A.dia_nd == 0) return CEL_OK;
    const size_t cnt = (size_t)A.dia_nd * (size_t)A.n;
    CEL_TRY(A.dia_vals32.alloc(cnt > 0 ? cnt : 1));
    return launch_to_f32(A.dia_vals.p, A.dia_vals32.p, cnt);
}

int launch_dia_spmv_f32(Mat& A, const float* x, float* y, int accumulate)
{
    if (A.n == 0) return CEL_OK;
    CEL_TRY(dia_prepare_f32(A));
    return launch_dia<float>(A, A.dia_vals32.p, x, y, accumulate, nullptr);
}

}  // namespace cel

using namespace cel;

extern "C" int cel_gpu_mat_to_dia(cel_gpu_mat* A)
{
    CEL_TRY(ensure_init());
    if (!A) return fail(CEL_ERR_ARG, "null matrix");
    Mat& M = A->m;
    if (M.dia_nd > 0) return CEL_OK;
    if (M.n == 0 || M.nnz == 0) return fail(CEL_ERR_BAD_MATRIX, "an empty block has no DIA form");
    // the DIA row sums read x through a resource of n entries (the row
    // count), so a column index must also be a row index
    if (M.ncols != M.n) return fail(CEL_ERR_BAD_MATRIX, "a non-square block has no DIA form");
    // the DIA kernels address a diagonal with 32-bit byte offsets
    if ((long long)M.n * (long long)sizeof(double) >= (1LL << 31))
        return fail(CEL_ERR_BAD_MATRIX, "more than 2^28 rows: no DIA form");
    hipStream_t st = rt().stream;
    const long long nnz = M.nnz;
    int nd = 0, hoff[kMaxDiag] = {};
    bool ascending = false;
    CEL_TRY(dia_offsets(M, kMaxDiag, &nd, hoff, &ascending));
    if (nd > kMaxDiag) CEL_TRY(offset_count(M, &nd, &ascending));
    if (!ascending) return fail(CEL_ERR_BAD_MATRIX, "columns not strictly ascending in every row: no DIA form");
    if (nd > kMaxDiag)
        return fail(CEL_ERR_BAD_MATRIX, std::to_string(nd) + " diagonals: more than the DIA form holds (32)");
    if ((long long)nd * M.n > 2 * nnz)
        return fail(CEL_ERR_BAD_MATRIX, "DIA would store more than twice nnz slots");
    const size_t cnt = (size_t)nd * (size_t)M.n;
    CEL_TRY(M.dia_vals.alloc(cnt));
    // exactly one mask array: the kernels read both (the other reads 0)
    if (nd <= 8) {
        M.dia_mask.release();
        CEL_TRY(M.dia_mask8.alloc(M.n));
    } else {
        M.dia_mask8.release();
        CEL_TRY(M.dia_mask.alloc(M.n));
    }
    if (nd > 8) CEL_HIP(hipMemsetAsync(M.dia_vals.p, 0, sizeof(double) * cnt, st));
    Offsets O{};
    O.nd = nd;
    for (int d = 0; d < nd; ++d) O.off[d] = hoff[d];
    hipLaunchKernelGGL((nd <= 8 ? k_dia_fill<double, true> : k_dia_fill<double, false>), dim3(grid_of(M.n)),
                       dim3(kBlock), 0, st, M.n, M.xadj.p, M.cols.p, M.vals.p, O, M.dia_vals.p,
                       nd <= 8 ? nullptr : M.dia_mask.p, nd <= 8 ? M.dia_mask8.p : nullptr);
    CEL_HIP(hipGetLastError());
    CEL_HIP(hipStreamSynchronize(st));
    M.dia_nd = nd;
    for (int d = 0; d < nd; ++d) M.dia_off[d] = hoff[d];
    M.dia_vals32.release();
    return CEL_OK;
}

extern "C" int cel_gpu_mat_dia_info(const cel_gpu_mat* A, int* ndiag, int* offsets)
{
    if (!A) return fail(CEL_ERR_ARG, "null matrix");
    if (ndiag) *ndiag = A->m.dia_nd;
    if (offsets)
        for (int d = 0; d < A->m.dia_nd; ++d) offsets[d] = A->m.dia_off[d];
    return CEL_OK;
}

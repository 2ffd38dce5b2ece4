// rowclass.hip -- derived forms of a block's CSR arrays for long solves (no
// reference counterpart).
//
// A solve reads its matrix hundreds of times, and the matrices of structured
// grids repeat themselves: the rows of a constant-coefficient stencil on a
// box differ only by which neighbours exist (27 kinds of row for 7 points),
// piecewise constant coefficients add one kind per material boundary.  A
// block whose entries lie on at most 8 diagonals and whose rows take at
// most 256 different forms (offsets, value bits, Jacobi value) is kept as
// one byte per row and a table of the forms: the product then reads 1 byte
// per row instead of 84 (FP64 CSR) or 57 (DIA), and the vector kernels take
// the Jacobi value from the table too.  A block on at most 8 diagonals with
// more forms than that (variable coefficients) is kept in diagonal storage,
// as cel_gpu_mat_to_dia builds it, for solves that asked for CSR.
//
// Where diagonal storage holds the same value at (i, j) and (j, i), bit for
// bit (checked once; the caller's own DIA form too), the product reads the
// diagonals above the main one for both and leaves those below it alone.
//
// All forms visit a row's entries in the CSR column order with the same
// values, so the sums are the CSR sums bit for bit.  The table is verified
// entry by entry against the matrix (the 64-bit keys only find candidates).
// They are built on the first long solve of a matrix (rule at
// derived_prepare), belong to the handle, and are dropped when the values,
// the Jacobi vector or the scaling change.  A matrix off the diagonals costs a
// pass over its columns that stops early, one of too many forms that pass and
// a look at 1,024 rows; without memory for them the solve runs on the CSR
// arrays.  The memory they take is returned when another allocation needs
// it (device_malloc) and no solve is reading them.
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "cel_internal.hpp"
#include "device_common.hpp"
#include "spmv_device.hpp"

namespace cel {
namespace {

constexpr int kKeySlots = 1024;  // open addressing, at most 256 keys
constexpr int kProbes = 32;
constexpr int kNear = 512;       // keys a block remembers (direct mapped)

struct KeyTable {
    unsigned long long key[kKeySlots];  // 0: free
    int cls[kKeySlots];
    int row[kMaxClass];                 // a row of each class
    int count;
    int over;  // more than kMaxClass classes, or a row that has no form
    int bad;   // a row that differs from its class (keys collided)
};

struct Offs {
    int nd;
    int off[kClassDiag];
};

// The finaliser of SplitMix64 (Steele, Lea, Flood 2014).
__device__ __forceinline__ unsigned long long mix(unsigned long long h)
{
    h ^= h >> 30;
    h *= 0xbf58476d1ce4e5b9ull;
    h ^= h >> 27;
    h *= 0x94d049bb133111ebull;
    return h ^ (h >> 31);
}

// A row's entries by diagonal, and its key (never 0).
struct RowForm {
    unsigned mask;
    double v[kClassDiag];
    unsigned long long key;
};

// false: the row has more entries than diagonals (a repeated column)
__device__ __forceinline__ bool row_form(long long i, const int* __restrict__ xadj,
                                         const int* __restrict__ cols,
                                         const double* __restrict__ vals, double jac, const Offs& O,
                                         RowForm& f)
{
    const int lo = xadj[i], len = xadj[i + 1] - lo;
    f.mask = 0;
#pragma unroll
    for (int d = 0; d < kClassDiag; ++d) f.v[d] = 0.0;
    if (len > O.nd) return false;
    int c[kClassDiag];
    double a[kClassDiag];
#pragma unroll
    for (int k = 0; k < kClassDiag; ++k) {
        c[k] = k < len ? cols[lo + k] - (int)i : 0;
        a[k] = k < len ? vals[lo + k] : 0.0;
    }
#pragma unroll
    for (int k = 0; k < kClassDiag; ++k)
#pragma unroll
        for (int d = 0; d < kClassDiag; ++d)
            if (k < len && d < O.nd && c[k] == O.off[d]) {
                f.mask |= 1u << d;
                f.v[d] = a[k];
            }
    unsigned long long h = mix(f.mask + 0x9e3779b97f4a7c15ull);
#pragma unroll
    for (int d = 0; d < kClassDiag; ++d)
        h = mix(h + __builtin_bit_cast(unsigned long long, f.v[d]) + (unsigned long long)d);
    h = mix(h + __builtin_bit_cast(unsigned long long, jac));
    f.key = h ? h : 1;
    return true;
}

__global__ void __launch_bounds__(kBlock) k_keys_clear(KeyTable* T)
{
    for (int i = threadIdx.x; i < kKeySlots; i += kBlock) {
        T->key[i] = 0;
        T->cls[i] = -1;
    }
    if (threadIdx.x == 0) T->count = T->over = T->bad = 0;
}

// Classes of the rows 0, step, 2 step, ...: one thread per row puts its key
// into the table unless the block has met it before.  Bound by one read of
// the matrix; it stops as soon as there are too many classes.  (Every
// resident block has put rows into the table before the first of them can
// see that: 254 us on 128^3, 814 us on 256^3.  Hence the sample, a row per
// thread of a few blocks, ahead of the whole block: the first solve of a
// matrix with variable coefficients takes 207 us more than the next one at
// 857,000 rows, 351 us at 128^3, 403 and 589 us without.)
constexpr int kSample = 1024;
__global__ void __launch_bounds__(kBlock)
k_class_scan(int n, long long step, const int* __restrict__ xadj, const int* __restrict__ cols,
             const double* __restrict__ vals, const double* __restrict__ jac, Offs O, KeyTable* T)
{
    __shared__ unsigned long long near_key[kNear];
    __shared__ int stop;
    for (int i = threadIdx.x; i < kNear; i += kBlock) near_key[i] = 0;
    __syncthreads();
    for (long long i0 = (long long)blockIdx.x * kBlock; i0 * step < n; i0 += (long long)gridDim.x * kBlock) {
        const long long i = (i0 + threadIdx.x) * step;
        if (i < n) {
            RowForm f;
            if (!row_form(i, xadj, cols, vals, jac[i], O, f)) {
                atomicOr(&T->over, 1);
            } else {
                const int at = (int)(f.key % kNear);
                if (near_key[at] != f.key && !*(volatile int*)&T->over) {
                    bool found = false;
                    int s = (int)(f.key >> 32) & (kKeySlots - 1);
                    for (int k = 0; k < kProbes && !found; ++k, s = (s + 1) & (kKeySlots - 1)) {
                        // (a plain look first: atomics of every row on the same
                        // few keys took 11 ms on the 256^3 block)
                        unsigned long long old = T->key[s];
                        if (old == 0) old = atomicCAS(&T->key[s], 0ull, f.key);
                        if (old == 0) {
                            const int id = atomicAdd(&T->count, 1);
                            if (id < kMaxClass) {
                                T->row[id] = (int)i;
                                T->cls[s] = id;
                            } else {
                                atomicOr(&T->over, 1);
                            }
                        }
                        found = old == 0 || old == f.key;
                    }
                    if (!found) atomicOr(&T->over, 1);
                    near_key[at] = f.key;
                }
            }
        }
        __syncthreads();
        if (threadIdx.x == 0) stop = *(volatile int*)&T->over;
        __syncthreads();
        if (stop) break;  // uniform
    }
}

// The table of the forms: thread c writes class c.
__global__ void __launch_bounds__(kBlock)
k_class_table(int count, const KeyTable* __restrict__ T, const int* __restrict__ xadj,
              const int* __restrict__ cols, const double* __restrict__ vals,
              const double* __restrict__ jac, const float* __restrict__ jac32, Offs O,
              RowClasses out)
{
    const int c = threadIdx.x;
    RowForm f;
    f.mask = 0;
    double j64 = 0.0;
    float j32 = 0.0f;
#pragma unroll
    for (int d = 0; d < kClassDiag; ++d) f.v[d] = 0.0;
    if (c < count) {
        const int i = T->row[c];
        j64 = jac[i];
        j32 = jac32[i];
        (void)row_form(i, xadj, cols, vals, j64, O, f);
    }
#pragma unroll
    for (int d = 0; d < kClassDiag; ++d) {
        out.val64[c * kClassDiag + d] = f.v[d];
        out.val32[c * kClassDiag + d] = (float)f.v[d];
    }
    out.mask[c] = f.mask;
    out.jac64[c] = j64;
    out.jac32[c] = j32;
}

// Every row's class, checked against the table bit for bit.
__global__ void __launch_bounds__(kBlock)
k_class_assign(int n, const int* __restrict__ xadj, const int* __restrict__ cols,
               const double* __restrict__ vals, const double* __restrict__ jac,
               const float* __restrict__ jac32, Offs O, KeyTable* T, RowClasses tab,
               uint8_t* __restrict__ cls)
{
    __shared__ unsigned long long near_key[kNear];
    __shared__ int near_cls[kNear];
    for (int i = threadIdx.x; i < kNear; i += kBlock) near_key[i] = 0;
    __syncthreads();
    int any = 0;
    for (long long i0 = (long long)blockIdx.x * kBlock; i0 < n; i0 += (long long)gridDim.x * kBlock) {
        const long long i = i0 + threadIdx.x;
        int id = -1;
        RowForm f;
        f.key = 0;
        const double j = i < n ? jac[i] : 0.0;
        if (i < n && row_form(i, xadj, cols, vals, j, O, f)) {
            const int at = (int)(f.key % kNear);
            if (near_key[at] == f.key) {
                id = near_cls[at];
            } else {
                int s = (int)(f.key >> 32) & (kKeySlots - 1);
                for (int k = 0; k < kProbes; ++k, s = (s + 1) & (kKeySlots - 1)) {
                    if (T->key[s] != f.key) continue;
                    id = T->cls[s];
                    break;
                }
            }
        }
        __syncthreads();  // every lookup of the block is done
        if (id >= 0) {  // the threads of one slot write whole pairs one after another, checked below
            const int at = (int)(f.key % kNear);
            near_key[at] = f.key;
        }
        __syncthreads();
        if (id >= 0 && near_key[(int)(f.key % kNear)] == f.key) near_cls[(int)(f.key % kNear)] = id;
        __syncthreads();
        if (i >= n) continue;
        bool same = id >= 0;
        if (same) {
            same = tab.mask[id] == f.mask &&
                   __builtin_bit_cast(unsigned long long, tab.jac64[id]) == __builtin_bit_cast(unsigned long long, j) &&
                   __builtin_bit_cast(unsigned, tab.jac32[id]) == __builtin_bit_cast(unsigned, jac32[i]);
#pragma unroll
            for (int d = 0; d < kClassDiag; ++d)
                same = same && __builtin_bit_cast(unsigned long long, tab.val64[id * kClassDiag + d]) ==
                                   __builtin_bit_cast(unsigned long long, f.v[d]);
        }
        if (!same) any = 1;
        cls[i] = (uint8_t)(same ? id : 0);
    }
    if (any) atomicOr(&T->bad, 1);
}

// Whether every entry below the main diagonal has its value bit for bit
// above it (entry (i, i + o), o < 0, in the array of -o at i + o).  One read
// of the arrays; a diagonal without a partner is read from its own.
template <typename VT>
__global__ void __launch_bounds__(kBlock)
k_dia_symmetric(int n, Offs O, const VT* __restrict__ vals, const uint8_t* __restrict__ mask, int* bad)
{
    using Bits = std::conditional_t<sizeof(VT) == 8, unsigned long long, unsigned>;
    int differs = 0;
    for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long long)gridDim.x * kBlock) {
        const unsigned m = mask[i];
#pragma unroll
        for (int d = 0; d < kClassDiag; ++d)
#pragma unroll
            for (int u = d + 1; u < kClassDiag; ++u)
                if (u < O.nd && O.off[d] < 0 && O.off[u] == -O.off[d] && ((m >> d) & 1u))
                    differs |= __builtin_bit_cast(Bits, vals[(long long)d * n + i]) !=
                               __builtin_bit_cast(Bits, vals[(long long)u * n + i + O.off[d]]);
    }
    if (differs) *(volatile int*)bad = 1;
}

int grid_of(long long n)
{
    const long long g = (n + kBlock - 1) / kBlock, cap = (long long)rt().num_cus * 16;
    return (int)(g < 1 ? 1 : g > cap ? cap : g);
}

// The classes of A's rows into A.derived; *ok = false: the rows do not fit.
int build_classes(Mat& A, const Offs& O, bool* ok)
{
    *ok = false;
    Derived& D = A.derived;
    hipStream_t st = rt().stream;
    DevBuf<KeyTable> T;
    CEL_TRY(T.alloc(1));
    hipLaunchKernelGGL(k_keys_clear, dim3(1), dim3(kBlock), 0, st, T.p);
    int h[3];
    const long long sample = std::max(1LL, (long long)A.n / kSample);
    for (const long long step : {sample, 1LL}) {
        const long long rows = (A.n + step - 1) / step;
        hipLaunchKernelGGL(k_class_scan, dim3(grid_of(rows)), dim3(kBlock), 0, st, A.n, step, A.xadj.p, A.cols.p,
                           A.vals.p, A.jac.p, O, T.p);
        CEL_HIP(hipGetLastError());
        CEL_HIP(hipMemcpyAsync(h, &T.p->count, sizeof(h), hipMemcpyDeviceToHost, st));
        CEL_HIP(hipStreamSynchronize(st));
        if (h[1] || h[0] > kMaxClass) return CEL_OK;
    }
    CEL_TRY(D.cls.alloc((size_t)A.n, true));
    CEL_TRY(D.tab64.alloc((size_t)kMaxClass * (kClassDiag + 1), true));
    CEL_TRY(D.tab32.alloc((size_t)kMaxClass * (kClassDiag + 1), true));
    CEL_TRY(D.tabm.alloc(kMaxClass, true));
    const RowClasses tab = D.classes();
    hipLaunchKernelGGL(k_class_table, dim3(1), dim3(kBlock), 0, st, h[0], T.p, A.xadj.p, A.cols.p, A.vals.p,
                       A.jac.p, A.jac32.p, O, tab);
    hipLaunchKernelGGL(k_class_assign, dim3(grid_of(A.n)), dim3(kBlock), 0, st, A.n, A.xadj.p, A.cols.p, A.vals.p,
                       A.jac.p, A.jac32.p, O, T.p, tab, D.cls.p);
    CEL_HIP(hipGetLastError());
    CEL_HIP(hipMemcpyAsync(h, &T.p->count, sizeof(h), hipMemcpyDeviceToHost, st));
    CEL_HIP(hipStreamSynchronize(st));
    *ok = !h[2];
    return CEL_OK;
}

template <typename VT>
int dia_symmetric(const Mat& A, int nd, const int* off, const VT* vals, const uint8_t* mask, signed char* sym)
{
    if (*sym >= 0) return CEL_OK;
    *sym = 0;
    Offs O{};
    O.nd = nd;
    for (int d = 0; d < nd; ++d) O.off[d] = off[d];
    hipStream_t st = rt().stream;
    DevBuf<int> bad;
    CEL_TRY(bad.alloc(1));
    CEL_HIP(hipMemsetAsync(bad.p, 0, sizeof(int), st));
    hipLaunchKernelGGL(k_dia_symmetric<VT>, dim3(grid_of(A.n)), dim3(kBlock), 0, st, A.n, O, vals, mask, bad.p);
    CEL_HIP(hipGetLastError());
    int h = 1;
    CEL_HIP(hipMemcpyAsync(&h, bad.p, sizeof(int), hipMemcpyDeviceToHost, st));
    CEL_HIP(hipStreamSynchronize(st));
    *sym = !h;
    return CEL_OK;
}

}  // namespace

int dia_bases(int n, int nd, const int* off, bool symmetric, long long* base)
{
    int arrays = nd;
    for (int d = 0; d < nd; ++d) {
        base[d] = (long long)d * n;
        if (!symmetric || off[d] >= 0) continue;
        for (int u = d + 1; u < nd; ++u)
            if (off[u] == -off[d]) {
                base[d] = (long long)u * n + off[d];
                --arrays;
                break;
            }
    }
    return arrays;
}

// The forms that a solve has looked at, as a list through them.
static std::mutex forms_lock;
static Derived* forms = nullptr;

void DerivedUse::begin(Derived& D)
{
    end();
    std::lock_guard<std::mutex> lock(forms_lock);
    if (!D.listed) {
        D.listed = true;
        D.after = forms;
        if (forms) forms->before = &D;
        forms = &D;
    }
    ++D.users;
    d = &D;
}

void DerivedUse::end()
{
    if (!d) return;
    std::lock_guard<std::mutex> lock(forms_lock);
    --d->users;
    d = nullptr;
}

bool derived_give_back()
{
    std::lock_guard<std::mutex> lock(forms_lock);
    bool any = false;
    for (Derived* D = forms; D; D = D->after)
        if (D->users == 0 && (D->cls.p || D->mask8.p || D->vals.p || D->vals32.p)) {
            D->release();
            any = true;
        }
    return any;
}

Derived::~Derived()
{
    std::lock_guard<std::mutex> lock(forms_lock);
    if (!listed) return;
    if (after) after->before = before;
    (before ? before->after : forms) = after;
}

void Derived::drop()
{
    std::lock_guard<std::mutex> lock(forms_lock);
    release();
}

void Derived::release()
{
    kind = kNone;
    tried = tried32 = tried64 = false;
    nd = 0;
    sym[0] = sym[1] = sym[2] = -1;
    cls.release();
    tab64.release();
    tab32.release();
    tabm.release();
    vals.release();
    vals32.release();
    mask8.release();
}

// Which derived form a solve of A (CSR or DIA form, no halo blocks) runs on;
// builds it on the first call that wants it.  Never fails: what cannot be
// built is not used.
int derived_prepare(Mat& A, int fmt, bool mixed, int iter_max, bool* symmetric)
{
    *symmetric = false;
    Derived& D = A.derived;
    // Smaller solves live in the caches and their iterations are launches;
    // few iterations do not pay for the passes over the matrix.  Measured per
    // iteration, CSR arrays / classes / diagonal storage: 64^3 FP64 17.2 /
    // 17.0 / 17.1 us; 80^3 29.1 / 25.4 / 27.8, mixed 22.9 / 22.0 / 21.4;
    // 100^3 39.6 / 26.5 / 30.7, mixed 31.8 / 22.5 / 28.4; 256^3 618 / 240 /
    // 411, mixed 358 / 127 / 232 (FP64 diagonals of 100^3 and 256^3
    // symmetric).  Building (a first solve less the next one): classes 0.21 ms
    // at 857,000 rows, 0.30 at 128^3, 0.8 at 200^3, 1.6 at 256^3, diagonals
    // 0.21, 0.35, 1.1, 1.7: what 5 (256^3) to 25 iterations save, in the mixed
    // form at 80^3 200.  (FP64 classes would pay there after 60.)  The
    // solve's length is not known here, only iter_max: one that stops after
    // 10 iterations has paid for more than it saved (128^3 Poisson FP64 0.93
    // ms, the next one 0.60).
    if (A.n < kDerivedRows || (iter_max < 32 && !D.tried) || !A.jac.p || !A.jac32.p) return Derived::kNone;
    const std::string err = last_error();
    int rc = CEL_OK;
    if (!D.tried) {
        D.tried = true;
        bool asc = false;
        int nd = 0;
        if (A.ncols == A.n && A.nnz > 0 && (long long)A.n * 8 < (1LL << 31))
            rc = dia_offsets(A, kClassDiag, &nd, D.off, &asc);
        if (rc == CEL_OK && asc && nd <= kClassDiag) {
            D.nd = nd;
            Offs O{};
            O.nd = nd;
            for (int d = 0; d < nd; ++d) O.off[d] = D.off[d];
            bool ok = false;
            rc = build_classes(A, O, &ok);
            if (rc == CEL_OK && ok) D.kind = Derived::kClasses;
        }
        if (D.kind == Derived::kNone) {
            D.cls.release();
            D.tab64.release();
            D.tab32.release();
            D.tabm.release();
        }
    }
    int use = D.kind;
    if (use == Derived::kNone && fmt == CEL_FMT_CSR && D.nd > 0 && (long long)D.nd * A.n <= 2LL * A.nnz) {
        // diagonal storage in the precision of the solve; the matrix's own
        // DIA form, where the caller has built one, is the same
        bool& tried = mixed ? D.tried32 : D.tried64;
        const size_t cnt = (size_t)D.nd * (size_t)A.n;
        if (!tried) {
            tried = true;
            rc = D.mask8.p ? CEL_OK : D.mask8.alloc((size_t)A.n, true);
            if (rc == CEL_OK) rc = mixed ? D.vals32.alloc(cnt, true) : D.vals.alloc(cnt, true);
            if (rc == CEL_OK)
                rc = dia_fill(A, D.nd, D.off, mixed ? nullptr : D.vals.p, mixed ? D.vals32.p : nullptr, D.mask8.p);
            if (rc != CEL_OK) {
                if (mixed) D.vals32.release();
                else D.vals.release();
            }
        }
        if (D.mask8.p && (mixed ? (const void*)D.vals32.p : (const void*)D.vals.p)) {
            use = Derived::kDiagonals;
            signed char& y = D.sym[mixed ? Derived::kVals32 : Derived::kVals];
            if (rc == CEL_OK)
                rc = mixed ? dia_symmetric(A, D.nd, D.off, D.vals32.p, D.mask8.p, &y)
                           : dia_symmetric(A, D.nd, D.off, D.vals.p, D.mask8.p, &y);
            *symmetric = y == 1;
        }
    }
    // the caller's diagonal storage; the line of the rule above holds here too:
    // per iteration FP64 70^3 20.8 us either way, 80^3 23.4 without / 24.8
    // with the symmetric walk, 90^3 27.1 / 26.9, 100^3 33.1 / 30.7, 112^3 41.6
    // / 38.8, 128^3 58.3 / 51.8.  In the mixed form the other way is two
    // kernels per iteration (but for long rows): 804,264 rows 21.0 / 21.5, 820,911 21.5 / 21.6,
    // 100^3 23.2 / 21.0, 1,092,624 25.0 / 22.8, 1,179,780 25.9 / 24.8
    constexpr int kSymmetricMixed = 850000;
    const bool look = !mixed || A.n >= kSymmetricMixed || csr_long_rows(A);
    if (use == Derived::kNone && fmt == CEL_FMT_DIA && look && A.dia_nd > 0 && A.dia_nd <= kClassDiag && A.dia_mask8.p) {
        signed char& y = D.sym[Derived::kOwnDia];  // (the FP32 copy of the values follows the FP64 ones)
        if (rc == CEL_OK) rc = dia_symmetric(A, A.dia_nd, A.dia_off, A.dia_vals.p, A.dia_mask8.p, &y);
        *symmetric = y == 1;
    }
    if (rc != CEL_OK) {  // no memory: no error of the solve
        set_error(err);
        (void)hipGetLastError();
    }
    return use;
}

// The matrices of a batch are read by one K1 per iteration however small each
// of them is, so those below kDerivedRows get diagonal storage too, built
// with two synchronisations for all of them.  One costs about 33 us of
// kernels and its allocations, and saves 2.2 ns a row in 200 iterations.
constexpr int kBatchRows = 20000;

// Whether derived_prepare_all would try the matrix: as derived_prepare (large),
// or in diagonal storage.
static bool wanted_large(const Mat& A)
{
    const Derived& D = A.derived;
    return A.n >= kDerivedRows && (!D.tried || (D.kind == Derived::kNone && D.nd > 0 && !D.tried64 &&
                                                (long long)D.nd * A.n <= 2LL * A.nnz));
}
static bool wanted_small(const Mat& A)
{
    return A.n < kDerivedRows && A.n >= kBatchRows && !A.derived.tried64 && A.nnz > 0 && A.ncols == A.n;
}
bool derived_wanted(const std::vector<Mat*>& mats, int iter_max)
{
    return iter_max >= 32 && std::any_of(mats.begin(), mats.end(),
                                         [](const Mat* A) { return wanted_large(*A) || wanted_small(*A); });
}

void derived_prepare_all(const std::vector<Mat*>& mats, int iter_max)
{
    if (iter_max < 32) return;
    const std::string err = last_error();
    std::vector<Mat*> todo;
    for (Mat* A : mats) {
        bool sym;
        if (wanted_large(*A)) {
            (void)derived_prepare(*A, CEL_FMT_CSR, false, iter_max, &sym);
        } else if (wanted_small(*A)) {
            A->derived.tried64 = true;  // (a matrix may be in the batch twice)
            todo.push_back(A);
        }
    }
    if (todo.empty()) return;
    std::vector<DiagonalSet> sets;
    int rc = dia_offsets_all(todo, kClassDiag, sets);
    hipStream_t st = rt().stream;
    DevBuf<int> bad;
    if (rc == CEL_OK) rc = bad.alloc(todo.size());
    if (rc == CEL_OK && hipMemsetAsync(bad.p, 0, sizeof(int) * todo.size(), st) != hipSuccess)
        rc = CEL_ERR_HIP;
    std::vector<char> built(todo.size(), 0);
    for (size_t q = 0; q < todo.size() && rc == CEL_OK; ++q) {
        Mat& A = *todo[q];
        Derived& D = A.derived;
        if (!sets[q].ascending || sets[q].nd > kClassDiag || (long long)sets[q].nd * A.n > 2LL * A.nnz) continue;
        rc = D.mask8.alloc((size_t)A.n, true);
        if (rc == CEL_OK) rc = D.vals.alloc((size_t)sets[q].nd * (size_t)A.n, true);
        if (rc == CEL_OK) rc = dia_fill(A, sets[q].nd, sets[q].off, D.vals.p, nullptr, D.mask8.p);
        if (rc != CEL_OK) break;
        Offs O{};
        O.nd = sets[q].nd;
        for (int d = 0; d < O.nd; ++d) O.off[d] = sets[q].off[d];
        hipLaunchKernelGGL(k_dia_symmetric<double>, dim3(grid_of(A.n)), dim3(kBlock), 0, st, A.n, O, D.vals.p,
                           D.mask8.p, bad.p + q);
        built[q] = 1;
    }
    std::vector<int> h(todo.size(), 1);
    if (bad.p) {
        const bool ok = hipGetLastError() == hipSuccess &&
                        hipMemcpyAsync(h.data(), bad.p, sizeof(int) * h.size(), hipMemcpyDeviceToHost, st) == hipSuccess &&
                        hipStreamSynchronize(st) == hipSuccess;
        for (size_t q = 0; q < todo.size(); ++q) {
            Derived& D = todo[q]->derived;
            if (ok && built[q]) {
                D.nd = sets[q].nd;
                for (int d = 0; d < D.nd; ++d) D.off[d] = sets[q].off[d];
                D.sym[Derived::kVals] = !h[q];
            } else {
                D.vals.release();
                D.mask8.release();
            }
        }
    }
    if (rc != CEL_OK) {  // no memory: those matrices are read as they are
        set_error(err);
        (void)hipGetLastError();
    }
}

}  // namespace cel

// cel_internal.hpp -- shared declarations of the gfx950 library behind the
// C ABI in include/cel_gpu.h.  Host code is C++17, device code is HIP for
// CDNA4 (64-lane wavefronts).  Nothing here is visible outside the library.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <string>
#include <vector>

#include "../../include/cel_gpu.h"

namespace cel {

// ---------------------------------------------------------------- errors
void set_error(const std::string& msg);
const std::string& last_error();
int fail(int code, const std::string& msg);

#define CEL_HIP(call)                                                              \
    do {                                                                           \
        hipError_t e_ = (call);                                                    \
        if (e_ != hipSuccess)                                                      \
            return ::cel::fail(CEL_ERR_HIP, std::string(#call) + ": " +            \
                                                hipGetErrorString(e_));            \
    } while (0)

#define CEL_TRY(call)                      \
    do {                                   \
        int s_ = (call);                   \
        if (s_ < 0) return s_;             \
    } while (0)

// ---------------------------------------------------------------- runtime
struct Runtime {
    int device = -1;
    hipStream_t stream = nullptr;
    int num_cus = 0;
    bool ready = false;
};
Runtime& rt();
int ensure_init();

// Blocks of `kernel` (256 threads) resident on the whole GPU at once; a
// persistent grid never exceeds this, so no block waits for a second wave.
int resident_grid(const void* kernel, long long work_items);

// Device memory of the library's buffers.  A freed block is kept for the next
// buffer of about its size instead of going back to the driver, whose
// allocations and (synchronising) frees of large blocks cost 0.1-0.2 ms
// each.  Kept blocks are bounded (kPoolBytes in all), go back when an
// allocation of the library fails (device_malloc: cel_gpu_malloc's too) and
// with cel_gpu_finalize.  A reused block may still be
// read by work on the library's stream, so that is waited for before it is
// handed out; the lists are per device and locked.
constexpr size_t kPoolBytes = size_t(2) << 30;
void* pool_alloc(size_t bytes, size_t* got, int* device, bool spare);  // null: no memory
void pool_free(void* p, size_t bytes, int device);
// hipMalloc; before it fails (null) it gives the kept blocks back and, unless
// the memory is only wanted where there is some to spare, the derived forms
// that no solve is reading.
void* device_malloc(size_t bytes, bool spare = false);
void pool_release();

// Device buffer owned by the library.
template <typename T>
struct DevBuf {
    T* p = nullptr;
    size_t n = 0;
    size_t bytes = 0;  // of the block
    int device = -1;
    DevBuf() = default;
    DevBuf(const DevBuf&) = delete;
    DevBuf& operator=(const DevBuf&) = delete;
    ~DevBuf() { release(); }
    int alloc(size_t count, bool spare = false) {
        if (count == n && p) return CEL_OK;
        release();
        if (count == 0) return CEL_OK;
        p = static_cast<T*>(pool_alloc(count * sizeof(T), &bytes, &device, spare));
        if (!p) {
            return fail(CEL_ERR_OOM, "hipMalloc of " + std::to_string(count * sizeof(T)) + " bytes failed");
        }
        n = count;
        return CEL_OK;
    }
    // at least `count` elements, keeping a larger allocation (a workspace
    // reused from call to call)
    int reserve(size_t count) {
        if (p && n >= count) return CEL_OK;
        return alloc(count);
    }
    void release() {
        if (p) pool_free(p, bytes, device);
        p = nullptr;
        n = 0;
    }
};

// The events, pinned host buffers and graph one host routine creates on a
// stream, released on every return path once the stream has drained (so no
// copy still targets a pinned buffer).
struct StreamScope {
    hipStream_t s;
    std::vector<hipEvent_t> ev;
    std::vector<void*> pinned;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    explicit StreamScope(hipStream_t st) : s(st) {}
    StreamScope(const StreamScope&) = delete;
    StreamScope& operator=(const StreamScope&) = delete;
    ~StreamScope()
    {
        (void)hipStreamSynchronize(s);
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
        for (hipEvent_t e : ev) (void)hipEventDestroy(e);
        for (void* q : pinned) (void)hipHostFree(q);
    }
    int event(hipEvent_t& e, unsigned flags = hipEventDefault)
    {
        if (hipEventCreateWithFlags(&e, flags) != hipSuccess) return fail(CEL_ERR_HIP, "hipEventCreate failed");
        ev.push_back(e);
        return CEL_OK;
    }
    template <typename T>
    int host_alloc(T*& p, size_t count)
    {
        void* q = nullptr;
        if (hipHostMalloc(&q, sizeof(T) * (count > 0 ? count : 1), hipHostMallocDefault) != hipSuccess)
            return fail(CEL_ERR_OOM, "hipHostMalloc failed");
        pinned.push_back(q);
        p = static_cast<T*>(q);
        return CEL_OK;
    }
};

// ---------------------------------------------------------------- matrix
struct Workspace;  // PCG work vectors, owned by the matrix handle (pcg.hip)
// One halo block: entries of local rows whose columns belong to another
// rank's range, stored row-sorted.  Column indices are positions in that
// block's receive buffer (ghost slot), so the halo SpMV reads the packed
// face values directly instead of a full-length copy of the neighbour's
// vector.
struct HaloBlock {
    int proc = -1;        // owning rank of the columns
    int nnz = 0;
    int col_offset = 0;   // vtxdist(proc+1)-1, as the reference stores it
    int proc_len = 0;     // rows owned by proc
    int recv_len = 0;     // number of distinct referenced columns
    int recv_base = 0;    // offset of this block's slots in the ghost region
    // host copies kept for getters (reference layout, 1-based, global ids)
    std::vector<int> h_rows, h_cols;
    std::vector<double> h_vals;
    std::vector<int> h_xadj;       // cel_sp_mat_to_csr of this block
    std::vector<int> h_recv_perm;  // ascending local column ids (1-based)
};

// Derived forms of a block for long solves (rowclass.hip).  They only save
// time: they are built in memory that is to spare, and those no solve is
// reading go back when an allocation of the library fails.
constexpr int kMaxClass = 256;   // row forms a byte tells apart
constexpr int kClassDiag = 8;    // diagonals of a row form
constexpr int kDerivedRows = 800000;

// Table of the row forms, by class: values by diagonal, presence mask,
// Jacobi value (device pointers).
struct RowClasses {
    double *val64, *jac64;
    float *val32, *jac32;
    uint32_t* mask;
};

struct Derived {
    enum { kNone = 0, kClasses, kDiagonals };
    int kind = kNone;  // kClasses once the classes are built
    bool tried = false, tried32 = false, tried64 = false;
    int nd = 0;        // diagonals (0: more than kClassDiag, or unsorted rows)
    int off[32] = {};  // ascending
    enum { kOwnDia = 0, kVals, kVals32 };
    signed char sym[3] = {-1, -1, -1};  // symmetric: Mat::dia_vals, vals, vals32 (-1: not looked at)
    DevBuf<uint8_t> cls;      // per row: its class
    DevBuf<double> tab64;     // val64, then jac64
    DevBuf<float> tab32;
    DevBuf<uint32_t> tabm;
    DevBuf<double> vals;      // diagonal storage of a CSR solve, as Mat::dia_vals
    DevBuf<float> vals32;
    DevBuf<uint8_t> mask8;
    RowClasses classes() const
    {
        return RowClasses{tab64.p, tab64.p + kMaxClass * kClassDiag, tab32.p, tab32.p + kMaxClass * kClassDiag,
                          tabm.p};
    }
    int users = 0;   // solves that read it (DerivedUse)
    bool listed = false;  // among the forms derived_give_back looks at
    Derived *before = nullptr, *after = nullptr;
    ~Derived();
    void release();
    void drop();     // release, for a handle that no solve is reading
};
bool derived_give_back();  // drops every form without users; false: there was none

// Marks a handle's form as being read (or built) until it goes out of scope.
struct DerivedUse {
    Derived* d = nullptr;
    DerivedUse() = default;
    DerivedUse(const DerivedUse&) = delete;
    DerivedUse& operator=(const DerivedUse&) = delete;
    ~DerivedUse() { end(); }
    void begin(Derived& D);
    void end();
};

// The kernels the last PCG or GMRES solve of a handle ran on: what
// cel_gpu_internal_path reports, so that tests see which path they are on.
struct SolvePath {
    const char* form = "";  // the K1's matrix: csr, csr-long, dia, jad, classes; gmres
    bool step = false;      // two kernels per iteration (GMRES: one launch per column)
    bool direct = false;    // the step reads every row by its own thread
    bool window = false;    // x of a band, or of a chunk, in LDS
    bool wide = false;      // several rows per lane
    bool deep = false;      // long rows several entries at a time
    bool keep = false;      // the matrix loaded to stay in the cache
    int stream = 0;         // vectors marked as read once: 0 none, 1 x, 2 all
};

struct Mat {
    int n = 0;          // local rows
    int ncols = 0;      // local columns (== n for a square local block)
    int nnz = 0;        // local block entries
    int row_offset = 0; // global row of local row 1 is row_offset+1
    int col_offset = 0; // subtracted from global columns of the local block

    // local block, CSR, 0-based on the device
    DevBuf<int> xadj, cols;
    DevBuf<double> vals;
    DevBuf<float> vals32;  // FP32 copy for the mixed-precision inner solve

    // diagonal, Jacobi vector, row scaling
    DevBuf<double> diag, jac, scaled_diag;
    DevBuf<float> jac32;
    bool has_diag = false, has_jac = false, jac_row_scaled = false, is_scaled = false;

    // JAD (0-based on the device)
    int jad_mmax = 0, jad_ilo = 0, jad_ndef = 0, jad_mode = -1;
    long long jad_nnz = 0;
    DevBuf<int> jad_perm, jad_begin, jad_cols;
    DevBuf<double> jad_vals;
    DevBuf<float> jad_vals32;
    // the JAD columns renumbered into the permuted row order (pinv[cols]),
    // for solves that keep their vectors in that order; built on first use
    DevBuf<int> jad_pcols;

    // DIA (cel_gpu_mat_to_dia): values [ndiag][n], presence mask per row
    int dia_nd = 0;                 // 0: no DIA form
    int dia_off[32] = {};           // ascending column - row offsets
    DevBuf<double> dia_vals;
    DevBuf<float> dia_vals32;
    DevBuf<uint32_t> dia_mask;      // presence bits per row (more than 8 diagonals)
    DevBuf<uint8_t> dia_mask8;      // the same in one byte (at most 8 diagonals)
    std::vector<int> h_jad_begin;  // host copy (0-based starts, mmax+1)

    Derived derived;
    int band = -1;     // largest |column - row| of the block (-1: not looked up)
    int longest = -1;  // most entries of a row (-1: not looked up)
    SolvePath path;

    // halo (distributed block split of one rank)
    std::vector<HaloBlock> halo;
    int ghost_len = 0;             // sum of recv_len over halo blocks
    DevBuf<int> halo_xadj;         // CSR over local rows of the merged halo entries (n+1)
    DevBuf<int> halo_rows;         // rows having halo entries (compact list)
    DevBuf<int> halo_rowq;         // per local row: its compact index, or -1
    DevBuf<uint8_t> halo_flag;     // per local row: min(halo entries, 255); [n] = 0
    DevBuf<int> halo_wq;           // per 64-row group g: halo rows below row 64 g
    DevBuf<int> halo_ptr;          // per compact row: start into halo_cols/vals (+1 end)
    DevBuf<int> halo_cols;         // ghost slot per entry, in block order
    DevBuf<double> halo_vals;
    int halo_nrows = 0;
    DevBuf<int> send_perm;         // 0-based local indices packed per send list
    std::vector<int> send_len, send_base, send_proc;
    int send_total = 0;
    int nranks = 1, my_rank = 0;
    std::vector<int> vtxdist;      // 1-based starts, nranks+1
    std::vector<double> h_diag_split;  // diagonal captured during the split
    std::vector<int> h_local_rows, h_local_cols;  // local block in input order (global ids)
    std::vector<double> h_local_vals;

    Workspace* ws = nullptr;
};

void pcg_release_workspace(Mat* A);

// Whether the CSR kernels split the block's tiles by entries
// (CsrLongStream) instead of rows (CsrTileStream, whose stage holds 2,044
// entries of a 256-row tile; a larger tile is summed row by row from
// global memory).  The line lies just below the average at which a tile
// fills the stage (7.98), above the 7-point stencils, whose gathers of one
// diagonal by 64 neighbouring rows are contiguous: measured FP64, one
// product, split by rows / by entries: 100^3 7-point 21.7 / 25.4 us, 256^3
// 328 / 382 us; 1,000,003 mesh rows of 6.1 entries 43.3 / 41.4 us, of 11.1
// (split by rows: unstaged) 256 / 70 us.
inline bool csr_long_rows(const Mat& A) { return (double)A.nnz > 7.5 * (double)A.n; }

}  // namespace cel

// the opaque handle of the C ABI
struct cel_gpu_mat {
    cel::Mat m;
};

namespace cel {

// ---------------------------------------------------------------- kernels (host launchers)
// All launches go to rt().stream.
int launch_gen_poisson7(int nx, int ny, int nz, const double* kappa, int* xadj, int* cols,
                        double* vals);
// skip (may be null): the launch returns at once when *skip is non-zero on
// the device (for launches captured in a graph whose later replays must do
// nothing)
// coo = 1: the COO product of the same (row-sorted) entries, y(row) += a x
// entry by entry (from y itself when accumulating, else from 0)
int launch_csr_spmv(const Mat& A, const double* x, double* y, int accumulate,
                    const int* skip = nullptr, int coo = 0);
int launch_csr_spmv_f32(const Mat& A, const float* x, float* y, int accumulate, int coo = 0);
int launch_jad_spmv(const Mat& A, const double* x, double* y, int accumulate,
                    const int* skip = nullptr);
int launch_jad_spmv_f32(const Mat& A, const float* x, float* y, int accumulate);
int launch_dia_spmv(const Mat& A, const double* x, double* y, int accumulate,
                    const int* skip = nullptr);
int launch_dia_spmv_f32(Mat& A, const float* x, float* y, int accumulate);
// FP64 products fused with the dot product that follows them in the GMRES
// loop, over G fixed row chunks of `chunk` rows (a multiple of 256): block b
// covers rows [b*chunk, b*chunk + chunk) and writes part[b].
//   kFuseDot:   y = A x,        part[b] = sum of aux_i * y_i over chunk b
//   kFuseResid: y = aux - A x,  part[b] = sum of y_i * y_i over chunk b
// y holds the plain product's values bit for bit, and each thread adds its
// rows in ascending order before the block sum, so part[b] equals what a
// separate chunked dot kernel forms over the same rows.
enum { kFuseDot = 1, kFuseResid = 2 };
int launch_csr_spmv_fused(const Mat& A, int fuse, long long chunk, int G, const double* x,
                          double* y, const double* aux, double* part, const int* skip);
int launch_dia_spmv_fused(const Mat& A, int fuse, long long chunk, int G, const double* x,
                          double* y, const double* aux, double* part, const int* skip);
int dia_prepare_f32(Mat& A);
// The largest |column - row| of a square block.
int block_bandwidth(const Mat& A, int& bw);
// The most entries of a row.
int block_longest(const Mat& A, int& longest);
// The derived form (Derived::k*) a PCG solve of at most iter_max iterations
// runs on, built on the first call that wants it; never an error.  The caller
// holds a DerivedUse of A and has made its own allocations.
// *symmetric: the diagonal storage the solve runs on (its own or a derived
// one) holds bit for bit the same value at (i, j) and (j, i).
int derived_prepare(Mat& A, int fmt, bool mixed, int iter_max, bool* symmetric);
// The FP64 derived forms of a batch's matrices, smaller ones too.
void derived_prepare_all(const std::vector<Mat*>& mats, int iter_max);
// Whether it would try anything.
bool derived_wanted(const std::vector<Mat*>& mats, int iter_max);
// Where the wide walks find the values of nd <= kClassDiag diagonals: entry
// (i, d) at base[d] + i of storage [nd][n].  Symmetric: those below the main
// diagonal in the arrays above it, as entry (i, i + o), o < 0, is entry (i +
// o, i) of the diagonal -o, so a product reads 4 of 7 arrays.  Returns the
// number of arrays.
int dia_bases(int n, int nd, const int* off, bool symmetric, long long* base);
// The distinct offsets col - row of the local block, ascending, at most
// `most` (<= 32) of them: *nd = most + 1 when there are more.  *ascending:
// every row's columns strictly ascend (known only when *nd <= most).
int dia_offsets(const Mat& A, int most, int* nd, int* off, bool* ascending);
// dia_offsets of several matrices, with one synchronisation
struct DiagonalSet {
    int nd;
    int off[32];
    bool ascending;
};
int dia_offsets_all(const std::vector<Mat*>& mats, int most, std::vector<DiagonalSet>& out);
// Diagonal-major values (v64, or v32 rounded to FP32) and row masks on at
// most 8 diagonals; slots without an entry hold 0.
int dia_fill(const Mat& A, int nd, const int* off, double* v64, float* v32, uint8_t* mask8);
int launch_halo_spmv(const Mat& A, const double* ghost, double* y);
int launch_face_pack(const Mat& A, const double* x, double* sendbuf);
int launch_extract_diag(Mat& A);
int launch_set_jacobi(Mat& A, int row_scaled);
int launch_scale_rows(Mat& A);
int launch_scale_vec(const Mat& A, double* b);
int launch_to_f32(const double* src, float* dst, size_t n);
int launch_coo_to_csr(int nrows, int nnz, const int* rows0, int* xadj);  // rows 0-based local
// Frees the workspace the COO sort and row-offset routines keep between calls.
void coo_release_workspace();
int jad_convert_device(Mat& A, int mode);
// Builds A.jad_pcols (once per conversion).
int jad_prepare_permuted(Mat& A);
int launch_sddmm(const Mat& A, const double* lambda, const double* x, double* g);
int launch_kappa_grad(int nx, int ny, int nz, const double* kappa, const double* x,
                      const double* lambda, double* grad);

// bytes one y = A x moves, counted algorithmically (index + value streams,
// row pointers, one read of x and one write of y)
double spmv_bytes(const Mat& A, int format, int precision);

}  // namespace cel

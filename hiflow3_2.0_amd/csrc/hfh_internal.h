// hfh_internal.h -- private definitions of the gfx950 HIP platform library.
//
// Layout in HBM (all arrays 256-byte aligned by hipMalloc):
//   vector  : T[n] contiguous
//   CSR     : int32 row[nrow+1], int32 col[nnz] (ascending per row), T val[nnz],
//             int32 rblk[nrblk+1] row-block boundaries for the streaming SpMV,
//             int32 diag[nrow] position of the diagonal entry (-1 if absent)
//   reductions: per-context scratch of FP64 workgroup partials
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>
#include <cstdio>
#include <string>
#include <vector>

#include "../../include/hfh.h"

namespace hfh {

void set_error(const char *fmt, ...);

// Kernel launch geometry shared by the library.
constexpr int kBlock = 256;          // threads per workgroup (4 wave64)
constexpr int kSpmvTile = 1024;      // nnz staged per workgroup by the streaming SpMV
constexpr int kRedBlocks = 1024;     // max partials per reduction
// Dictionary-coded SELL copies (SpMV, MC-SGS sweeps): the code of a padding
// slot (a slot past its row's length), so kernels need no row lengths;
// dictionaries therefore hold at most 255 offsets
constexpr unsigned kPadCode = 255;
constexpr size_t kReportBytes = 8 << 10;   // pinned reports behind host_res
constexpr int kHostDot = 255;        // word of host_res that such a dot's result arrives in
constexpr int kNumXcd = 8;           // MI355X: 8 accelerator complex dies
// Size of the per-device static array that the allocation-free CG
// (hfh_pcg_solve_noalloc) works in: FP64 systems up to 2,096,000 rows.
constexpr size_t kStaticScratch = static_cast<size_t>(64) << 20;

struct Timing {
    bool on = false;
    long long launches[4] = {0, 0, 0, 0};
    double ms[4] = {0, 0, 0, 0};
};

}  // namespace hfh

namespace hfh {
struct JacobiSpace;
void jacobi_space_free(JacobiSpace *s);
}  // namespace hfh

struct hfh_ctx {
    int device = 0;
    int num_cu = 0;
    long long hbm = 0;
    char name[128] = {0};
    hipStream_t stream = nullptr;
    // reduction scratch: partials[kRedBlocks * 8] doubles, then result slots
    double *red = nullptr;            // device
    double *host_res = nullptr;       // pinned host mirror for results
    void *host_reports = nullptr;     // pinned, behind it: rows reported by a search for pairs
    unsigned long long *dot_slots = nullptr;   // partials of dots that the host waits for (in red)
    hfh::Timing timing;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    int live = 0;                     // vectors, matrices and preconditioners created on the context
    // device address of this device's static scratch array (hfh_krylov.hip)
    void *scratch = nullptr;
    int wait_polls = 0;               // hfh_ctx_set_wait_polls (0: each kernel's own)
    long long copy_limit = 0;         // hfh_ctx_set_copy_limit (0: none)
    long long cg_resident = 0, cg_gave_up = 0;   // one-launch CG solves, those that fell back
    // work space of the last Jacobi solve, for the next one (hfh_jacobi.hip)
    std::atomic<hfh::JacobiSpace *> jacobi{nullptr};
};

struct hfh_vec {
    hfh_ctx *ctx = nullptr;
    int n = 0;
    int dtype = HFH_F64;
    void *d = nullptr;
    // index set (lVector::set_indexset): device copy for the gather / scatter
    // of GetIndexedValues / SetIndexedValues, host copy for get_indexset
    int *iset = nullptr;
    std::vector<int> h_iset;
    size_t elem() const { return dtype == HFH_F64 ? 8 : 4; }
};

struct hfh_csr {
    hfh_ctx *ctx = nullptr;
    int nrow = 0, ncol = 0, nnz = 0, dtype = HFH_F64;
    int *row = nullptr, *col = nullptr;
    void *val = nullptr;
    int *rblk = nullptr;   // streaming row blocks
    int nrblk = 0;
    int spmv_algo = HFH_SPMV_STREAM, spmv_p1 = 2048;   // configured kernel
    int spmv_algo_req = 0, spmv_p1_req = 0, spmv_p2_req = 0;  // requested (0 = automatic)
    int nwg = 1;           // SpMV workgroups = partial sums of a fused dot
    std::vector<int> h_col;    // host copy of the columns, kept for the analyses
    // SELL-64 copy for HFH_SPMV_SELL: slices of 64 rows stored column-major
    int nslice = 0;
    int *sl_ptr = nullptr;     // [nslice+1] element offset of each slice
    int *sl_len = nullptr;     // [nrow] row lengths
    int *sl_col = nullptr;     // padded columns (padding points at the row itself)
    void *sl_val = nullptr;    // padded values (padding 0)
    bool sell_dirty = false;   // SELL copy must be rebuilt from the CSR arrays
    // HFH_SPMV_SELL_DICT: columns as one-byte codes into a table of distinct
    // column offsets (col - row); four codes of consecutive slots per word
    int *sd_dict = nullptr;    // [sd_ndict] offsets
    int sd_ndict = 0;
    unsigned *sd_code = nullptr;   // code words, column-major per slice
    int *sd_wptr = nullptr;    // [nslice+1] word offset of each slice
    int sd_code0 = 0;          // code of offset 0 (the diagonal)
    // HFH_SPMV_SELL_LDS: the pair layout's values with each slot's column as a
    // 16-bit index into its slice's LDS image of x (the slice's distinct
    // chunks of x, ascending): chunk position * sx_chunk + column % sx_chunk
    unsigned short *sx_code = nullptr;   // [slots] pair layout, padding 0
    unsigned short *sx_dcode = nullptr;  // [nrow] code of the diagonal (0xffff: none)
    int *sx_cptr = nullptr;    // [nslice+1] offset of each slice's chunk list
    int *sx_cid = nullptr;     // chunk ids (x index / sx_chunk)
    int sx_chunk = 0;          // elements per chunk (16)
    int sx_img = 0;            // largest image of a slice (chunks * sx_chunk)
    // Matrices of a few distinct (offset, value) pairs (hfh_pattern.hip), on
    // top of an automatically chosen SELL layout of one wave per slice
    bool pt_want = false;          // the layout was chosen automatically
    int pt_pairs = 0;              // pairs (0: the values do not repeat)
    int pt_omin = 0, pt_omax = 0;  // smallest and largest offset
    int pt_ngroups = 0;            // runs of up to three neighbouring offsets
    bool pt_tri = false;           // all of three
    void *pt_block = nullptr;      // device memory of the arrays below
    std::vector<char> pt_lists;    // the runs and the pairs' values, the kernel's argument
    int *pt_offs = nullptr;        // offsets of the pairs, ascending
    unsigned *pt_set = nullptr;    // [nrow] the pairs of each row, one bit each
    int *pt_partial = nullptr;     // [nslice] some row of the slice lacks a pair
    int *diag = nullptr;   // diagonal position per row
    // longest row and how far its columns reach below / above the row, of
    // square matrices small enough for the resident CG (else shape_len 0)
    int shape_len = 0, shape_lo = 0, shape_hi = 0;
    bool has_structure = false;
    bool sorted = true;      // columns ascending in every row (false after a diagonal-first swap)
    unsigned version = 0;    // bumped whenever the values or the structure change
    std::vector<int> h_row;  // host copy of the row pointer (for analysis)
    size_t elem() const { return dtype == HFH_F64 ? 8 : 4; }
};

// Level schedule on the device: rows in level order, level boundaries on host.
struct hfh_levels {
    int nlev = 0;
    std::vector<int> ptr;      // host, nlev+1
    int *rows = nullptr;       // device, nrow
    int *ptr_d = nullptr;      // device copy of ptr
    std::vector<std::pair<int, int>> runs;   // launch plan: level ranges [first, last)
};

// Rows of a preconditioner sweep in SELL-64 form, slices of 64 consecutive
// rows of one colour, column-major, padded to the longest row of the slice.
struct hfh_sweep {
    int nslice = 0;
    int *ptr = nullptr;        // [nslice+1] element offset of each slice
    int *len = nullptr;        // [nrow] entries of each row in this sweep
    int *col = nullptr;        // padded columns (padding: a row of the same slice)
    void *val = nullptr;       // padded values (padding 0)
    std::vector<int> slice0;   // host: first slice of each colour (ncolors+1)
    // with at most 256 distinct offsets col - row over the sweep's entries,
    // the columns are one-byte codes into `dict` instead (col is null):
    // code word w of a lane holds slots 4w..4w+3; the values keep the
    // slice's width, its code words cover it rounded up to 4 slots
    unsigned *code = nullptr;  // code words
    int *wptr = nullptr;       // [nslice+1] word offset of each slice
    int *dict = nullptr;       // [ndict] offsets, ascending (0 included: padding)
    int ndict = 0;
};

// Rows of a level-scheduled triangular sweep, sliced in level order: the rows
// of level l fill slices lslice[l] .. lslice[l+1] (64 rows each, lane = row),
// each slice column-major and padded to its longest row.  A row's entries are
// its lower (forward sweep) or upper (backward sweep) ones in stored order;
// its diagonal value sits beside them.  Values are refilled from the CSR
// arrays through the position maps when the matrix's values change.
struct hfh_tsweep {
    int nslice = 0;
    long long nent = 0;
    std::vector<int> lslice;   // host: first slice of each level (nlev + 1)
    int *lslice_d = nullptr;   // device copy
    int *ptr = nullptr;        // [nslice + 1] element offset of each slice
    int *row = nullptr;        // [64 nslice] row of each lane (-1: padding lane)
    int *len = nullptr;        // [64 nslice] entries of each lane
    int *col = nullptr;        // [nent] columns (padding: 0)
    int *pos = nullptr;        // [nent] CSR position of each entry (-1: padding)
    int *dpos = nullptr;       // [64 nslice] CSR position of each lane's diagonal (-1: padding)
    void *val = nullptr;       // [nent] values
    void *dval = nullptr;      // [64 nslice] diagonal values
    // Blocked form only (slices are geometric blocks of a structured grid,
    // in block-level order): a column below 0 names the lane -(col + 1) of
    // the same block, whose result arrives through a cross-lane shuffle
    int *lev = nullptr;        // [64 nslice] level of each lane inside its block (-1: padding)
    int *bnl = nullptr;        // [nslice] levels inside each block
    int kmax = 0;              // most entries of any lane
};

// SGS / ILU0 on a 5- / 7-point natural-order grid: the sweeps by pencils of
// 64 lines along x (hfh_pencil.hip).
struct hfh_pencil {
    int np = 0;                // pencils (0: none)
    int nx = 0, ny = 0, nz = 0, npy = 0, npz = 0;
    int ng = 0;                // groups of 4 steps of a pencil
    int *order = nullptr;      // device: pencils in dependency order
    void *fval = nullptr, *bval = nullptr;   // forward / backward values by (pencil, step, lane)
    void *y = nullptr;         // forward results by (pencil, step, lane)
    void *fbox = nullptr, *bbox = nullptr;   // face values received by each pencil
    int *ctl = nullptr;        // tickets, slow-division flag
};

struct hfh_prec {
    int kind = HFH_PREC_NONE;
    hfh_ctx *ctx = nullptr;
    const hfh_csr *A = nullptr;     // operator (SGS, MC-SGS) or LU factors (ILU0)
    int n = 0;
    int dtype = HFH_F64;
    void *invd = nullptr;           // Jacobi / MC-SGS: 1/a_ii
    void *dv = nullptr;             // MC-SGS: -a_ii / (omega (2 - omega))
    void *sval = nullptr;           // MC-SGS: omega-scaled values (nullptr when omega == 1)
    double omega = 1.0;
    int ncolors = 0;
    std::vector<int> color_off;     // host, ncolors+1
    hfh_levels lo, up;              // SGS / ILU0 level schedules
    hfh_sweep fw, bw;               // MC-SGS: lower-colour / upper-colour entries per row
    hfh_tsweep tlo, tup;            // SGS / ILU0: forward / backward sweep rows by level
    hfh_tsweep blo, bup;            // SGS / ILU0 on a structured grid: the sweeps by geometric block
    hfh_pencil pen;                 // SGS / ILU0 on a 5- / 7-point grid: by pencils instead of blocks
    unsigned tversion = 0;          // A->version the sweep values were copied at
    // SGS / ILU0 outside the fused drivers: both sweeps captured once as a
    // hipGraph on internal in/out buffers (one launch instead of one per level)
    void *gin = nullptr, *gout = nullptr;
    hipGraph_t sweep_graph = nullptr;
    hipGraphExec_t sweep_exec = nullptr;
    bool graph_failed = false;
    // SGS / ILU0 sweep schedule: sync-free (one launch per sweep) or one
    // launch per level; the sync-free form keeps the forward results in sf_y
    // and its ticket counters and failure word in sf_ctl
    int sweep_mode = HFH_SWEEP_SYNCFREE;
    int sf_waves = 0;                  // sync-free: waves per CU (0: from the level widths)
    void *sf_y = nullptr;
    int *sf_ctl = nullptr;
};

namespace hfh {

inline int hip_fail(hipError_t e, const char *what) {
    set_error("%s: %s", what, hipGetErrorString(e));
    return HFH_ERR_HIP;
}

#define HFH_HIP(call)                                          \
    do {                                                       \
        hipError_t e_ = (call);                                \
        if (e_ != hipSuccess) return hfh::hip_fail(e_, #call); \
    } while (0)

#define HFH_CHECK(cond, code, ...)           \
    do {                                     \
        if (!(cond)) {                       \
            hfh::set_error(__VA_ARGS__);     \
            return (code);                   \
        }                                    \
    } while (0)

int dev_alloc(void **p, size_t bytes);
// For copies of a matrix that only make it faster: HFH_ERR_NOMEM (also above
// the context's limit) means that the caller does without.
int copy_alloc(hfh_ctx *c, void **p, size_t bytes);
int launch_check(const char *what);
// False when the environment sets HFH_GRAPHS=0: the drivers and the serving
// engine then launch every iteration directly instead of replaying a
// captured graph (the same kernels in the same order, the same results).
bool graphs_enabled();
// Device address of the static scratch array on `device` (current), looked
// up once per device (hfh_krylov.hip).
int static_scratch(int device, void **ptr);
// HFH_ERR_HIP (and the failure word cleared) when a sync-free sweep of P gave
// up waiting since the last check; HFH_OK otherwise (also for P = NULL).
int sweep_failed(hfh_prec *P);

// Reductions (hfh_blas1.hip).  Results land in ctx->red + slot (device).
int dot_async(hfh_ctx *ctx, int dtype, int n, const void *x, const void *y, double *dst);
int fetch(hfh_ctx *ctx, const double *dsrc, double *host, int count);
// Sums the first nb single-quantity partials of ctx->red into dst (device) in
// fixed order (one finisher workgroup).
int partials_sum(hfh_ctx *ctx, int nb, double *dst);

// Timing helpers.
struct ScopedKernelTimer {
    hfh_ctx *ctx;
    int kclass;
    bool on;
    ScopedKernelTimer(hfh_ctx *c, int k);
    ~ScopedKernelTimer();
};

// SpMV launch used by the drivers (hfh_spmv.hip).  mode 0: y = A x;
// mode 1: y += A x.  When w is non-null each workgroup also stores its
// partial sum of y_i * w_i at part[row block] (A->nrblk partials), to be
// summed by a finisher kernel (A->nwg partials).
int spmv_launch(const hfh_csr *A, const void *x, void *y, int mode);
int spmv_configure(hfh_csr *A, int algo, int p1, int p2);
int spmv_sell_fill(hfh_csr *A, bool search = true);
// After the device columns changed order: diagonal positions, SpMV layout
// and SELL copy rebuilt from the CSR arrays (host copies already updated).
int spmv_refresh_structure(hfh_csr *A);
int spmv_launch_ex(const hfh_csr *A, const void *x, void *y, int mode, const void *w, double *part,
                   const int *done);
// SpMV by (offset, value) pairs (hfh_pattern.hip): pattern_fill looks at the
// structure and the values (A->pt_pairs 0 where they do not qualify; waits
// for the stream), pattern_scale follows a scaling of the values (the pairs
// found stay the pairs, none found stays none: no search), pattern_free forgets them, pattern_spmv launches (as
// spmv_launch_ex, A->nwg workgroups and partials of the same rows as the SELL
// kernels).
int pattern_fill(hfh_csr *A);
void pattern_scale(hfh_csr *A, double alpha, bool offdiag_only);
void pattern_free(hfh_csr *A);
int pattern_spmv(const hfh_csr *A, const void *x, void *y, int mode, const void *w, double *part, const int *done);
// One Jacobi step xn = update(b - sum_{j != r} a_rj x_j) over the LDS-staged
// or the dictionary-coded SELL copy (A->spmv_algo HFH_SPMV_SELL_LDS or
// HFH_SPMV_SELL_DICT); T is A's value type.
template <typename T>
int spmv_coded_jacobi(const hfh_csr *A, const T *x, T *xn, const T *b, bool damped, T w, T omw);

// Preconditioner apply on raw device pointers (hfh_prec.hip).  `done`
// (device, nullable): every kernel returns at once when *done != 0.
// mc_first_done: for a multicolour SGS of two or more colours, the first
// forward step (colour 0) is already in `out` (the CG update computes it).
// rzp / rz_out (multicolour SGS only): the apply also forms in.out (r.z of a
// CG step) through partials in rzp (mcsgs_rz_slots(P) doubles) into *rz_out.
int prec_apply_raw(hfh_prec *P, const void *in, void *out, const int *done = nullptr, bool mc_first_done = false,
                   double *rzp = nullptr, double *rz_out = nullptr);
int mcsgs_rz_slots(const hfh_prec *P);
// Brings a preconditioner's copies of the matrix values up to date (after the
// matrix's values changed); a no-op while the stream is being captured.
int prec_sync(hfh_prec *P);

// Loads the one-launch CG's code (2 MB of device memory), so that the first
// allocation-free solve does not.
int resident_load();
// CG of a small enough system in one launch (hfh_cgres.hip): x is the initial
// guess and the result; z0, z1, slots and keep (n elements each) are work
// space.  *ran false: the system does not qualify, or a wait gave up; x is the
// initial guess as before.  noalloc: nothing is allocated, by the runtime
// neither.
constexpr int kResidentRows = 4 * 512 * 256;
constexpr long long kResidentLds = 158 * 1024;
template <typename T>
int cg_resident(const hfh_csr *A, const T *invd, const T *b, T *x, T *z0, T *z1, void *slots, T *keep,
                double *hist, const hfh_control &ctl, bool noalloc, hfh_solve_info *info, bool *ran);

// SGS / ILU0 sweeps by pencils (hfh_pencil.hip).  pencil_build leaves P->pen
// empty where the pattern is not a full 5- / 7-point stencil of the grid
// (nx, and nxy in 3D, else 0); pencil_fill copies the matrix's values;
// pencil_apply runs both sweeps (in and out natural order, not aliased).
int pencil_build(hfh_prec *P, int nx, long long nxy);
int pencil_fill(hfh_prec *P);
void pencil_free(hfh_pencil &G);
int pencil_apply(hfh_prec *P, const void *in, void *out, const int *done);

// XCD-aware workgroup remap: consecutive logical tiles land on one XCD so its
// L2 keeps the shared gather window.
__device__ __forceinline__ int xcd_remap(int b, int nb) {
    const int per = nb / kNumXcd, rem = nb % kNumXcd;
    const int xcd = b % kNumXcd, idx = b / kNumXcd;
    // XCDs [0, rem) own per+1 tiles, the rest own per tiles
    const int base = xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per;
    return base + idx;
}

// 16-byte vectors of a stream: 2 doubles or 4 floats.
template <typename T> struct V16;
template <> struct V16<double> {
    typedef double type __attribute__((ext_vector_type(2)));
    static constexpr int W = 2;
};
template <> struct V16<float> {
    typedef float type __attribute__((ext_vector_type(4)));
    static constexpr int W = 4;
};

// Separately rounded product and sum.  The contraction pragma sits inside
// the helpers so that it also holds where they are inlined into code
// compiled with contraction on.
template <typename T>
__device__ __forceinline__ T mul_rn(T a, T b) {
#pragma clang fp contract(off)
    return a * b;
}
template <typename T>
__device__ __forceinline__ T add_rn(T a, T b) {
#pragma clang fp contract(off)
    return a + b;
}

// 1 / d, rounded once (the diagonal's inverse, extract_invdiagelements).
template <typename T>
__device__ __forceinline__ T inverse(T d) {
    return static_cast<T>(1) / d;
}

// Jacobi step epilogue for row r given s = sum_{j != r} a_rj x_j
// (DoNormalIteration / DoDampedIteration, linear_solver/jacobi.cc):
// y = (b_r - s) * inv_diag_r; damped: (1 - w) x_r + w y, each step rounded.
template <typename T, bool DAMPED>
__device__ __forceinline__ T jacobi_update(T s, T xr, T br, T dr, T w, T omw) {
    const T y = mul_rn(add_rn(br, -s), dr);
    if (!DAMPED) return y;
    return add_rn(mul_rn(xr, omw), mul_rn(w, y));
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// A 32-bit value moved between lanes by a DPP control (0 where the source
// lane does not exist or the row is masked out).
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_move(double v) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = __builtin_amdgcn_update_dpp(0u, static_cast<unsigned>(u), CTRL, ROWS, 0xf, false);
    const unsigned hi = __builtin_amdgcn_update_dpp(0u, static_cast<unsigned>(u >> 32), CTRL, ROWS, 0xf, false);
    return __builtin_bit_cast(double, static_cast<unsigned long long>(hi) << 32 | lo);
}

// Sum over the wave, the same value in every lane: rows of 16 lanes by shifts,
// then the rows by broadcasts, with vector moves instead of the LDS unit's
// permutes (a dependent chain of six of those takes about 0.3 us).  Another
// order of adds than wave_sum.
__device__ __forceinline__ double wave_sum_dpp(double v) {
    v += dpp_move<0x111, 0xf>(v);   // row_shr:1
    v += dpp_move<0x112, 0xf>(v);   // row_shr:2
    v += dpp_move<0x114, 0xf>(v);   // row_shr:4
    v += dpp_move<0x118, 0xf>(v);   // row_shr:8
    v += dpp_move<0x142, 0xa>(v);   // row_bcast:15 into rows 1 and 3
    v += dpp_move<0x143, 0xc>(v);   // row_bcast:31 into rows 2 and 3
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = __builtin_amdgcn_readlane(static_cast<unsigned>(u), 63);
    const unsigned hi = __builtin_amdgcn_readlane(static_cast<unsigned>(u >> 32), 63);
    return __builtin_bit_cast(double, static_cast<unsigned long long>(hi) << 32 | lo);
}

__device__ __forceinline__ int wave_max(int v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = max(v, __shfl_xor(v, off, 64));
    return v;
}

// Deterministic block sum of kBlock threads; result valid in thread 0.
template <typename T>
__device__ __forceinline__ T block_sum(T v, T *sh /* >= kBlock/64 */) {
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) sh[w] = v;
    __syncthreads();
    T s = 0;
    if (threadIdx.x == 0)
        for (int i = 0; i < kBlock / 64; ++i) s += sh[i];
    return s;
}

// Cross-workgroup reductions never synchronise inside a kernel: on gfx950
// an agent-scope release fence writes back the XCD's L2, so a per-workgroup
// fence + atomic costs far more than the reduction itself.  Each workgroup
// stores its partial sums with plain stores; a finisher kernel launched
// next on the same stream (the kernel boundary makes the partials visible)
// sums them in a fixed order, so results are bit-reproducible.
template <int NQ>
__device__ __forceinline__ void store_partials(const double (&v)[NQ], double *part, int stride, int slot) {
    if (threadIdx.x == 0) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) part[q * stride + slot] = v[q];
    }
}

constexpr int kFinBlock = 1024;  // threads of a finisher workgroup

// Sums part[q*stride + b], b < nb, with one workgroup of kFinBlock threads:
// lane-strided sums in ascending b, then a fixed tree.  Valid in thread 0.
template <int NQ>
__device__ __forceinline__ void reduce_partials(const double *part, int stride, int nb, double (&out)[NQ]) {
    __shared__ double sh[kFinBlock / 64];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        double s = 0;
        // unrolled so that the loads issue together; the adds keep their order
#pragma unroll 8
        for (int b = threadIdx.x; b < nb; b += kFinBlock) s += part[q * stride + b];
        s = wave_sum(s);
        const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
        if (lane == 0) sh[w] = s;
        __syncthreads();
        double t = 0;
        if (threadIdx.x == 0)
            for (int i = 0; i < kFinBlock / 64; ++i) t += sh[i];
        out[q] = t;
        __syncthreads();
    }
}

// The sum reduce_partials<1> returns, computed by a kBlock-thread workgroup
// (every workgroup of a kernel that needs it, in place of a finisher
// launch).  Thread t stands in for the finisher's threads t + kBlock k,
// k < kFinBlock / kBlock: those sit in lane t mod 64 of the finisher's waves
// t / 64 + (kBlock / 64) k, so each stand-in's strided sum and wave tree are
// the finisher's own and the wave totals meet in the same order: the result
// has the finisher's bits.  Valid in every thread.
__device__ __forceinline__ double fin_sum_all(const double *__restrict__ part, int nb,
                                              double *sh /* kFinBlock/64 */, double *bc) {
    constexpr int K = kFinBlock / kBlock;
    double s[K];
#pragma unroll
    for (int k = 0; k < K; ++k) s[k] = 0;
    for (int b0 = 0; b0 < nb; b0 += kFinBlock) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int b = b0 + static_cast<int>(threadIdx.x) + kBlock * k;
            if (b < nb) s[k] += part[b];
        }
    }
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const double t = wave_sum(s[k]);
        if (lane == 0) sh[w + (kBlock / 64) * k] = t;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0;
        for (int i = 0; i < kFinBlock / 64; ++i) t += sh[i];
        *bc = t;
    }
    __syncthreads();
    const double v = *bc;
    __syncthreads();
    return v;
}

}  // namespace hfh

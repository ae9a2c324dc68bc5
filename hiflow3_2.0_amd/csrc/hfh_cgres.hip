// hfh_cgres.hip -- CG of systems that fit on the chip, in one launch.
//
// The launched CG (hfh_krylov.hip) pays three dependent launches per step,
// about 13 us on anything up to a few hundred thousand rows, while the work
// of such a step is one or two microseconds.  Here every row's matrix values
// stay in registers for the whole solve, r, x and the diagonal beside them,
// and the window of p that a workgroup's rows gather from (its rows and the
// bandwidth on both sides) in LDS; a step moves only the z of the window's
// far rows and two sums across the workgroups.
//
//   A  Ap = A p from LDS; sum of p.Ap over the grid; alpha
//   B  x += alpha p, r -= alpha Ap, z = M r stored for the neighbours; sums
//      of r.r and r.z over the grid; IterateControl on sqrt(r.r); then
//      p = z + ratio p over the whole window, each workgroup forming its
//      neighbours' rows itself from their z (the same bits they hold)
//
// Nothing is fenced.  Every value that crosses the grid is its own flag: it
// is stored and polled with agent-scope relaxed atomics over a signalling-NaN
// sentinel, which arithmetic never yields.  z alternates between two buffers
// and the sums over four rows of slots.  A workgroup returns its own entries
// of a buffer to the sentinel when a later sum shows that everybody has read
// them, and publishes its next A sum only when those stores have completed,
// so nobody can poll the buffer again before.  Every wait is bounded: where
// other work holds compute units for longer than that, so that some of the
// workgroups cannot start, the launch ends with the failure word raised, the
// initial guess (kept beside the solve) is put back and the launched form
// solves the system.
//
// The step's arithmetic is the launched form's (cg.cc:163-248): row sums in
// stored order with separate products and sums, FP64 sums over the rows in a
// fixed order.
//
// Measured per step (Jacobi, FP64; launched -> resident): 1,517 rows (2D FV,
// one workgroup) 13.8 -> 2.5 us, 8,000 rows (3D Q1) 22.6 -> 6.6, 65,025 rows
// (2D Q1) 14.8 -> 4.7 to 5.6 from process to process, 125,000 rows (3D Q1)
// 22.8 -> 9.3, 250,047 rows (3D FV) 19.3 -> 11.3, 490,000 rows (2D Q1) 30.4 ->
// 8.0.  The largest form (3D Q1, two rows of 27 entries per thread) takes
// 10.8 us at 175,616 rows and 13.0 at 250,047; with its codes unpacked once and
// 86 registers spilled 12.3 and 16.8.  What remains is the two sums (1.8 us each
// on 128 workgroups) and the far z.
#include "hfh_internal.h"

#include <algorithm>

namespace hfh {

namespace {

constexpr int kResBlock = 512;      // threads of a workgroup (one per CU)
constexpr int kResWaves = kResBlock / 64;
constexpr int kResRows = 4;         // slot rows of the sums
constexpr int kCopies = 16;         // copies of each workgroup's sums
constexpr int kResPolls = 1 << 16;   // of one wait: some tens of ms
constexpr int kPre = 4;             // far z per thread received while the B sum is under way
constexpr int kMaxGroups = 256;
constexpr unsigned long long kResSentinel = 0x7FF4DEAD5EEDBEEFull;   // exponent all ones, quiet bit clear

template <typename T> struct Flag;
template <> struct Flag<double> {
    typedef unsigned long long U;
    static constexpr U sentinel = kResSentinel;
};
template <> struct Flag<float> {
    typedef unsigned U;
    static constexpr U sentinel = 0x7FA5EED5u;
};

template <typename U>
__device__ __forceinline__ U far_load(const U *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename U>
__device__ __forceinline__ void far_store(U *p, U v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// polls p until it holds something else than the sentinel; a thread that has
// given up once waits no more
template <typename U>
__device__ __forceinline__ U far_wait(const U *p, U u, U sentinel, int &polls, int *s_fail) {
    for (int k = 0; u == sentinel; u = far_load(p))
        if (++k >= polls) {
            *s_fail = 1;
            polls = 1;
            break;
        }
    return u;
}

__device__ __forceinline__ double fma_t(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fma_t(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

}  // namespace

template <typename T>
struct ResidentArgs {
    int n, lo, hi;            // rows; columns reach lo below and hi above the row
    const int *row, *col;
    const T *val;
    const T *b, *invd;        // invd: Jacobi, or null
    T *x;
    T *z[2];
    unsigned long long *slots;   // [kResRows][kCopies][2][G]
    double *hist;             // residuals, maxits + 1, or null
    double *out;              // pinned: iterations, state, residual, first residual, failure
    double atol, rtol, dtol;
    int maxits;
    int polls;                // of one wait
};

// Sums of NQ values over the grid, the same bits in every thread: wave
// trees, the waves in order, then (several workgroups) the workgroups' sums
// polled by the first threads and summed the same way.  Each workgroup stores
// its sums in kCopies copies and polls one of them: with one copy for all,
// the polls of the same lines queue up (128 workgroups: 2.7 us a sum, 1.8 us
// with 16 copies; 256: 2.9 and 2.3).  seq counts the sums; `between` runs
// after the workgroup's sums are out.
template <int NQ, typename F>
__device__ __forceinline__ void grid_sum(double (&v)[NQ], int seq, unsigned long long *slots, double *sh, int &polls,
                                         int *s_fail, F between) {
    const int G = gridDim.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    double *s1 = sh + (seq & 1) * 4 * kResWaves, *s2 = s1 + 2 * kResWaves;
    static_assert(kResWaves == 8, "the sum of the waves");
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        v[q] = wave_sum_dpp(v[q]);
        if (lane == 0) s1[q * kResWaves + w] = v[q];
    }
    __syncthreads();
    auto waves = [](const double *s) { return ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7])); };
    if (G == 1) {
        between();
#pragma unroll
        for (int q = 0; q < NQ; ++q) v[q] = waves(s1 + q * kResWaves);
        return;
    }
    const size_t part = static_cast<size_t>(2) * G;    // a copy of a slot row
    unsigned long long *row = slots + static_cast<size_t>(seq & (kResRows - 1)) * kCopies * part;
    if (tid < NQ * kCopies) {
        const int q = tid / kCopies;
        far_store(row + (tid % kCopies) * part + q * G + blockIdx.x,
                  __builtin_bit_cast(unsigned long long, waves(s1 + q * kResWaves)));
    }
    between();
    const unsigned long long *mine = row + (blockIdx.x % kCopies) * part;
    if (w * 64 < G) {
        unsigned long long u[NQ];
#pragma unroll
        for (int q = 0; q < NQ; ++q) u[q] = tid < G ? far_load(mine + q * G + tid) : 0;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            if (tid < G) u[q] = far_wait(mine + q * G + tid, u[q], kResSentinel, polls, s_fail);
            const double t = wave_sum_dpp(__builtin_bit_cast(double, u[q]));
            if (lane == 0) s2[q * kResWaves + w] = t;
        }
    }
    __syncthreads();
    // everybody has published this sum, hence read the previous one
    if (tid < 2 * kCopies)
        far_store(slots + (static_cast<size_t>((seq - 1) & (kResRows - 1)) * kCopies + tid % kCopies) * part +
                      tid / kCopies * G + blockIdx.x,
                  kResSentinel);
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        double s = s2[q * kResWaves];
        for (int k = 1; k < (G + 63) / 64; ++k) s += s2[q * kResWaves + k];
        v[q] = s;
    }
}

// L bounds the entries of a row, E the rows of a thread.
template <typename T, int L, int E>
__global__ __launch_bounds__(kResBlock) void k_cg_resident(ResidentArgs<T> a) {
    typedef typename Flag<T>::U U;
    constexpr U kS = Flag<T>::sentinel;
    extern __shared__ __align__(16) unsigned char lds[];
    T *const pw = reinterpret_cast<T *>(lds);     // p over the window, then a zero
    __shared__ double sh[8 * kResWaves];
    // waits given up in a sum / for a far z; each is read only where no thread
    // can be setting it, so every thread takes the same branch
    __shared__ int s_fail, s_far;
    const int tid = threadIdx.x, G = gridDim.x, R = kResBlock * E;
    const int r0 = blockIdx.x * R, r1 = min(a.n, r0 + R);
    const int w0 = max(0, r0 - a.lo), w1 = r1 > a.n - a.hi ? a.n : r1 + a.hi;
    const int wlen = w1 - w0, own0 = r0 - w0, nown = r1 - r0, nfar = wlen - nown;
    auto far_pos = [&](int h) { return h < own0 ? h : h + nown; };
    // The largest form's values and codes leave few registers, and its first
    // launch must not make the runtime reserve scratch.  It unpacks its codes
    // anew in every step (`step` hides that they never change; the compiler
    // kept all unpacked codes too and spilled 86 registers) and reads the rows
    // once more for the first residual.
    constexpr bool kFew = sizeof(T) * L * E > 256;
    T v[E][L], xr[E], r[E], z[E], d[E], Ap[E];
    unsigned code[E][(L + 1) / 2];
    bool in[E];
    if (tid == 0) s_fail = s_far = 0;
    for (int k = tid; k < wlen; k += kResBlock) pw[k] = a.x[w0 + k];
    if (tid == 0) pw[wlen] = T(0);
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int i = r0 + e * kResBlock + tid;
        in[e] = i < r1;
        const int j0 = in[e] ? a.row[i] : 0, len = in[e] ? a.row[i + 1] - j0 : 0;
        d[e] = in[e] && a.invd ? a.invd[i] : T(1);
#pragma unroll
        for (int k = 0; k < L; ++k) {
            v[e][k] = k < len ? a.val[j0 + k] : T(0);
            const unsigned c = k < len ? static_cast<unsigned>(a.col[j0 + k] - w0) : static_cast<unsigned>(wlen);
            if (k & 1) code[e][k >> 1] |= c << 16;
            else code[e][k >> 1] = c;
        }
    }
    __syncthreads();
    auto spmv = [&](int step) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
            T s = T(0);
#pragma unroll
            for (int k = 0; k < L; k += 2) {
                unsigned c = code[e][k >> 1];
                if (kFew) asm("" : "+v"(c) : "v"(step));
                s = add_rn(s, mul_rn(v[e][k], pw[c & 0xffffu]));
                if (k + 1 < L) s = add_rn(s, mul_rn(v[e][k + 1], pw[c >> 16]));
            }
            Ap[e] = s;
        }
    };
    // step 0: r = b - A x
    if (kFew) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int i = r0 + e * kResBlock + tid, j0 = in[e] ? a.row[i] : 0, j1 = in[e] ? a.row[i + 1] : 0;
            T s = T(0);
#pragma unroll 4
            for (int j = j0; j < j1; ++j) s = add_rn(s, mul_rn(a.val[j], pw[a.col[j] - w0]));
            Ap[e] = s;
        }
    } else {
        spmv(0);
    }
    double s[2] = {0, 0};
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int i = r0 + e * kResBlock + tid;
        xr[e] = in[e] ? pw[own0 + e * kResBlock + tid] : T(0);
        r[e] = in[e] ? add_rn(mul_rn(static_cast<T>(-1), Ap[e]), a.b[i]) : T(0);
    }
    int seq = 1, it = 0, state = HFH_ITERATE;
    T beta = T(1);
    double res = 0, res0 = 0;
    int polls = a.polls;
    bool failed = false;
    U zf[kPre];
    for (;;) {
        // ---- B: z, the sums of r.r and r.z, the test, the new direction
        T *const zb = a.z[it & 1];
        s[0] = s[1] = 0;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            z[e] = a.invd ? r[e] * d[e] : r[e];
            if (in[e]) {
                if (G > 1) far_store(reinterpret_cast<U *>(zb) + r0 + e * kResBlock + tid, __builtin_bit_cast(U, z[e]));
                s[0] += static_cast<double>(r[e]) * static_cast<double>(r[e]);
                s[1] += static_cast<double>(r[e]) * static_cast<double>(z[e]);
            }
        }
        grid_sum<2>(s, seq++, a.slots, sh, polls, &s_fail, [&]() {
#pragma unroll
            for (int q = 0; q < kPre; ++q) {
                const int h = tid + q * kResBlock;
                zf[q] = h < nfar ? far_load(reinterpret_cast<const U *>(zb) + w0 + far_pos(h)) : U(0);
            }
#pragma unroll
            for (int q = 0; q < kPre; ++q) {
                const int h = tid + q * kResBlock;
                if (h < nfar) zf[q] = far_wait(reinterpret_cast<const U *>(zb) + w0 + far_pos(h), zf[q], kS, polls, &s_far);
            }
        });
        const T rrT = static_cast<T>(s[0]);
        res = static_cast<double>(static_cast<T>(sqrt(static_cast<double>(rrT))));
        if (it == 0) res0 = res;
        if (a.hist && blockIdx.x == 0 && tid == 0) a.hist[it] = res;
        if (res < a.atol) state = HFH_SUCCESS_ABS;
        else if (res < a.rtol * res0) state = HFH_SUCCESS_REL;
        else if (res > a.dtol * res0) state = HFH_FAIL_DIV;
        else if (it >= a.maxits) state = HFH_FAIL_MAXITS;
        const T gamma = a.invd ? static_cast<T>(s[1]) : rrT;
        const T ratio = gamma / beta;   // (unused at step 0)
        failed = s_fail != 0;
        if (state != HFH_ITERATE || failed) break;
        beta = gamma;
        auto turn = [&](int pos, T zj) {
            pw[pos] = it == 0 ? zj : fma_t(ratio, pw[pos], zj);
        };
#pragma unroll
        for (int e = 0; e < E; ++e)
            if (in[e]) turn(own0 + e * kResBlock + tid, z[e]);
#pragma unroll
        for (int q = 0; q < kPre; ++q) {
            const int h = tid + q * kResBlock;
            if (h < nfar) turn(far_pos(h), __builtin_bit_cast(T, zf[q]));
        }
        for (int h0 = tid + kPre * kResBlock; h0 < nfar; h0 += kPre * kResBlock) {
            U u[kPre];
#pragma unroll
            for (int q = 0; q < kPre; ++q) {
                const int h = h0 + q * kResBlock;
                u[q] = h < nfar ? far_load(reinterpret_cast<const U *>(zb) + w0 + far_pos(h)) : U(0);
            }
#pragma unroll
            for (int q = 0; q < kPre; ++q) {
                const int h = h0 + q * kResBlock;
                if (h < nfar) {
                    const int pos = far_pos(h);
                    turn(pos, __builtin_bit_cast(T, far_wait(reinterpret_cast<const U *>(zb) + w0 + pos, u[q], kS, polls, &s_far)));
                }
            }
        }
        __syncthreads();
        // ---- A: Ap, the sum of p.Ap, alpha
        ++it;
        spmv(it);
        double t[1] = {0};
#pragma unroll
        for (int e = 0; e < E; ++e)
            if (in[e]) t[0] += static_cast<double>(Ap[e]) * static_cast<double>(pw[own0 + e * kResBlock + tid]);
        // this thread's returns to the sentinel have completed before its
        // workgroup's sum is published (the barrier in grid_sum)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        grid_sum<1>(t, seq++, a.slots, sh, polls, &s_fail, []() {});
        // everybody has formed its p of this step: the z of the last one is read
        if (G > 1) {
            U *const zo = reinterpret_cast<U *>(a.z[(it - 1) & 1]);
#pragma unroll
            for (int e = 0; e < E; ++e)
                if (in[e]) far_store(zo + r0 + e * kResBlock + tid, kS);
        }
        const T alpha = static_cast<T>(beta / static_cast<T>(t[0]));
#pragma unroll
        for (int e = 0; e < E; ++e)
            if (in[e]) {
                xr[e] = fma_t(alpha, pw[own0 + e * kResBlock + tid], xr[e]);
                r[e] = fma_t(-alpha, Ap[e], r[e]);
            }
        failed = s_fail != 0 || s_far != 0;
        if (failed) break;
    }
    if (failed) {
        // vector store of system scope: the host reads it after the launch
        if (tid == 0) __hip_atomic_store(a.out + 4, 1.0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        return;
    }
#pragma unroll
    for (int e = 0; e < E; ++e)
        if (in[e]) a.x[r0 + e * kResBlock + tid] = xr[e];
    if (blockIdx.x == 0 && tid == 0) {
        a.out[0] = it;
        a.out[1] = state;
        a.out[2] = res;
        a.out[3] = res0;
    }
}

// Everything that is polled to the sentinel, and the initial guess kept.
template <typename T, typename U>
__global__ __launch_bounds__(kBlock) void k_resident_fill(int n, U *z0, U *z1, U v, int ns, unsigned long long *slots,
                                                          const T *x, T *keep) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) {
        z0[i] = v;
        z1[i] = v;
        keep[i] = x[i];
    }
    if (i < ns) slots[i] = kResSentinel;
}

// Rows per thread for a system of n rows, 0 where it does not fit the
// registers of all CUs (the launched form then streams it; at the largest
// fitting sizes it takes 1.5 to 3 times as long).  One workgroup, with no sum
// across the grid, is kept up to four rows per thread (1,517 rows: 2.5 us a
// step; five workgroups on 2,500 rows: 4.3); otherwise as few rows per thread
// as the CUs allow.
// The slots fit n elements: 1024 G bytes, and n > 512 (G - 1) rows of at
// least 4 bytes.
static_assert(kResRows * kCopies * 2 * sizeof(unsigned long long) <= 1024 && kResBlock * 4 >= 2048, "slots in n elements");
static int resident_rows(const hfh_ctx *c, int n, int L) {
    const int emax = L <= 9 ? 4 : 2;
    if (n <= kResBlock * emax) return n <= kResBlock ? 1 : n <= 2 * kResBlock ? 2 : 4;
    const int ncu = std::min(std::max(c->num_cu, 1), kMaxGroups);
    for (int e = 1; e <= emax; e *= 2)
        if ((n + kResBlock * e - 1) / (kResBlock * e) <= ncu) return e;
    return 0;
}

// The most far rows of a window.  A workgroup receives their z in rounds of
// kPre 512, about 0.3 us per 500 of them, which in the end takes longer than
// the launched step's three launches (FP32, us per step, one launch /
// launched; FP64 windows end before, at the LDS's size):
//   100,000 rows of 5   far 20,000 11.5 / 12.2, 25,000 13.3 / 12.1, 39,000 17.6 / 12.1
//   260,000 rows of 5   far 20,000 13.5 / 14.1, 22,000 14.1 / 13.9, 39,000 19.1 / 13.9
//   130,000 rows of 15  far 22,000 12.7 / 13.5, 25,000 13.5 / 13.1
//   500,000 rows of 5   far 25,000 17.4 / 18.2, 28,000 18.2 / 18.5, 36,000 20.8 / 18.8
//   500,000 rows of 9   far 32,000 20.1 / 22.0, 36,000 21.4 / 21.2
//   100,000 rows of 27  far 39,000 17.5 / 18.9; 260,000 rows 19.6 / 26.8
static int resident_far(int E, int L) {
    return L > 16 ? 65536 : E < 4 ? 21000 : L <= 5 ? 28000 : 34000;
}

template <typename T, int L, int E>
static int resident_launch(const hfh_csr *A, ResidentArgs<T> &a, T *keep, bool noalloc, bool &ran) {
    hfh_ctx *c = A->ctx;
    const int R = kResBlock * E, G = (a.n + R - 1) / R;
    const size_t shm = sizeof(T) * (static_cast<size_t>(std::min(R + a.lo + a.hi, a.n)) + 1);
    const void *f = reinterpret_cast<const void *>(k_cg_resident<T, L, E>);
    if (shm > 64 * 1024 && hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(shm)) != hipSuccess) {
        (void)hipGetLastError();
        return HFH_OK;
    }
    hipStream_t s = c->stream;
    if (G > 1) {
        const int ns = kResRows * kCopies * 2 * G, m = std::max(a.n, ns);
        typedef typename Flag<T>::U U;
        hipLaunchKernelGGL((k_resident_fill<T, U>), dim3((m + kBlock - 1) / kBlock), dim3(kBlock), 0, s, a.n,
                           reinterpret_cast<U *>(a.z[0]), reinterpret_cast<U *>(a.z[1]), Flag<T>::sentinel, ns, a.slots,
                           (const T *)a.x, keep);
        if (int rc = launch_check("k_resident_fill")) return rc;
        void *args[] = {&a};
        // Cooperative launches of one process run one after the other, so two
        // solves never hold half of the compute units each.  The first one
        // makes the runtime allocate a queue (8 MB); where nothing may be
        // allocated a plain launch has the bounded waits to rely on.
        if (noalloc) {
            hipLaunchKernelGGL((k_cg_resident<T, L, E>), dim3(G), dim3(kResBlock), shm, s, a);
            if (int rc = launch_check("k_cg_resident")) return rc;
        } else if (hipLaunchCooperativeKernel(f, dim3(G), dim3(kResBlock), args, static_cast<unsigned>(shm), s) != hipSuccess) {
            (void)hipGetLastError();
            return HFH_OK;
        }
    } else {
        hipLaunchKernelGGL((k_cg_resident<T, L, E>), dim3(1), dim3(kResBlock), shm, s, a);
        if (int rc = launch_check("k_cg_resident")) return rc;
    }
    ran = true;
    return HFH_OK;
}

int resident_load() {
    hipFuncAttributes attr;
    HFH_HIP(hipFuncGetAttributes(&attr, reinterpret_cast<const void *>(k_cg_resident<double, 5, 1>)));
    return HFH_OK;
}

template <typename T>
int cg_resident(const hfh_csr *A, const T *invd, const T *b, T *x, T *z0, T *z1, void *slots, T *keep,
                double *hist, const hfh_control &ctl, bool noalloc, hfh_solve_info *info, bool *ran) {
    *ran = false;
    hfh_ctx *c = A->ctx;
    const int n = A->nrow, L = A->shape_len;
    if (c->timing.on || A->spmv_algo_req != 0 || !A->sorted || L <= 0 || L > 28) return HFH_OK;
    const int E = resident_rows(c, n, L);
    if (E == 0) return HFH_OK;
    const long long window = std::min<long long>(static_cast<long long>(kResBlock) * E + A->shape_lo + A->shape_hi, n) + 1;
    if (window * static_cast<long long>(sizeof(T)) > kResidentLds || window >= 65536) return HFH_OK;
    if (window - 1 - kResBlock * E > resident_far(E, L)) return HFH_OK;
    ResidentArgs<T> a{n, A->shape_lo, A->shape_hi, A->row, A->col, static_cast<const T *>(A->val), b, invd, x, {z0, z1},
                      reinterpret_cast<unsigned long long *>(slots), hist, c->host_res, ctl.atol, ctl.rtol, ctl.dtol,
                      ctl.maxits, c->wait_polls > 0 ? c->wait_polls : kResPolls};
    c->host_res[4] = 0;
    int rc;
#define HFH_RES(LL)                                                         \
    (E == 1 ? resident_launch<T, LL, 1>(A, a, keep, noalloc, *ran)                         \
            : E == 2 ? resident_launch<T, LL, 2>(A, a, keep, noalloc, *ran)                \
                     : resident_launch<T, LL, (LL <= 9 ? 4 : 2)>(A, a, keep, noalloc, *ran))
    if (L <= 5) rc = HFH_RES(5);
    else if (L <= 7) rc = HFH_RES(7);
    else if (L <= 9) rc = HFH_RES(9);
    else if (L <= 16) rc = HFH_RES(16);
    else rc = HFH_RES(28);
#undef HFH_RES
    if (rc || !*ran) return rc;
    HFH_HIP(hipStreamSynchronize(c->stream));
    if (c->host_res[4] != 0) {   // x may hold some workgroups' rows of the solution
        ++c->cg_gave_up;
        *ran = false;
        HFH_HIP(hipMemcpyAsync(x, keep, sizeof(T) * static_cast<size_t>(n), hipMemcpyDeviceToDevice, c->stream));
        return HFH_OK;
    }
    ++c->cg_resident;
    info->iters = static_cast<int>(c->host_res[0]);
    info->state = static_cast<int>(c->host_res[1]);
    info->res = c->host_res[2];
    info->res0 = c->host_res[3];
    return HFH_OK;
}

template int cg_resident<double>(const hfh_csr *, const double *, const double *, double *, double *, double *, void *,
                                 double *, double *, const hfh_control &, bool, hfh_solve_info *, bool *);
template int cg_resident<float>(const hfh_csr *, const float *, const float *, float *, float *, float *, void *,
                                float *, double *, const hfh_control &, bool, hfh_solve_info *, bool *);

}  // namespace hfh

// hfh_pattern.hip -- SpMV of matrices whose rows repeat a few (offset, value)
// pairs: constant-coefficient operators on a structured grid.
//
// Such a matrix is one short list of pairs (column offset col - row, value),
// ascending by offset, and for every row the set of pairs it holds: an
// interior row of the Q1 Laplacian holds all 27, a row beside the boundary
// leaves some out.  The SpMV then reads x, a 4-byte set per row (only in
// slices where some row leaves a pair out) and writes y; offsets and values
// are wave-uniform and come through scalar loads.  The general layouts stream
// 10 to 12 bytes per entry from HBM for the same result.
//
// Row sums are the CSR loop's: the row's own entries in ascending column
// order, products and sums rounded separately, entries that a row does not
// hold skipped (not added as zeros), so the results are bit-identical to the
// other layouts.
#include "hfh_internal.h"

#include <algorithm>
#include <cstring>

namespace hfh {
namespace {

constexpr int kMaxPairs = 32;      // bits of a row's set

// Pairs with neighbouring offsets share one load of x.
struct Group {
    int off;       // offset of the loaded entries: the middle pair of three, else the first
    int bit, n;    // pairs bit .. bit + n - 1, n = 1 .. 3
};

// Offsets of the pairs, ascending.
struct Offsets {
    int v[kMaxPairs];
};

// The lists as a kernel argument: with compile-time positions all of them
// come in a few wide scalar loads before the first load of x (read from
// memory one by one, each load of x waited for its group: 25.1 us).
template <typename T>
struct Lists {
    Group grp[kMaxPairs];
    T val[kMaxPairs];
};

// A row as the host sees it (pinned memory).
struct RowReport {
    int len;                       // entries, -1: no report
    int row;
    int off[kMaxPairs];
    unsigned long long val[kMaxPairs];   // the value's bits
};
constexpr int kProbes = 8;         // rows spread over the matrix, then the first and the last one
constexpr int kReports = 16;
static_assert(kProbes + 2 <= kReports && sizeof(RowReport) * kReports <= kReportBytes, "the context's pinned reports");

__device__ __forceinline__ unsigned long long bits_of(double a) { return __builtin_bit_cast(unsigned long long, a); }
__device__ __forceinline__ unsigned long long bits_of(float a) { return __builtin_bit_cast(unsigned, a); }

// One lane per entry (the lanes of a wave, of which the first kMaxPairs write).
template <typename T>
__device__ __forceinline__ void report_row(RowReport *out, int r, int j0, int len, int lane, const int *__restrict__ col,
                                           const T *__restrict__ val) {
    if (lane < min(len, kMaxPairs)) {
        out->off[lane] = col[j0 + lane] - r;
        out->val[lane] = bits_of(val[j0 + lane]);
    }
    if (lane == 0) {
        out->row = r;
        out->len = len;
    }
}

template <typename T>
__global__ __launch_bounds__(64) void k_pattern_probe(int nrow, const int *__restrict__ row, const int *__restrict__ col,
                                                      const T *__restrict__ val, RowReport *out, int *count, int rounds) {
    const int i = blockIdx.x;
    if (i == 0 && static_cast<int>(threadIdx.x) < rounds) count[threadIdx.x] = 0;
    const int r = i < kProbes ? static_cast<int>(static_cast<long long>(nrow) * (i + 1) / (kProbes + 1))
                              : i == kProbes ? 0 : nrow - 1;
    report_row(out + i, r, row[r], row[r + 1] - row[r], threadIdx.x, col, val);
}

// Every row's set of pairs and, per slice of 64 rows, whether some row lacks
// one; a row with an entry that is no pair is reported (one per slice, the
// first kReports of them), and the sets then mean nothing.
// One wave per slice, 64 / W rows at a time with W lanes each, so that the
// entries are read in memory order (a thread per row: 1,851 us on the 127^3
// Q1 Laplacian in FP64, 177 us this way).  Entry k of a complete row is
// pair k, so a row's set is mostly the lanes' ballot; the others search.  The
// offsets also go to memory, for the SpMV.
template <typename T, int W>
__global__ __launch_bounds__(kBlock) void k_pattern_sets(int nrow, int nslice, int npair, Lists<T> L, Offsets offs,
                                                         const int *__restrict__ row, const int *__restrict__ col,
                                                         const T *__restrict__ val, int *__restrict__ offs_out,
                                                         unsigned *__restrict__ set, int *__restrict__ partial,
                                                         int *count, RowReport *out) {
    __shared__ int s_off[kMaxPairs];
    __shared__ T s_val[kMaxPairs];
    __shared__ unsigned s_set[kBlock];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid < kMaxPairs) {
        s_off[tid] = tid < npair ? offs.v[tid] : 0x7fffffff;
        s_val[tid] = L.val[tid];
        if (blockIdx.x == 0) offs_out[tid] = s_off[tid];
    }
    s_set[tid] = 0;
    __syncthreads();
    const int s = blockIdx.x * (kBlock / 64) + wave;
    if (s >= nslice) return;
    unsigned *const sets = s_set + wave * 64;
    const int r0 = s * 64, rows = min(64, nrow - r0);
    const int rp = row[r0 + min(lane, rows)], re = row[r0 + rows];   // 65 row pointers of the slice
    const unsigned all = npair == 32 ? ~0u : (1u << npair) - 1;
    const int sub = lane / W, k0 = lane % W;
    int bad = -1;
#pragma unroll 4
    for (int q = 0; q < W; ++q) {
        const int i = q * (64 / W) + sub;          // this lane's row of the slice
        const int j0 = __shfl(rp, i, 64), up = __shfl(rp, min(i + 1, 63), 64);   // all lanes take part
        const int j1 = i == 63 ? re : up;
        const int len = i < rows ? j1 - j0 : 0;
        unsigned got = 0;
        bool wrong = len > kMaxPairs;
        for (int k = k0; __any(k - k0 < min(len, kMaxPairs)); k += W) {
            bool match = false;
            if (k < min(len, kMaxPairs)) {
                const int o = col[j0 + k] - (r0 + i);
                const unsigned long long v = bits_of(val[j0 + k]);
                match = s_off[k] == o && bits_of(s_val[k]) == v;
                if (!match) {
                    int p = 0;
                    for (int h = kMaxPairs / 2; h > 0; h >>= 1)
                        if (s_off[p + h - 1] < o) p += h;
                    while (p < npair && s_off[p] == o && bits_of(s_val[p]) != v) ++p;
                    if (p < npair && s_off[p] == o) got |= 1u << p;
                    else wrong = true;
                }
            }
            const unsigned long long m = __builtin_amdgcn_ballot_w64(match);
            const unsigned part = static_cast<unsigned>(m >> (sub * W)) & (W == 32 ? ~0u : (1u << (W & 31)) - 1);
            if (k0 == 0) got |= part << (k - k0);
        }
        if (got) atomicOr(&sets[i], got);
        const unsigned long long w = __builtin_amdgcn_ballot_w64(wrong);
        if (w && bad < 0) bad = q * (64 / W) + static_cast<int>(__builtin_ctzll(w)) / W;
    }
    if (bad >= 0) {
        int at = 0;
        if (lane == 0) {   // a look first: thousands of slices' additions would queue up
            at = __hip_atomic_load(count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (at < kReports) at = atomicAdd(count, 1);
        }
        at = __builtin_amdgcn_readfirstlane(at);
        const int j0 = __shfl(rp, bad, 64), up = __shfl(rp, min(bad + 1, 63), 64);
        const int j1 = bad == 63 ? re : up;
        if (at < kReports) report_row(out + at, r0 + bad, j0, j1 - j0, lane, col, val);
    }
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");   // a wave's LDS accesses execute in order
    const unsigned m = sets[lane];
    if (lane < rows) set[r0 + lane] = m;
    const bool some = __any(lane < rows && m != all);
    if (lane == 0) partial[s] = some ? 1 : 0;
}

// One wave per slice of 64 rows, lane = row.  The loads of U groups of a
// slice go out together, each one 64 consecutive entries of x at a scalar
// address, and one more load brings the entries past both ends of the groups'
// windows; a group's other pairs read their neighbours' entries through a
// window in the wave's LDS, since the loads' return path bounds the kernel.
// 127^3 Q1 Laplacian, FP64: 27 loads per slice 28.9 us; 9 loads with the
// neighbours by lane shifts and scalar loads 23.4 us; this form 22.0 us
// (general layout, k_spmv_sellx: 99.0 us).
// TRI: every group has three pairs; EXACT: there are U groups, one pass.
// Slices whose window leaves x (r0 + omin < 0, or r0 past `last`, the last first
// row whose 64 rows' largest columns exist) clamp a load per pair.  Workgroups are dealt so that an XCD takes consecutive rows: nothing
// but x is read more than once, and its window of a few grid planes stays in
// the XCD's L2.
template <typename T, bool ADD, bool DOT, int U, bool TRI, bool EXACT>
__global__ __launch_bounds__(kBlock) void k_spmv_pattern(Lists<T> L, int nrow, int ncol, int nslice, int npair, int ngroup, int omin,
                                                         int last, const int *__restrict__ offs,
                                                         const unsigned *__restrict__ set,
                                                         const int *__restrict__ partial, const T *__restrict__ x,
                                                         T *__restrict__ y, const T *__restrict__ w, double *part,
                                                         const int *__restrict__ done) {
    if (done && *done) return;
    constexpr int WPB = kBlock / 64, WIN = 66;
    __shared__ T win[WPB][U * WIN];
    __shared__ double shd[WPB];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int g = xcd_remap(blockIdx.x, gridDim.x);
    T *const mid = &win[wave][1 + lane];   // this lane's entry of group 0's window; entries 0 and 65 its ends
    double dsum = 0;
    for (int s = g * WPB + wave; s < nslice; s += gridDim.x * WPB) {
        const int r0 = s * 64, r = r0 + lane;
        const bool cut = partial[s] != 0;
        unsigned m = ~0u;
        if (cut) m = r < nrow ? set[r] : 0;
        T acc = 0;
        if (r0 + omin >= 0 && r0 <= last) {
            const T *xs = x + r0;
            auto add = [&](int k, T xk) {
                const T t = add_rn(acc, mul_rn(L.val[k], xk));
                acc = !cut || ((m >> k) & 1u) ? t : acc;
            };
            for (int g0 = 0; g0 < (EXACT ? 1 : ngroup); g0 += U) {
                T xv[U];
                int eoff = 0;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int o = L.grp[EXACT ? u : min(g0 + u, ngroup - 1)].off;
                    xv[u] = (xs + o)[lane];
                    eoff = (lane >> 1) == u ? o : eoff;
                }
                // lanes 2 u and 2 u + 1: the entries below and above group u's window
                if (lane < 2 * U) {
                    const int e = r0 + eoff + (lane & 1 ? 64 : -1);
                    win[wave][(lane >> 1) * WIN + (lane & 1 ? WIN - 1 : 0)] = x[TRI ? e : min(max(e, 0), ncol - 1)];
                }
#pragma unroll
                for (int u = 0; u < U; ++u) mid[u * WIN] = xv[u];
                // the windows are private to this wave, whose LDS accesses execute in order
                __builtin_amdgcn_wave_barrier();
                asm volatile("" ::: "memory");
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if (!EXACT && g0 + u >= ngroup) break;
                    Group q = L.grp[g0 + u];
                    if (TRI && EXACT) q.bit = 3 * u;
                    if (TRI || q.n == 3) {
                        add(q.bit, mid[u * WIN - 1]);
                        add(q.bit + 1, xv[u]);
                        add(q.bit + 2, mid[u * WIN + 1]);
                    } else {
                        add(q.bit, xv[u]);
                        if (q.n == 2) add(q.bit + 1, mid[u * WIN + 1]);
                    }
                }
                __builtin_amdgcn_wave_barrier();
                asm volatile("" ::: "memory");
            }
        } else {
            for (int k = 0; k < npair; ++k) {
                const long long at = static_cast<long long>(r) + offs[k];
                const T xv = x[min(max(at, 0LL), static_cast<long long>(ncol) - 1)];
                const T t = add_rn(acc, mul_rn(L.val[k], xv));
                acc = (m >> k) & 1u ? t : acc;
            }
        }
        if (r < nrow) {
            if (ADD) acc = y[r] + acc;
            y[r] = acc;
            if (DOT) dsum += static_cast<double>(acc) * static_cast<double>(w[r]);
        }
    }
    if (DOT) {
        const double vv[1] = {block_sum(dsum, shd)};
        store_partials<1>(vv, part, 0, g);
    }
}

// A value of type T from its bits.
template <typename T>
T value_of(unsigned long long u) {
    T v;
    std::memcpy(&v, &u, sizeof(T));   // the low half holds a float (little endian)
    return v;
}

// The distinct pairs of a search, ascending by offset.
struct Found {
    std::vector<std::pair<int, unsigned long long>> p;
    // false: more than a set holds
    bool add(const RowReport &q) {
        if (q.len > kMaxPairs) return false;
        for (int k = 0; k < q.len; ++k) {
            const std::pair<int, unsigned long long> e(q.off[k], q.val[k]);
            if (std::find(p.begin(), p.end(), e) != p.end()) continue;
            if (p.size() == static_cast<size_t>(kMaxPairs)) return false;
            p.push_back(e);
        }
        return true;
    }
};

// Rows spread over the matrix: false when three of them with the same offsets
// hold three different lists of values, so that a matrix of variable
// coefficients is known without a look at every row.
bool repeats(const RowReport *q) {
    auto differ = [&](int i, int j) {
        return q[i].len == q[j].len && std::memcmp(q[i].off, q[j].off, sizeof(int) * q[i].len) == 0 &&
               std::memcmp(q[i].val, q[j].val, sizeof(q[i].val[0]) * q[i].len) != 0;
    };
    for (int i = 0; i < kProbes; ++i)
        for (int j = 0; j < i; ++j)
            for (int k = 0; k < j; ++k)
                if (differ(i, j) && differ(j, k) && differ(i, k)) return false;
    return true;
}

// Rounds of the search: each looks at all rows with the pairs known so far and
// reports rows that hold others (the classes of boundary rows of a grid).
constexpr int kRounds = 8;

template <typename T>
int search(hfh_csr *A) {
    hfh_ctx *c = A->ctx;
    hipStream_t s = c->stream;
    const int n = A->nrow, nsl = (n + 63) / 64;
    RowReport *rep = static_cast<RowReport *>(c->host_reports);
    int *count = reinterpret_cast<int *>(c->red);   // rows that hold no known pair, by round
    const T *val = static_cast<const T *>(A->val);
    hipLaunchKernelGGL(k_pattern_probe<T>, dim3(kProbes + 2), dim3(64), 0, s, n, A->row, A->col, val, rep, count, kRounds);
    int rc = launch_check("k_pattern_probe");
    if (rc) return rc;
    HFH_HIP(hipStreamSynchronize(s));
    Found found;
    for (int i = 0; i < kProbes + 2; ++i)
        if (!found.add(rep[i])) return HFH_OK;
    if (!repeats(rep)) return HFH_OK;
    // one block: the offsets, the slices' flags, the sets
    const size_t at_part = sizeof(int) * kMaxPairs, at_set = at_part + sizeof(int) * nsl,
                 bytes = at_set + sizeof(unsigned) * static_cast<size_t>(n);
    if (!A->pt_block) {
        rc = copy_alloc(c, &A->pt_block, bytes);
        if (rc) return rc == HFH_ERR_NOMEM ? HFH_OK : rc;   // the general layout serves
    }
    char *blk = static_cast<char *>(A->pt_block);
    A->pt_offs = reinterpret_cast<int *>(blk);
    A->pt_partial = reinterpret_cast<int *>(blk + at_part);
    A->pt_set = reinterpret_cast<unsigned *>(blk + at_set);
    for (int round = 0; round < kRounds; ++round) {
        // A row costs its list's pairs whatever it holds: with less than a
        // quarter of them per row the entries cost less (2^20 rows, FP64; 16
        // pairs 18.7 us, 4 / 8 entries per row 17.0 / 24.9; 32 pairs 30.0 us,
        // 4 / 8 / 16 entries 19.2 / 28.5 / 44.7; 8 pairs 11.8 us, 1 / 2
        // entries 12.3 / 13.9).
        const int K = static_cast<int>(found.p.size());
        if (K == 0 || static_cast<long long>(K) * n > 4LL * A->nnz) return HFH_OK;
        std::sort(found.p.begin(), found.p.end());
        Lists<T> L{};
        Offsets O{};
        for (int k = 0; k < K; ++k) {
            O.v[k] = found.p[k].first;
            L.val[k] = value_of<T>(found.p[k].second);
        }
        for (int i = 0; i < kReports; ++i) rep[i].len = -1;
        const dim3 g((nsl + kBlock / 64 - 1) / (kBlock / 64)), bl(kBlock);
        const long long mean = (A->nnz + static_cast<long long>(n) - 1) / n;
        if (mean <= 8)
            hipLaunchKernelGGL((k_pattern_sets<T, 8>), g, bl, 0, s, n, nsl, K, L, O, A->row, A->col, val, A->pt_offs, A->pt_set, A->pt_partial, count + round, rep);
        else if (mean <= 16)
            hipLaunchKernelGGL((k_pattern_sets<T, 16>), g, bl, 0, s, n, nsl, K, L, O, A->row, A->col, val, A->pt_offs, A->pt_set, A->pt_partial, count + round, rep);
        else
            hipLaunchKernelGGL((k_pattern_sets<T, 32>), g, bl, 0, s, n, nsl, K, L, O, A->row, A->col, val, A->pt_offs, A->pt_set, A->pt_partial, count + round, rep);
        if ((rc = launch_check("k_pattern_sets"))) return rc;
        HFH_HIP(hipStreamSynchronize(s));
        bool complete = true;
        for (int i = 0; i < kReports; ++i)
            if (rep[i].len >= 0) {
                complete = false;
                if (!found.add(rep[i])) return HFH_OK;
            }
        if (!complete) continue;
        // runs of up to three neighbouring offsets; an offset with several values
        // stands alone, as a row adds its pairs in the order of the list
        const int *ho = O.v;
        int ngroup = 0;
        auto alone = [&](int k) { return (k > 0 && ho[k - 1] == ho[k]) || (k + 1 < K && ho[k + 1] == ho[k]); };
        bool tri = true;
        for (int k = 0; k < K;) {
            int m = 1;
            while (m < 3 && k + m < K && !alone(k) && !alone(k + m) && ho[k + m] == ho[k] + m) ++m;
            L.grp[ngroup++] = Group{m == 3 ? ho[k] + 1 : ho[k], k, m};
            tri = tri && m == 3;
            k += m;
        }
        A->pt_pairs = K;
        A->pt_ngroups = ngroup;
        const char *lists = reinterpret_cast<const char *>(&L);
        A->pt_lists.assign(lists, lists + sizeof(L));
        A->pt_tri = tri;
        A->pt_omin = ho[0];
        A->pt_omax = ho[K - 1];
        return HFH_OK;
    }
    return HFH_OK;
}

template <typename T>
void scale_lists(hfh_csr *A, T a, bool offdiag_only) {
    Lists<T> L;
    std::memcpy(&L, A->pt_lists.data(), sizeof(L));
    for (int g = 0; g < A->pt_ngroups; ++g) {
        const Group &q = L.grp[g];
        const int off = q.n == 3 ? q.off - 1 : q.off;   // of the group's first pair
        for (int i = 0; i < q.n; ++i)
            if (!offdiag_only || off + i != 0) L.val[q.bit + i] *= a;   // one rounding, as the entries'
    }
    std::memcpy(A->pt_lists.data(), &L, sizeof(L));
}

template <typename T, bool ADD, bool DOT, int U, bool TRI, bool EXACT>
void launch_u(const hfh_csr *A, const T *x, T *y, const T *w, double *part, const int *done) {
    Lists<T> L;
    std::memcpy(&L, A->pt_lists.data(), sizeof(L));
    const long long last = std::min(static_cast<long long>(A->ncol) - 64 - A->pt_omax, 0x7fffffffLL);
    hipLaunchKernelGGL((k_spmv_pattern<T, ADD, DOT, U, TRI, EXACT>), dim3(A->nwg), dim3(kBlock), 0, A->ctx->stream, L,
                       A->nrow, A->ncol, A->nslice, A->pt_pairs, A->pt_ngroups, A->pt_omin, static_cast<int>(std::max(last, -1LL)), A->pt_offs,
                       A->pt_set, A->pt_partial, x, y, w, part, done);
}

// The box stencils in 2D (3 groups of three) and 3D (9), the face stencils in
// 2D (3 groups) and 3D (5) in one pass, anything else in passes of 5.
template <typename T, bool ADD, bool DOT>
void launch(const hfh_csr *A, const T *x, T *y, const T *w, double *part, const int *done) {
    const int G = A->pt_ngroups;
    if (A->pt_tri && G == 3) launch_u<T, ADD, DOT, 3, true, true>(A, x, y, w, part, done);
    else if (A->pt_tri && G == 9) launch_u<T, ADD, DOT, 9, true, true>(A, x, y, w, part, done);
    else if (G == 3) launch_u<T, ADD, DOT, 3, false, true>(A, x, y, w, part, done);
    else if (G == 5) launch_u<T, ADD, DOT, 5, false, true>(A, x, y, w, part, done);
    else launch_u<T, ADD, DOT, 5, false, false>(A, x, y, w, part, done);
}

template <typename T>
void launch_modes(const hfh_csr *A, const void *x, void *y, int mode, const void *w, double *part, const int *done) {
    const T *xv = static_cast<const T *>(x), *wv = static_cast<const T *>(w);
    T *yv = static_cast<T *>(y);
    if (mode == 0 && !w) launch<T, false, false>(A, xv, yv, wv, part, done);
    else if (mode == 0) launch<T, false, true>(A, xv, yv, wv, part, done);
    else if (!w) launch<T, true, false>(A, xv, yv, wv, part, done);
    else launch<T, true, true>(A, xv, yv, wv, part, done);
}

}  // namespace

void pattern_free(hfh_csr *A) {
    if (A->pt_block) (void)hipFree(A->pt_block);
    A->pt_block = nullptr;
    A->pt_pairs = 0;
    A->pt_want = false;
}

int pattern_fill(hfh_csr *A) {
    A->pt_pairs = 0;
    if (!A->pt_want || !A->sorted || A->nrow == 0 || A->nnz == 0) return HFH_OK;
    return A->dtype == HFH_F64 ? search<double>(A) : search<float>(A);
}

void pattern_scale(hfh_csr *A, double alpha, bool offdiag_only) {
    if (A->pt_pairs == 0) return;
    if (A->dtype == HFH_F64) scale_lists<double>(A, alpha, offdiag_only);
    else scale_lists<float>(A, static_cast<float>(alpha), offdiag_only);
}

int pattern_spmv(const hfh_csr *A, const void *x, void *y, int mode, const void *w, double *part, const int *done) {
    if (A->dtype == HFH_F64) launch_modes<double>(A, x, y, mode, w, part, done);
    else launch_modes<float>(A, x, y, mode, w, part, done);
    return launch_check("k_spmv_pattern");
}

}  // namespace hfh

using namespace hfh;

extern "C" int hfh_csr_pattern_pairs(const hfh_csr *A, int *pairs) {
    HFH_CHECK(A && pairs, HFH_ERR_INVALID, "hfh_csr_pattern_pairs: null argument");
    *pairs = A->pt_pairs;
    return HFH_OK;
}

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
#include <thread>

namespace hfh {
namespace {

constexpr int kMaxPatterns = 64;   // distinct rows of offsets looked at
constexpr int kMaxPairs = 32;      // bits of a row's set

// Values of the listed rows, one workgroup per row, at out[g * kMaxPairs].
template <typename T>
__global__ void k_pattern_gather(const int *__restrict__ rows, const int *__restrict__ row,
                                 const T *__restrict__ val, T *__restrict__ out) {
    const int r = rows[blockIdx.x], j0 = row[r], len = row[r + 1] - j0;
    const int k = threadIdx.x;
    if (k < kMaxPairs) out[blockIdx.x * kMaxPairs + k] = k < len ? val[j0 + k] : static_cast<T>(0);
}

__device__ __forceinline__ bool same_bits(double a, double b) { return __builtin_bit_cast(unsigned long long, a) == __builtin_bit_cast(unsigned long long, b); }
__device__ __forceinline__ bool same_bits(float a, float b) { return __builtin_bit_cast(unsigned, a) == __builtin_bit_cast(unsigned, b); }

// Every row's set of pairs and, per slice of 64 rows, whether all its rows
// hold all pairs; *fail when a row has an entry that is no pair.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_pattern_sets(int nrow, int npair, const int *__restrict__ offs,
                                                         const T *__restrict__ vals, const int *__restrict__ row,
                                                         const int *__restrict__ col, const T *__restrict__ val,
                                                         unsigned *__restrict__ set, int *__restrict__ partial,
                                                         int *fail) {
    const int r = blockIdx.x * kBlock + threadIdx.x;
    const unsigned all = npair == 32 ? ~0u : (1u << npair) - 1;
    unsigned m = 0;
    bool bad = false;
    if (r < nrow) {
        int k = 0;
        for (int j = row[r]; j < row[r + 1] && !bad; ++j) {
            const int o = col[j] - r;
            const T v = val[j];
            while (k < npair && (offs[k] < o || (offs[k] == o && !same_bits(vals[k], v)))) ++k;
            if (k < npair && offs[k] == o) m |= 1u << k++;
            else bad = true;
        }
        set[r] = m;
    }
    const bool some = __any(r < nrow && m != all);
    if ((threadIdx.x & 63) == 0 && r < nrow) partial[r >> 6] = some ? 1 : 0;
    if (bad) *fail = 1;
}

// Pairs with neighbouring offsets share one load of x.
struct Group {
    int off;       // offset of the loaded entries: the middle pair of three, else the first
    int bit, n;    // pairs bit .. bit + n - 1, n = 1 .. 3
};

// The lists as a kernel argument: with compile-time positions all of them
// come in a few wide scalar loads before the first load of x (read from
// memory one by one, each load of x waited for its group: 25.1 us).
template <typename T>
struct Lists {
    Group grp[kMaxPairs];
    T val[kMaxPairs];
};

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

template <typename T>
bool same_value(T a, T b) { return std::memcmp(&a, &b, sizeof(T)) == 0; }

bool same_offsets(const hfh_csr *A, int a, int b) {
    const int *row = A->h_row.data(), *col = A->h_col.data();
    const int ja = row[a], jb = row[b], len = row[a + 1] - ja;
    if (row[b + 1] - jb != len) return false;
    for (int k = 0; k < len; ++k)
        if (col[ja + k] - a != col[jb + k] - b) return false;
    return true;
}

template <typename T>
int fill(hfh_csr *A) {
    hipStream_t s = A->ctx->stream;
    const int np = static_cast<int>(A->pt_rows.size()), n = A->nrow, nsl = (n + 63) / 64;
    // one block: the sets, the slices' flags, the lists, then what only this
    // function uses (the sample rows, their values, the failure word)
    const size_t samples = static_cast<size_t>(np) * kMaxPairs * sizeof(T);
    const size_t at_vals = 0, at_smp = at_vals + kMaxPairs * sizeof(T), at_offs = at_smp + samples, at_rows = at_offs + kMaxPairs * sizeof(int),
                 at_fail = at_rows + sizeof(int) * np, at_part = at_fail + sizeof(int),
                 at_set = at_part + sizeof(int) * nsl, bytes = at_set + sizeof(unsigned) * static_cast<size_t>(n);
    if (!A->pt_block) {
        const int rc = copy_alloc(A->ctx, &A->pt_block, bytes);
        if (rc) return rc == HFH_ERR_NOMEM ? HFH_OK : rc;   // the general layout serves
    }
    char *blk = static_cast<char *>(A->pt_block);
    T *d_vals = reinterpret_cast<T *>(blk + at_vals);
    A->pt_offs = reinterpret_cast<int *>(blk + at_offs);
    A->pt_partial = reinterpret_cast<int *>(blk + at_part);
    A->pt_set = reinterpret_cast<unsigned *>(blk + at_set);
    int *d_rows = reinterpret_cast<int *>(blk + at_rows), *d_fail = reinterpret_cast<int *>(blk + at_fail);
    T *d_smp = reinterpret_cast<T *>(blk + at_smp);
    std::vector<T> hv(static_cast<size_t>(np) * kMaxPairs);
    HFH_HIP(hipMemcpyAsync(d_rows, A->pt_rows.data(), sizeof(int) * np, hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_pattern_gather<T>, dim3(np), dim3(64), 0, s, d_rows, A->row, static_cast<const T *>(A->val),
                       d_smp);
    HFH_HIP(hipMemcpyAsync(hv.data(), d_smp, samples, hipMemcpyDeviceToHost, s));
    HFH_HIP(hipStreamSynchronize(s));
    // the distinct pairs of the sample rows, ascending by offset
    std::vector<std::pair<int, T>> pairs;
    for (int i = 0; i < np; ++i) {
        const int r = A->pt_rows[i], j0 = A->h_row[r], len = A->h_row[r + 1] - j0;
        for (int k = 0; k < len; ++k) {
            const int o = A->h_col[j0 + k] - r;
            const T v = hv[static_cast<size_t>(i) * kMaxPairs + k];
            bool known = false;
            for (const auto &q : pairs) known = known || (q.first == o && same_value(q.second, v));
            if (!known) {
                if (static_cast<int>(pairs.size()) == kMaxPairs) return HFH_OK;
                pairs.emplace_back(o, v);
            }
        }
    }
    if (pairs.empty()) return HFH_OK;
    std::stable_sort(pairs.begin(), pairs.end(), [](const auto &a, const auto &b) { return a.first < b.first; });
    const int K = static_cast<int>(pairs.size());
    Lists<T> L{};
    std::vector<int> ho(K);
    for (int k = 0; k < K; ++k) {
        ho[k] = pairs[k].first;
        L.val[k] = pairs[k].second;
    }
    // runs of up to three neighbouring offsets; an offset with several values
    // stands alone, as a row adds its pairs in the order of the list
    int ngroup = 0;
    auto alone = [&](int k) { return (k > 0 && ho[k - 1] == ho[k]) || (k + 1 < K && ho[k + 1] == ho[k]); };
    bool tri = true;
    for (int k = 0; k < K;) {
        int c = 1;
        while (c < 3 && k + c < K && !alone(k) && !alone(k + c) && ho[k + c] == ho[k] + c) ++c;
        L.grp[ngroup++] = Group{c == 3 ? ho[k] + 1 : ho[k], k, c};
        tri = tri && c == 3;
        k += c;
    }
    int fail = 0;
    HFH_HIP(hipMemcpyAsync(A->pt_offs, ho.data(), sizeof(int) * K, hipMemcpyHostToDevice, s));
    HFH_HIP(hipMemcpyAsync(d_vals, L.val, sizeof(T) * K, hipMemcpyHostToDevice, s));
    HFH_HIP(hipMemcpyAsync(d_fail, &fail, sizeof(int), hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_pattern_sets<T>, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, n, K, A->pt_offs,
                       d_vals, A->row, A->col, static_cast<const T *>(A->val), A->pt_set, A->pt_partial, d_fail);
    HFH_HIP(hipMemcpyAsync(&fail, d_fail, sizeof(int), hipMemcpyDeviceToHost, s));
    HFH_HIP(hipStreamSynchronize(s));
    if (fail) return HFH_OK;
    A->pt_pairs = K;
    A->pt_ngroups = ngroup;
    const char *lists = reinterpret_cast<const char *>(&L);
    A->pt_lists.assign(lists, lists + sizeof(L));
    A->pt_tri = tri;
    A->pt_omin = ho[0];
    A->pt_omax = ho[K - 1];
    return HFH_OK;
}

// Rows spread over the matrix: false when three of them with the same offsets
// hold three different lists of values, so that a matrix of variable
// coefficients is known without a look at every row.
template <typename T>
int probe(const hfh_csr *A, bool *repeat) {
    constexpr int N = 8;
    hipStream_t s = A->ctx->stream;
    T v[N][kMaxPairs];
    int r[N], len[N];
    *repeat = false;
    for (int i = 0; i < N; ++i) {
        r[i] = static_cast<int>(static_cast<long long>(A->nrow) * (i + 1) / (N + 1));
        len[i] = A->h_row[r[i] + 1] - A->h_row[r[i]];
        if (len[i] > kMaxPairs) return HFH_OK;
        if (len[i] > 0)
            HFH_HIP(hipMemcpyAsync(v[i], static_cast<const T *>(A->val) + A->h_row[r[i]], sizeof(T) * len[i],
                                   hipMemcpyDeviceToHost, s));
    }
    HFH_HIP(hipStreamSynchronize(s));
    auto differ = [&](int i, int j) { return same_offsets(A, r[i], r[j]) && std::memcmp(v[i], v[j], sizeof(T) * len[i]) != 0; };
    for (int i = 0; i < N; ++i)
        for (int j = 0; j < i; ++j)
            for (int k = 0; k < j; ++k)
                if (differ(i, j) && differ(j, k) && differ(i, k)) return HFH_OK;
    *repeat = true;
    return HFH_OK;
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
    A->pt_rows.clear();
    A->pt_want = A->pt_scanned = false;
}

// Sample rows: the first and the last row of every pattern of offsets that
// each host thread's range holds.  None are kept when there are too many
// patterns, a row is longer than a set can hold or its columns do not ascend
// (a diagonal-first matrix).
static void sample(hfh_csr *A) {
    const int n = A->nrow;
    const int *row = A->h_row.data(), *col = A->h_col.data();
    auto same = [&](int a, int b) { return same_offsets(A, a, b); };
    struct Found {
        std::vector<int> first, last;
        bool over = false;
    };
    auto add = [&](Found &f, int r, int at) -> int {   // the pattern of row r, or -1 when there are too many
        if (at >= 0 && same(f.last[at], r)) {
            f.last[at] = r;
            return at;
        }
        for (size_t i = 0; i < f.first.size(); ++i)
            if (same(f.first[i], r)) {
                f.last[i] = r;
                return static_cast<int>(i);
            }
        const int j0 = row[r], j1 = row[r + 1];
        bool ok = static_cast<int>(f.first.size()) < kMaxPatterns && j1 - j0 <= kMaxPairs;
        for (int j = j0 + 1; ok && j < j1; ++j) ok = col[j] > col[j - 1];
        if (!ok) {
            f.over = true;
            return -1;
        }
        f.first.push_back(r);
        f.last.push_back(r);
        return static_cast<int>(f.first.size()) - 1;
    };
    const int nt = n < 4096 ? 1 : static_cast<int>(std::min(16u, std::max(1u, std::thread::hardware_concurrency())));
    std::vector<Found> found(nt);
    auto scan = [&](int t) {
        const int lo = static_cast<int>(static_cast<long long>(n) * t / nt);
        const int hi = static_cast<int>(static_cast<long long>(n) * (t + 1) / nt);
        int at = -1;
        for (int r = lo; r < hi && !found[t].over; ++r) at = add(found[t], r, at);
    };
    if (nt == 1) {
        scan(0);
    } else {
        std::vector<std::thread> th;
        for (int t = 0; t < nt; ++t) th.emplace_back(scan, t);
        for (auto &t : th) t.join();
    }
    Found all;
    for (const Found &f : found) {
        if (f.over) return;
        for (int r : f.first)
            if (add(all, r, -1) < 0) return;
        for (int r : f.last)
            if (add(all, r, -1) < 0) return;
    }
    A->pt_rows = all.first;
    for (size_t i = 0; i < all.first.size(); ++i)
        if (all.last[i] != all.first[i]) A->pt_rows.push_back(all.last[i]);
}

int pattern_fill(hfh_csr *A) {
    A->pt_pairs = 0;
    if (!A->pt_want || A->nrow == 0 || A->nnz == 0) return HFH_OK;
    bool repeat = false;
    int rc = A->dtype == HFH_F64 ? probe<double>(A, &repeat) : probe<float>(A, &repeat);
    if (rc || !repeat) return rc;
    if (!A->pt_scanned) sample(A);
    A->pt_scanned = true;
    if (A->pt_rows.empty()) return HFH_OK;
    return A->dtype == HFH_F64 ? fill<double>(A) : fill<float>(A);
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

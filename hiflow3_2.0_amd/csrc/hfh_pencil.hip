// hfh_pencil.hip -- SGS / ILU(0) triangular sweeps of 5- and 7-point
// natural-order grids, streamed along x by pencils of 64 lines.
//
// A triangular sweep of such a grid is a wavefront over x + y + z: the chain
// of dependent rows (nx + ny + nz) bounds it, not the bytes.  The sweep by
// 4x4x4 blocks (k_bsweep_sf) pays one cross-CU round trip per block level, 94
// of them on 128^3.  Here one wave owns a pencil: the 8 x 8 lines of (y, z)
// (64 lines of y in 2D) along the whole of x, lane = line.  At step s lane
// (yl, zl) computes x = s - yl - zl, so its y and z neighbours finished one
// step ago in lanes l - 1 and l - 8 (read from the LDS slots of the last
// step) and its x neighbour is its own last result.  Only the faces cross to
// another CU, as a stream: a pencil runs behind its predecessors by the skew
// of its cross-section plus one transfer, so the transfers of a chain of
// pencils overlap the steps, and 128^3 pays 30 of them instead of 94, with
// no wait inside a pencil.
//
// A workgroup is two waves.  Wave 0 computes: matrix values, right-hand side
// and diagonal come from registers loaded kAhead groups of 4 steps earlier.
// Wave 1 fetches: it polls the pencil's inbox (the predecessors' faces, one
// row per step, stored with agent-scope atomics over a signalling-NaN
// sentinel) and copies complete rows into the LDS slots, so that the polls'
// waits never queue behind the value loads of wave 0.  Rows move in groups
// of 4 steps: one 64-lane load or store carries 4 rows of 16 face values.
//
// Each row's arithmetic is the sequential loop's (the entries in stored
// order, product and difference rounded separately, then the division), so
// the results are bit-identical to the other schedules.  The division by the
// diagonal sits on the chain: with r = RN(1/d) stored beside d, q = a r and
// two corrections q += RN(a - d q) r give RN(a / d) exactly (Markstein: a
// faithful q, an exact remainder and a correctly rounded reciprocal round to
// the quotient) in 5 dependent operations instead of the compiler's 11;
// operands outside a range where that holds take the plain division.
//
// Measured (apply, both sweeps, FP64; blocks -> pencils): upwind 128^3 ILU(0)
// 480 -> 267 us, SGS 529 -> 284 us; 2D 701 x 509 SGS 896 -> 427 us; 40^3 SGS
// 136 -> 86 us; 16^3 51 -> 39 us; 64 x 64 89 -> 50 us.  A step took about 150
// ns and a hop to the next pencil about 2 us on top of its skew.  The step is
// bound by what a lone wave issues: a dependent FP64 operation 6 to 7 cycles, an
// LDS write and read back 66, a lane shift of a double 31, a branch on lanes'
// values 70.  Without branches in the steps, with lane shifts instead of LDS
// in 2D and plain value loads, 2D 701 x 509 SGS takes 383 us.
#include "hfh_internal.h"

#include <algorithm>

namespace hfh {

namespace {

// Groups of 4 steps whose operands are in flight (upwind 128^3 GMRES + ILU(0) /
// 2D 701 x 509 SGS: 4 groups 94.1 ms / 384 us, 6 93.9 / 383, 8 93.4 / 411).
// Both forms of a group issue the same number of accesses, so that the waits
// count them exactly: with two 16-byte accesses in place of four inside the
// lines GMRES took 100 ms.
constexpr int kAhead = 6;
constexpr int kSlots = 32;      // steps held in the LDS ring
constexpr int kPencilSpins = 1 << 20;

template <typename T> struct Bits;
template <> struct Bits<double> {
    typedef unsigned long long U;
    static constexpr U sentinel = 0x7FF4DEAD5EEDBEEFull;   // exponent all ones, quiet bit clear
    static constexpr U quiet = 1ull << 51;
    static constexpr double dlo = 0x1p-300, dhi = 0x1p300;
    // |a| in [2^-500, 2^500], as a range of the high word shifted left by one
    static constexpr unsigned alo = (1023u - 500u) << 21, alen = 1000u << 21;
    static __device__ __forceinline__ unsigned top(double a) {
        return static_cast<unsigned>(__builtin_bit_cast(U, a) >> 32);
    }
};
template <> struct Bits<float> {
    typedef unsigned int U;
    static constexpr U sentinel = 0x7FA5EED5u;
    static constexpr U quiet = 1u << 22;
    static constexpr float dlo = 0x1p-40f, dhi = 0x1p40f;
    static constexpr unsigned alo = (127u - 60u) << 24, alen = 120u << 24;
    static __device__ __forceinline__ unsigned top(float a) { return __builtin_bit_cast(U, a); }
};

__device__ __forceinline__ double fma_t(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fma_t(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// a / d rounded once, r = RN(1 / d) (see above), where |a| lies in the range
// of the fast form or a is +0; else `worst` becomes at least Bits<T>::alen and
// the caller divides plainly.
template <typename T>
__device__ __forceinline__ T quotient(T a, T d, T r, unsigned &worst) {
    typedef typename Bits<T>::U U;
    T q = mul_rn(a, r);
    q = fma_t(fma_t(-q, d, a), r, q);
    q = fma_t(fma_t(-q, d, a), r, q);
    const unsigned t = (Bits<T>::top(a) << 1) - Bits<T>::alo;
    worst = max(worst, __builtin_bit_cast(U, a) == 0 ? 0u : t);
    return q;
}

// The value of the lane below; lane 0 gets `edge`.
__device__ __forceinline__ unsigned lane_below(unsigned v, unsigned edge) {
    return __builtin_amdgcn_update_dpp(edge, v, 0x138, 0xf, 0xf, false);   // wave_shr:1
}
__device__ __forceinline__ float from_below(float v, float edge) {
    return __builtin_bit_cast(float, lane_below(__builtin_bit_cast(unsigned, v), __builtin_bit_cast(unsigned, edge)));
}
__device__ __forceinline__ double from_below(double v, double edge) {
    typedef unsigned long long U;
    const U a = __builtin_bit_cast(U, v), e = __builtin_bit_cast(U, edge);
    const unsigned lo = lane_below(static_cast<unsigned>(a), static_cast<unsigned>(e));
    const unsigned hi = lane_below(static_cast<unsigned>(a >> 32), static_cast<unsigned>(e >> 32));
    return __builtin_bit_cast(double, static_cast<U>(hi) << 32 | lo);
}

template <typename T>
__device__ __forceinline__ typename Bits<T>::U face_load(const T *p) {
    return __hip_atomic_load(reinterpret_cast<const typename Bits<T>::U *>(p), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
}

// Element access with a byte offset checked against the vector's size: a
// lane outside the grid uses kOutside, reads 0 and stores nothing.
// kOutside + a line's own offset is outside as well: vectors and inboxes are
// at most 2^31 bytes, a line's offsets below 2^30.
constexpr unsigned kOutside = 0xC0000000u;
typedef unsigned U2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ double vec_load(__amdgpu_buffer_rsrc_t b, unsigned off, double) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(b, off, 0, 0));
}
__device__ __forceinline__ float vec_load(__amdgpu_buffer_rsrc_t b, unsigned off, float) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(b, off, 0, 0));
}
__device__ __forceinline__ void vec_store(__amdgpu_buffer_rsrc_t b, unsigned off, double v) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, v), b, off, 0, 0);
}
__device__ __forceinline__ void vec_store(__amdgpu_buffer_rsrc_t b, unsigned off, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), b, off, 0, 0);
}
// A face value, visible to the other CUs (agent scope: sc1), without the
// branch that an exec-masked store costs.  It is the result of an addition,
// so never the sentinel: those quiet a signalling NaN.
constexpr int kAgentScope = 16;
typedef unsigned U4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void face_store(__amdgpu_buffer_rsrc_t b, unsigned off, double v) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, v), b, off, 0, kAgentScope);
}
__device__ __forceinline__ void face_store(__amdgpu_buffer_rsrc_t b, unsigned off, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), b, off, 0, kAgentScope);
}

// Four neighbouring face values, the lowest at `off` (aligned to an element).
__device__ __forceinline__ void face_store4(__amdgpu_buffer_rsrc_t b, unsigned off, const double (&v)[4]) {
    typedef double D2 __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(U4, D2{v[0], v[1]}), b, off, 0, kAgentScope);
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(U4, D2{v[2], v[3]}), b, off + 16, 0, kAgentScope);
}
__device__ __forceinline__ void face_store4(__amdgpu_buffer_rsrc_t b, unsigned off, const float (&v)[4]) {
    typedef float F4 __attribute__((ext_vector_type(4)));
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(U4, F4{v[0], v[1], v[2], v[3]}), b, off, 0, kAgentScope);
}

// The shape of a sweep's pencils.  Coordinates are the sweep's own: the
// backward sweep counts x, y and z from the far end, so both sweeps depend
// on lower coordinates only.
template <bool D3> struct Shape {
    static constexpr int BY = D3 ? 8 : 64;           // lines along y = steps a pencil runs behind its predecessor
    static constexpr int SKEW = D3 ? 14 : 63;        // last lane's delay
    static constexpr int H = D3 ? 16 : 1;            // face values of a step (y face, then z face)
    static constexpr int NV = D3 ? 3 : 2;            // neighbours a row waits for
    static constexpr int ZERO = 64 + H;              // LDS slot: 64 results, H face values, a zero
    static constexpr int SLOT = D3 ? 82 : 68;
};

}  // namespace

template <typename T>
struct PencilArgs {
    int nx, ny, nz, npy, npz, ng;
    const int *order;          // pencils by npy-diagonal: J | K << 16
    const T *val;              // values, (pencil, group, step pair, entry, lane, step of the pair)
    T *y;                      // forward results, (pencil, 4 + step, lane)
    const T *in;               // forward: right-hand side (natural order)
    T *out;                    // backward: result (natural order)
    T *box, *other_box;        // inboxes of this sweep / of the other one, (pencil, row, face value)
    int *ctl;                  // [0] / [32] tickets of the forward / backward sweep, [64] slow division
    int *fail;                 // [0] failure word, [1] the most polls for one row
    const int *done;
};

// One sweep: MODE 0 SGS forward, 1 SGS backward, 2 ILU forward, 3 ILU backward.
template <typename T, int MODE, bool D3>
__global__ __launch_bounds__(128) void k_pencil(PencilArgs<T> a) {
    typedef Shape<D3> S;
    typedef typename Bits<T>::U U;
    typedef T V2 __attribute__((ext_vector_type(2)));
    constexpr bool FW = MODE == 0 || MODE == 2, DIV = MODE != 2;
    constexpr int H = S::H, NV = S::NV, SLOT = S::SLOT, K = NV + (DIV ? 2 : 0);
    __shared__ T ring[kSlots * SLOT];
    __shared__ int s_ticket, s_ready, s_read;
    if (a.done && *a.done) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ng = a.ng, np = a.npy * a.npz;
    // the other sweep's ticket counter starts its next launch at 0
    if (blockIdx.x == 0 && threadIdx.x == 0) a.ctl[FW ? 32 : 0] = 0;
    const bool slow = DIV && a.ctl[64] != 0;   // some diagonal is outside [dlo, dhi]
    for (;;) {
        // Pencils are taken in dependency order, so the earliest unfinished
        // one never waits for a pencil that no workgroup holds.
        if (threadIdx.x == 0) {
            s_ticket = __hip_atomic_fetch_add(a.ctl + (FW ? 0 : 32), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            s_ready = 0;
            s_read = 0;
        }
        for (int k = threadIdx.x; k < kSlots * SLOT; k += 128) ring[k] = T(0);
        __syncthreads();
        const int t = __builtin_amdgcn_readfirstlane(s_ticket);
        if (t >= np) break;
        const int J = a.order[t] & 0xffff, KK = a.order[t] >> 16;
        const int pn = KK * a.npy + J;
        T *const inbox = a.box + static_cast<size_t>(pn) * ng * 4 * H;
        if (wave == 1) {
            // ---- the fetching wave: face rows S::BY .. of the inbox into
            // the slots of steps 0 .. , in order, complete rows only
            constexpr int RPL = 64 / H;                  // rows per load
            constexpr int W = D3 ? 4 : 1;                // loads in flight once rows arrive
            const int total = a.nx + (D3 ? 7 : 0);       // rows a pencil uses
            const int e = lane % H, lr = lane / H;
            const bool has = D3 ? (e < 8 ? J > 0 : KK > 0) : J > 0;
            const bool any = J > 0 || (D3 && KK > 0);
            int row = 0, spins = 0, most = 0, nw = 1;
            bool gave_up = false;
            while (any && row < total) {
                // slots free up as the computing wave passes them
                const int lim = min(total, 4 * __hip_atomic_load(&s_read, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) + kSlots);
                if (row >= lim) {
                    __builtin_amdgcn_s_sleep(1);
                    continue;
                }
                U u[W];
#pragma unroll
                for (int w = 0; w < W; ++w) {
                    const int r = row + w * RPL + lr;
                    u[w] = w < nw && has && r < total ? face_load(inbox + static_cast<size_t>(r + S::BY) * H + e) : U(0);
                }
                int cnt = 0;
#pragma unroll
                for (int w = 0; w < W; ++w) {
                    const unsigned long long m = __builtin_amdgcn_ballot_w64(u[w] == Bits<T>::sentinel && !gave_up);
                    if (w < nw && cnt == w * RPL) cnt += m ? __builtin_ctzll(m) / H : RPL;
                }
                cnt = min(cnt, lim - row);
#pragma unroll
                for (int w = 0; w < W; ++w) {
                    const int k = w * RPL + lr;
                    if (k < cnt) ring[((row + k) & (kSlots - 1)) * SLOT + 64 + e] = __builtin_bit_cast(T, u[w]);
                }
                row += cnt;
                asm volatile("" ::: "memory");   // a wave's LDS writes complete in order
                if (cnt > 0) {
                    if (lane == 0) __hip_atomic_store(&s_ready, row, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    nw = W;
                    most = max(most, spins);
                    spins = 0;
                    continue;
                }
                nw = 1;
                ++spins;
                if ((spins & 255) == 0 && (spins >= kPencilSpins || __hip_atomic_load(a.fail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
                    __hip_atomic_store(a.fail, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    gave_up = true;   // the sentinels go through as NaN
                }
                __builtin_amdgcn_s_sleep(1);
            }
            // the remaining rows carry no face: zeros
            for (; row < 4 * ng;) {
                const int lim = min(4 * ng, 4 * __hip_atomic_load(&s_read, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) + kSlots);
                if (row >= lim) {
                    __builtin_amdgcn_s_sleep(1);
                    continue;
                }
                for (; row < lim; ++row)
                    if (lane < H) ring[(row & (kSlots - 1)) * SLOT + 64 + lane] = T(0);
                asm volatile("" ::: "memory");
                if (lane == 0) __hip_atomic_store(&s_ready, row, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
            most = max(most, spins);
            if (lane == 0 && most > 0) __hip_atomic_fetch_max(a.fail + 1, most, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            // the other sweep's inbox of this pencil, back to the sentinel
            // (that sweep is over, or not yet launched)
            U *ob = reinterpret_cast<U *>(a.other_box + static_cast<size_t>(pn) * ng * 4 * H);
            for (int k = lane; k < ng * 4 * H; k += 64) ob[k] = Bits<T>::sentinel;
        } else {
            // ---- the computing wave
            const int yl = D3 ? lane & 7 : lane, zl = D3 ? lane >> 3 : 0;
            const int rp = np - 1 - pn;      // the same pencil counted from the other end
            const int y = FW ? J * S::BY + yl : (a.npy - J) * S::BY - 1 - yl;
            const int z = !D3 ? 0 : FW ? KK * 8 + zl : (a.npz - KK) * 8 - 1 - zl;
            const bool valid = y < a.ny && z < a.nz;
            // row of (x = 0 of the sweep's own count, this line), as a byte offset
            const long long r0 = static_cast<long long>(z * a.ny + y) * a.nx + (FW ? 0 : a.nx - 1);
            const int dir = FW ? static_cast<int>(sizeof(T)) : -static_cast<int>(sizeof(T));
            const int x00 = valid ? -yl - zl : -(1 << 30);   // x at step 0; a line outside the grid never starts
            const unsigned off00 = static_cast<unsigned>(r0 * static_cast<long long>(sizeof(T)) + static_cast<long long>(dir) * (-yl - zl));
            auto at = [&](int s) {
                return static_cast<unsigned>(x00 + s) < static_cast<unsigned>(a.nx) ? off00 + static_cast<unsigned>(dir * s) : kOutside;
            };
            const unsigned off0 = valid ? off00 : kOutside;
            // steps of a group past every line's start and before any one's end
            auto inside = [&](int gi) { return 4 * gi >= S::SKEW && 4 * gi + 3 < a.nx; };
            const unsigned nbytes = static_cast<unsigned>(static_cast<long long>(a.nx) * a.ny * a.nz * sizeof(T));
            const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(FW ? a.in : a.out), (short)0, nbytes, 0x00027000);
            const V2 *vbase = reinterpret_cast<const V2 *>(a.val) + static_cast<size_t>(pn) * ng * 2 * K * 64;
            const size_t slab = static_cast<size_t>(4) * ng + 4;
            // a line outside the grid stores nothing: its results stay 0 there
            const auto ys = __builtin_amdgcn_make_buffer_rsrc(a.y + static_cast<size_t>(pn) * slab * 64, (short)0,
                                                              static_cast<unsigned>(slab * 64 * sizeof(T)), 0x00027000);
            const unsigned yoff = valid ? (4 * 64 + lane) * static_cast<unsigned>(sizeof(T)) : kOutside;
            const T *const yr = a.y + (static_cast<size_t>(rp) * slab + 4 + a.nx + S::SKEW - 1) * 64 + 63 - lane;
            // where this wave's y / z neighbours' results stand in a slot
            const bool yin = yl > 0, zin = zl > 0;
            const int aB = !valid ? S::ZERO : yin ? lane - 1 : 64 + zl;   // 3D
            const int aC = !valid ? S::ZERO : zin ? lane - 8 : 72 + yl;
            // 3D, faces out: lane -> (row of the group, face value) -> the successor's inbox
            const int frow = lane / 16, fe = lane % 16;
            const bool yface = fe < 8;
            const int fsrc = yface ? 7 + 8 * fe : 56 + fe - 8;
            const auto bs = __builtin_amdgcn_make_buffer_rsrc(a.box, (short)0, static_cast<unsigned>(sizeof(T)) * np * ng * 4 * H, 0x00027000);
            const unsigned ES = sizeof(T);
            const unsigned fdst = !D3 ? (lane == 63 && J + 1 < a.npy ? ((pn + 1) * ng * 4 + 1) * ES : kOutside)
                                : (yface ? J + 1 < a.npy : KK + 1 < a.npz)
                                    ? (((yface ? pn + 1 : pn + a.npy) * ng * 4 + frow) * H + fe) * ES : kOutside;
            struct Grp {
                V2 v[2][K];
                T s[4];
            } grp[kAhead];
            auto load = [&](Grp &g, int gi) {
                gi = min(gi, ng - 1);
                const V2 *p = vbase + static_cast<size_t>(gi) * 2 * K * 64;
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int k = 0; k < K; ++k) g.v[h][k] = p[(h * K + k) * 64 + lane];
                if (!FW) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) g.s[j] = yr[-(4 * gi + j) * 64];
                } else {
                    const bool in = inside(gi);
#pragma unroll
                    for (int j = 0; j < 4; ++j) g.s[j] = vec_load(rs, in ? off0 + dir * (4 * gi + j) : at(4 * gi + j), T(0));
                }
            };
            T prev = T(0);
            int ready = 0;
            auto group = [&](const Grp &g, int gi, bool edge) {
                while (ready < 4 * gi + 4) {
                    ready = __builtin_amdgcn_readfirstlane(__hip_atomic_load(&s_ready, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
                }
                asm volatile("" ::: "memory");
                T *const base = ring + (gi & (kSlots / 4 - 1)) * 4 * SLOT;
                T *const next = ring + ((gi + 1) & (kSlots / 4 - 1)) * 4 * SLOT;
                T face[4], res[4], f = T(0);
                if (!D3) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) face[j] = base[j * SLOT + 64];
                }
                const T prev0 = prev;
                unsigned worst = 0;
                auto steps = [&](bool plain) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        // 2D: the y neighbour's result from its lane's register
                        const T B = D3 ? base[j * SLOT + aB] : from_below(prev, face[j]);
                        const T C = D3 ? base[j * SLOT + aC] : T(0);
                        const T A = prev;
                        const V2(&v)[K] = g.v[j >> 1];
                        T acc = g.s[j];
                        if (FW) {
                            if (D3) acc = add_rn(acc, -mul_rn(C, v[NV - 1][j & 1]));
                            acc = add_rn(acc, -mul_rn(B, v[1][j & 1]));
                            acc = add_rn(acc, -mul_rn(A, v[0][j & 1]));
                        } else {
                            if (MODE == 1) acc = mul_rn(acc, v[NV][j & 1]);
                            acc = add_rn(acc, -mul_rn(A, v[0][j & 1]));
                            acc = add_rn(acc, -mul_rn(B, v[1][j & 1]));
                            if (D3) acc = add_rn(acc, -mul_rn(C, v[NV - 1][j & 1]));
                        }
                        if (DIV && plain) acc = acc / v[K - 2][j & 1];
                        else if (DIV) acc = quotient<T>(acc, v[K - 2][j & 1], v[K - 1][j & 1], worst);
                        // a lane before or past its line holds 0, whatever its neighbours hold
                        if (edge) acc = at(4 * gi + j) != kOutside ? acc : T(0);
                        prev = res[j] = acc;
                        if (D3) {
                            (j < 3 ? base + (j + 1) * SLOT : next)[lane] = acc;
                            __builtin_amdgcn_wave_barrier();
                            // the group's four slots hold steps 4 gi - 1 .. 4 gi + 2
                            if (j == 2) f = base[frow * SLOT + fsrc];
                        }
                        if (FW) vec_store(ys, yoff + (4 * gi + j) * 64 * ES, acc);
                        else vec_store(rs, edge ? at(4 * gi + j) : off0 + dir * (4 * gi + j), acc);
                    }
                };
                // A branch on lanes' values costs a step half its time, so the
                // range of the divisions is looked at once per group, which is
                // then computed again; its faces leave after that.
                if (!slow) steps(false);
                if (DIV && (slow || __builtin_amdgcn_ballot_w64(worst >= Bits<T>::alen))) {
                    prev = prev0;
                    steps(true);
                }
                if (D3) face_store(bs, fdst + static_cast<unsigned>(gi) * 4 * H * ES, f);
                // 2D: the inbox rows lie side by side; the last step's row is
                // row 0 of the next inbox, which nobody reads
                else face_store4(bs, fdst + 4 * gi * ES, res);
                asm volatile("" ::: "memory");
                // every lane the same value: no branch
                __hip_atomic_store(&s_read, gi + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            };
#pragma unroll
            for (int k = 0; k < kAhead; ++k) load(grp[k], k);
            for (int g0 = 0; g0 < ng; g0 += kAhead) {
#pragma unroll
                for (int k = 0; k < kAhead; ++k) {
                    const int gi = g0 + k;
                    if (gi < ng) {
                        if (inside(gi)) group(grp[k], gi, false);
                        else group(grp[k], gi, true);
                    }
                    load(grp[k], gi + kAhead);
                }
            }
        }
        __syncthreads();
    }
}

namespace {

// Row (x, y, z) of the grid: the diagonal's position and the first entry's,
// from the row pointer alone (the pattern has been checked).
struct RowAt {
    int first, diag;
};

template <bool D3>
__device__ __forceinline__ RowAt row_at(const int *row, int i, int x, int y, int z) {
    const int b = row[i];
    return {b, b + (x > 0) + (y > 0) + (D3 && z > 0)};
}

}  // namespace

// Are the rows those of the full 5- / 7-point stencil of the grid?
template <bool D3>
__global__ __launch_bounds__(kBlock) void k_pencil_check(int n, int nx, int ny, int nz, const int *__restrict__ row,
                                                         const int *__restrict__ col, int *bad) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const int x = i % nx, t = i / nx, y = t % ny, z = t / ny;
    const int nxy = nx * ny;
    int p = row[i];
    const int e = row[i + 1];
    bool ok = true;
    auto need = [&](bool there, int c) {
        if (!there) return;
        ok = ok && p < e && col[p] == c;
        ++p;
    };
    need(D3 && z > 0, i - nxy);
    need(y > 0, i - nx);
    need(x > 0, i - 1);
    need(true, i);
    need(x < nx - 1, i + 1);
    need(y < ny - 1, i + nx);
    need(D3 && z < nz - 1, i + nxy);
    if (!ok || p != e) *bad = 1;
}

// The values of one sweep in the order its steps read them: per (pencil,
// step, lane) the entries of the x, y (and z) neighbour, then (DIV) the
// diagonal and its reciprocal; a missing neighbour 0, a slot outside the
// grid 0 with diagonal 1.
template <typename T, bool FW, bool DIV, bool D3>
__global__ __launch_bounds__(kBlock) void k_pencil_fill(int nx, int ny, int nz, int npy, int npz, int ng,
                                                        const int *__restrict__ row, const T *__restrict__ val,
                                                        T *__restrict__ out, int *slow) {
    typedef Shape<D3> S;
    constexpr int NV = S::NV, K = NV + (DIV ? 2 : 0);
    const long long id = blockIdx.x * static_cast<long long>(kBlock) + threadIdx.x;
    if (id >= static_cast<long long>(npy) * npz * ng * 256) return;
    const int lane = id & 63, j = (id >> 6) & 3;
    const long long pg = id >> 8;
    const int gi = pg % ng, pn = static_cast<int>(pg / ng), J = pn % npy, KK = pn / npy;
    const int yl = D3 ? lane & 7 : lane, zl = D3 ? lane >> 3 : 0;
    const int xs = 4 * gi + j - yl - zl;
    const int x = FW ? xs : nx - 1 - xs;
    const int y = FW ? J * S::BY + yl : (npy - J) * S::BY - 1 - yl;
    const int z = !D3 ? 0 : FW ? KK * 8 + zl : (npz - KK) * 8 - 1 - zl;
    T v[K];
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = T(k < NV ? 0 : 1);
    if (xs >= 0 && xs < nx && y < ny && z < nz) {
        const RowAt r = row_at<D3>(row, (z * ny + y) * nx + x, x, y, z);
        int p = FW ? r.diag : r.diag + 1;
        if (FW) {
            if (x > 0) v[0] = val[--p];
            if (y > 0) v[1] = val[--p];
            if (D3 && z > 0) v[NV - 1] = val[--p];
        } else {
            if (x < nx - 1) v[0] = val[p++];
            if (y < ny - 1) v[1] = val[p++];
            if (D3 && z < nz - 1) v[NV - 1] = val[p++];
        }
        if (DIV) {
            const T d = val[r.diag], m = d < T(0) ? -d : d;
            v[K - 2] = d;
            v[K - 1] = T(1) / d;
            if (!(m >= Bits<T>::dlo && m <= Bits<T>::dhi)) *slow = 1;
        }
    }
    T *o = out + ((pg * 2 + (j >> 1)) * K * 64 + lane) * 2 + (j & 1);
#pragma unroll
    for (int k = 0; k < K; ++k) o[k * 128] = v[k];
}

template <typename U>
__global__ __launch_bounds__(kBlock) void k_pencil_sentinel(long long m, U *a, U *b, U v) {
    const long long k = blockIdx.x * static_cast<long long>(kBlock) + threadIdx.x;
    if (k < m) {
        a[k] = v;
        b[k] = v;
    }
}

template <typename T, bool D3>
static int pencil_fill_t(hfh_prec *P) {
    const hfh_csr *A = P->A;
    hfh_pencil &G = P->pen;
    hipStream_t s = P->ctx->stream;
    HFH_HIP(hipMemsetAsync(G.ctl + 64, 0, sizeof(int), s));
    const long long m = static_cast<long long>(G.np) * G.ng * 256;
    const dim3 g(static_cast<unsigned>((m + kBlock - 1) / kBlock));
    const T *v = static_cast<const T *>(A->val);
    T *fv = static_cast<T *>(G.fval), *bv = static_cast<T *>(G.bval);
    if (P->kind == HFH_PREC_ILU0)
        hipLaunchKernelGGL((k_pencil_fill<T, true, false, D3>), g, dim3(kBlock), 0, s, G.nx, G.ny, G.nz, G.npy, G.npz,
                           G.ng, A->row, v, fv, G.ctl + 64);
    else
        hipLaunchKernelGGL((k_pencil_fill<T, true, true, D3>), g, dim3(kBlock), 0, s, G.nx, G.ny, G.nz, G.npy, G.npz,
                           G.ng, A->row, v, fv, G.ctl + 64);
    hipLaunchKernelGGL((k_pencil_fill<T, false, true, D3>), g, dim3(kBlock), 0, s, G.nx, G.ny, G.nz, G.npy, G.npz,
                       G.ng, A->row, v, bv, G.ctl + 64);
    return launch_check("k_pencil_fill");
}

int pencil_fill(hfh_prec *P) {
    if (P->pen.np == 0) return HFH_OK;
    if (P->dtype == HFH_F64) return P->pen.nz > 1 ? pencil_fill_t<double, true>(P) : pencil_fill_t<double, false>(P);
    return P->pen.nz > 1 ? pencil_fill_t<float, true>(P) : pencil_fill_t<float, false>(P);
}

int pencil_build(hfh_prec *P, int nx, long long nxy) {
    const hfh_csr *A = P->A;
    const int n = A->nrow;
    hipStream_t s = P->ctx->stream;
    hfh_pencil G;
    G.nx = nx;
    if (nxy) {
        if (n % nxy != 0 || n / nxy < 2) return HFH_OK;
        G.ny = static_cast<int>(nxy / nx);
        G.nz = static_cast<int>(n / nxy);
    } else {
        if (n % nx != 0) return HFH_OK;
        G.ny = n / nx;
        G.nz = 1;
    }
    const bool d3 = G.nz > 1;
    const long long es = static_cast<long long>(A->elem());
    // byte offsets of rows in 32 bits, pencil numbers in 16
    if (n * es > (1LL << 31)) return HFH_OK;
    G.npy = d3 ? (G.ny + 7) / 8 : (G.ny + 63) / 64;
    G.npz = d3 ? (G.nz + 7) / 8 : 1;
    if (G.npy >= (1 << 15) || G.npz >= (1 << 15)) return HFH_OK;
    G.np = G.npy * G.npz;
    // one step past the last lane's: the faces leave one step later
    G.ng = (nx + (d3 ? 15 : 64) + 3) / 4;
    // offsets within a pencil's inbox, results and values in 32 bits
    if (4LL * G.ng * (64 * 5) * es >= (1LL << 30)) return HFH_OK;
    // the skew's idle steps must not dominate the value copies
    const long long slots = 256LL * G.np * G.ng;
    if (slots > 4LL * n) return HFH_OK;
    hfh_ctx *c = P->ctx;
    int rc;
    // no memory for the pencils: the blocks take a part of it
    auto give_up = [&](int code) {
        pencil_free(G);
        return code == HFH_ERR_NOMEM ? static_cast<int>(HFH_OK) : code;
    };
    if ((rc = copy_alloc(c, reinterpret_cast<void **>(&G.ctl), sizeof(int) * 96))) return give_up(rc);
    int bad = 0;
    hipError_t e = hipMemsetAsync(G.ctl, 0, sizeof(int) * 96, s);
    if (e != hipSuccess) return give_up(hip_fail(e, "hipMemsetAsync"));
    const dim3 gc((n + kBlock - 1) / kBlock);
    if (d3)
        hipLaunchKernelGGL(k_pencil_check<true>, gc, dim3(kBlock), 0, s, n, G.nx, G.ny, G.nz, A->row, A->col, G.ctl + 80);
    else
        hipLaunchKernelGGL(k_pencil_check<false>, gc, dim3(kBlock), 0, s, n, G.nx, G.ny, G.nz, A->row, A->col, G.ctl + 80);
    if ((rc = launch_check("k_pencil_check"))) return give_up(rc);
    e = hipMemcpyAsync(&bad, G.ctl + 80, sizeof(int), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return give_up(hip_fail(e, "pencil check"));
    if (bad) return give_up(HFH_OK);
    // pencils by diagonal J + K: ascending tickets respect the dependencies
    std::vector<int> order;
    order.reserve(G.np);
    for (int d = 0; d <= G.npy + G.npz - 2; ++d)
        for (int k = std::max(0, d - G.npy + 1); k <= std::min(d, G.npz - 1); ++k) order.push_back((d - k) | (k << 16));
    const int nv = d3 ? 3 : 2, kf = nv + (P->kind == HFH_PREC_ILU0 ? 0 : 2), kb = nv + 2, H = d3 ? 16 : 1;
    const long long nbox = static_cast<long long>(G.np) * G.ng * 4 * H;
    const size_t ysize = static_cast<size_t>(es) * G.np * (4 * G.ng + 4) * 64;
    if ((rc = copy_alloc(c, reinterpret_cast<void **>(&G.order), sizeof(int) * G.np)) ||
        (rc = copy_alloc(c, &G.fval, static_cast<size_t>(es * slots * kf))) ||
        (rc = copy_alloc(c, &G.bval, static_cast<size_t>(es * slots * kb))) || (rc = copy_alloc(c, &G.y, ysize)) ||
        (rc = copy_alloc(c, &G.fbox, static_cast<size_t>(es * nbox))) || (rc = copy_alloc(c, &G.bbox, static_cast<size_t>(es * nbox))))
        return give_up(rc);
    e = hipMemcpyAsync(G.order, order.data(), sizeof(int) * G.np, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipMemsetAsync(G.y, 0, ysize, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return give_up(hip_fail(e, "pencil order"));
    const dim3 gb(static_cast<unsigned>((nbox + kBlock - 1) / kBlock));
    if (A->dtype == HFH_F64)
        hipLaunchKernelGGL(k_pencil_sentinel<unsigned long long>, gb, dim3(kBlock), 0, s, nbox,
                           (unsigned long long *)G.fbox, (unsigned long long *)G.bbox, Bits<double>::sentinel);
    else
        hipLaunchKernelGGL(k_pencil_sentinel<unsigned>, gb, dim3(kBlock), 0, s, nbox, (unsigned *)G.fbox,
                           (unsigned *)G.bbox, Bits<float>::sentinel);
    if ((rc = launch_check("k_pencil_sentinel"))) return give_up(rc);
    P->pen = G;
    return pencil_fill(P);
}

void pencil_free(hfh_pencil &G) {
    void *bufs[] = {G.order, G.fval, G.bval, G.y, G.fbox, G.bbox, G.ctl};
    for (void *b : bufs)
        if (b) (void)hipFree(b);
    G = hfh_pencil();
}

template <typename T, int FW, int BW>
static int pencil_apply_t(hfh_prec *P, const T *in, T *out, const int *done) {
    const hfh_pencil &G = P->pen;
    hipStream_t s = P->ctx->stream;
    const int ncu = std::max(P->ctx->num_cu, 1);
    const int grid = std::min(G.np, ncu * (P->sf_waves > 0 ? P->sf_waves : 4));
    PencilArgs<T> a{G.nx, G.ny, G.nz, G.npy, G.npz, G.ng, G.order, (const T *)G.fval, (T *)G.y, in, nullptr,
                    (T *)G.fbox, (T *)G.bbox, G.ctl, P->sf_ctl + 2, done};
    PencilArgs<T> b = a;
    b.val = static_cast<const T *>(G.bval);
    b.in = nullptr;
    b.out = out;
    b.box = static_cast<T *>(G.bbox);
    b.other_box = static_cast<T *>(G.fbox);
    if (G.nz > 1) {
        hipLaunchKernelGGL((k_pencil<T, FW, true>), dim3(grid), dim3(128), 0, s, a);
        hipLaunchKernelGGL((k_pencil<T, BW, true>), dim3(grid), dim3(128), 0, s, b);
    } else {
        hipLaunchKernelGGL((k_pencil<T, FW, false>), dim3(grid), dim3(128), 0, s, a);
        hipLaunchKernelGGL((k_pencil<T, BW, false>), dim3(grid), dim3(128), 0, s, b);
    }
    return launch_check("k_pencil");
}

int pencil_apply(hfh_prec *P, const void *in, void *out, const int *done) {
    if (P->dtype == HFH_F64)
        return P->kind == HFH_PREC_ILU0 ? pencil_apply_t<double, 2, 3>(P, (const double *)in, (double *)out, done)
                                        : pencil_apply_t<double, 0, 1>(P, (const double *)in, (double *)out, done);
    return P->kind == HFH_PREC_ILU0 ? pencil_apply_t<float, 2, 3>(P, (const float *)in, (float *)out, done)
                                    : pencil_apply_t<float, 0, 1>(P, (const float *)in, (float *)out, done);
}

}  // namespace hfh

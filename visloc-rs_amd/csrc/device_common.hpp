// device_common.hpp — device helpers shared by the kernel files: XCD-aware
// tile mapping, fixed-order wave / work-group reductions, compensated sums
// and the small symmetric-block algebra of the Schur path.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

#include "kernels.hpp"

namespace vba {
namespace {

// Work-groups are dispatched round-robin over the 8 XCDs. Give XCD k a
// contiguous range of tiles so that neighbouring cameras, which share
// landmarks, share that XCD's L2.
__device__ __forceinline__ int xcd_tile(int bid, int n) {
    const int per = (n + 7) >> 3;
    return (bid & 7) * per + (bid >> 3);
}
inline int xcd_grid(int n) { return ((n + 7) >> 3) << 3; }

// Float offsets of G0..G3 and of G4, G5 of the position with index pp in the
// lane-major FP32 G copy (its layout is described with kG32Chunk).
static_assert(kTileEdges == 256 && kG32Chunk == 6 * kTileEdges, "lane-major G chunk of one tile");
__device__ __forceinline__ size_t g32_off4(int pp) {
    return (size_t)(pp >> 8) * kG32Chunk + (pp & 3) * 384 + ((pp & 255) >> 2) * 4;
}
__device__ __forceinline__ size_t g32_off2(int pp) {
    return (size_t)(pp >> 8) * kG32Chunk + (pp & 3) * 384 + 256 + ((pp & 255) >> 2) * 2;
}
inline int blocks_for(int n, int per) { return (n + per - 1) / per; }

__device__ __forceinline__ double from_halves(unsigned lo, unsigned hi) {
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// The value of the partner lane under DPP control CTRL (within a row).
template <int CTRL>
__device__ __forceinline__ double dpp_partner(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)b, CTRL, 0xf, 0xf, false);
    const unsigned hi = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), CTRL, 0xf, 0xf, false);
    return from_halves(lo, hi);
}

// One halving step of wave_sum36: the lane and its partner sum a where the
// lane's `upper` is false and b where it is true.
template <int CTRL>
__device__ __forceinline__ double halve_dpp(double a, double b, bool upper) {
    return (upper ? b : a) + dpp_partner<CTRL>(upper ? a : b);
}
__device__ __forceinline__ double halve_rows(double a, double b) {
    const unsigned long long x = (unsigned long long)__double_as_longlong(a),
                             y = (unsigned long long)__double_as_longlong(b);
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
    return from_halves(lo[0], hi[0]) + from_halves(lo[1], hi[1]);
}
__device__ __forceinline__ double halve_wave(double a, double b) {
    const unsigned long long x = (unsigned long long)__double_as_longlong(a),
                             y = (unsigned long long)__double_as_longlong(b);
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
    return from_halves(lo[0], hi[0]) + from_halves(lo[1], hi[1]);
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    return v;
}
template <typename T>
__device__ __forceinline__ T wave_max(T v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_down(v, off, 64));
    return v;
}

// Sum N values over an NT-thread work-group; the result is valid in thread 0
// and the order of additions is fixed. lds must hold (NT/64)*N values.
template <int NT, typename T, int N>
__device__ __forceinline__ void block_sum(T (&v)[N], T* lds) {
    constexpr int NW = NT / 64;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = wave_sum(v[i]);
    if (lane == 0) {
#pragma unroll
        for (int i = 0; i < N; ++i) lds[wave * N + i] = v[i];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            T s = lds[i];
            for (int w = 1; w < NW; ++w) s += lds[w * N + i];
            v[i] = s;
        }
    }
    __syncthreads();
}
// Sums of N values over an NT-thread work-group, value i to out[i], with
// block_sum's additions in block_sum's order (so the same bits) but lane moves
// in the VALU and half as many values after each of the first two steps:
// lanes pair i with i + 32 and i + 16 by permlane swaps, one lane of a pair
// keeping one half of the values, then i + 8, 4, 2, 1 by row rotations. With
// 27 values, 147 VALU instructions a wave where shuffles take 324 LDS ones.
// lds must hold (NT / 64) * 4 * ceil(N / 4) values.
template <int NT, int N>
__device__ __forceinline__ void block_sum_out(const double (&v)[N], double* lds, double* out) {
    constexpr int NW = NT / 64, H = (N + 1) / 2, Q = (H + 1) / 2;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double a[H], b[Q];
#pragma unroll
    for (int i = 0; i < H; ++i) a[i] = halve_wave(v[i], i + H < N ? v[i + H] : 0.0);
#pragma unroll
    for (int i = 0; i < Q; ++i) {
        b[i] = halve_rows(a[i], i + Q < H ? a[i + Q] : 0.0);
        b[i] = b[i] + dpp_partner<0x128>(b[i]);  // row_ror:8
        b[i] = b[i] + dpp_partner<0x124>(b[i]);  // row_ror:4
        b[i] = b[i] + dpp_partner<0x122>(b[i]);  // row_ror:2
        b[i] = b[i] + dpp_partner<0x121>(b[i]);  // row_ror:1
    }
    // row r of the wave holds values H (r >> 1) + Q (r & 1) + i
    if ((lane & 15) == 0)
#pragma unroll
        for (int i = 0; i < Q; ++i) lds[(4 * wave + (lane >> 4)) * Q + i] = b[i];
    __syncthreads();
    if ((int)threadIdx.x < N) {
        const int i = threadIdx.x, h = i >= H, r = i - h * H, q = r >= Q;
        const double* p = lds + (2 * h + q) * Q + (r - q * Q);
        double s = p[0];
        for (int w = 1; w < NW; ++w) s += p[4 * w * Q];
        out[i] = s;
    }
}
// Sum broadcast to every thread.
template <int NT, typename T, int N>
__device__ __forceinline__ void block_sum_all(T (&v)[N], T* lds) {
    block_sum<NT, T, N>(v, lds);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int i = 0; i < N; ++i) lds[i] = v[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = lds[i];
    __syncthreads();
}
template <int NT>
__device__ __forceinline__ double block_max(double v, double* lds) {
    constexpr int NW = NT / 64;
    v = wave_max(v);
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = lds[0];
        for (int w = 1; w < NW; ++w) m = fmax(m, lds[w]);
        v = m;
    }
    __syncthreads();
    return v;
}

// One thread posts a value of its own: the number becomes visible to the host
// after the value (a system-scope release).
template <typename T>
__device__ __forceinline__ void post_mail(const Post<T>& post, const T& value) {
    if (!post.slot) return;
    post.slot->value = value;
    __threadfence_system();
    __hip_atomic_store(&post.slot->seq, post.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Neumaier compensated pair (sum, compensation) and its exact-order merge.
struct CSum {
    double s, c;
};
__device__ __forceinline__ void csum_add(CSum& a, double x) {
    double t = a.s + x;
    if (fabs(a.s) >= fabs(x)) a.c += (a.s - t) + x;
    else a.c += (x - t) + a.s;
    a.s = t;
}
__device__ __forceinline__ CSum csum_merge(CSum a, CSum b) {
    CSum r;
    r.s = a.s + b.s;
    double bp = r.s - a.s;
    double e = (a.s - (r.s - bp)) + (b.s - bp);
    r.c = a.c + b.c + e;
    return r;
}

// Compensated sum over an NT-thread work-group as a pairwise tree over the
// thread index (valid in thread 0): the order does not depend on NT for
// leaves that are zero from some thread on, so a window's cost is the same
// summed by 256 threads in a batch and by 1,024 alone. (A fold over the
// threads in one thread is up to 1,024 dependent merges, 26 to 40 us.)
template <int NT>
__device__ __forceinline__ CSum block_csum(CSum a, double (*lds)[2]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const CSum o{__shfl_down(a.s, off, 64), __shfl_down(a.c, off, 64)};
        if ((lane & (2 * off - 1)) == 0) a = csum_merge(a, o);
    }
    if (lane == 0) {
        lds[wave][0] = a.s;
        lds[wave][1] = a.c;
    }
    __syncthreads();
    if (wave == 0) {
        constexpr int NW = NT / 64;
        a = lane < NW ? CSum{lds[lane][0], lds[lane][1]} : CSum{0.0, 0.0};
#pragma unroll
        for (int off = 1; off < NW; off <<= 1) {
            const CSum o{__shfl_down(a.s, off, 64), __shfl_down(a.c, off, 64)};
            if ((lane & (2 * off - 1)) == 0) a = csum_merge(a, o);
        }
    }
    __syncthreads();
    return a;
}

// Packed upper-triangle index of a symmetric 6x6.
__host__ __device__ constexpr int up6(int i, int j) { return i * 6 - i * (i - 1) / 2 + (j - i); }

// Accumulate s * [[A, -A K], [K A, -K A K]] (upper triangle) with K = [X]x,
// A symmetric (a00 a01 a02 a11 a12 a22).
template <typename T>
__device__ __forceinline__ void add_schur_block(const T A[6], const T X[3], T s, T out[21]) {
    const T a[9] = {A[0], A[1], A[2], A[1], A[3], A[4], A[2], A[4], A[5]};
    const T K[9] = {T(0), -X[2], X[1], X[2], T(0), -X[0], -X[1], X[0], T(0)};
    T AK[9], KAK[9];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) AK[3 * i + j] = a[3 * i] * K[j] + a[3 * i + 1] * K[3 + j] + a[3 * i + 2] * K[6 + j];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) KAK[3 * i + j] = K[3 * i] * AK[j] + K[3 * i + 1] * AK[3 + j] + K[3 * i + 2] * AK[6 + j];
    out[up6(0, 0)] += s * a[0];
    out[up6(0, 1)] += s * a[1];
    out[up6(0, 2)] += s * a[2];
    out[up6(1, 1)] += s * a[4];
    out[up6(1, 2)] += s * a[5];
    out[up6(2, 2)] += s * a[8];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) out[up6(i, 3 + j)] -= s * AK[3 * i + j];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = i; j < 3; ++j) out[up6(3 + i, 3 + j)] -= s * KAK[3 * i + j];
}

// y = sym(A) x for packed symmetric 3x3.
template <typename T>
__device__ __forceinline__ void sym3_mul(const T A[6], const T x[3], T y[3]) {
    y[0] = A[0] * x[0] + A[1] * x[1] + A[2] * x[2];
    y[1] = A[1] * x[0] + A[3] * x[1] + A[4] * x[2];
    y[2] = A[2] * x[0] + A[4] * x[1] + A[5] * x[2];
}
// y = sym(U) x for packed symmetric 6x6.
__device__ __forceinline__ void sym6_mul(const double* U, const double* x, double* y) {
#pragma unroll
    for (int i = 0; i < 6; ++i) {
        double s = 0.0;
#pragma unroll
        for (int j = 0; j < 6; ++j) s += U[i <= j ? up6(i, j) : up6(j, i)] * x[j];
        y[i] = s;
    }
}

// Sums of 36 values over a wave, one sum per lane: a lane of each pair keeps
// half of the values and takes the partner's part of them (halves of the
// wave, row pairs, then mirror and neighbour lanes: 36, 18, 9, 5, 3, 2, 1
// values), in 38 exchanges where a butterfly that leaves every sum in every
// lane takes 216. Fixed order; all lanes must be active. The lane's sum is
// entry wave_entry36(lane); lanes with -1 hold none.
__device__ __forceinline__ double wave_sum36(const double v[36], int lane) {
    double a[18], b[9], c[5], d[3], e[2];
#pragma unroll
    for (int i = 0; i < 18; ++i) a[i] = halve_wave(v[i], v[i + 18]);
#pragma unroll
    for (int i = 0; i < 9; ++i) b[i] = halve_rows(a[i], a[i + 9]);
#pragma unroll
    for (int i = 0; i < 5; ++i) c[i] = halve_dpp<0x140>(b[i], i < 4 ? b[i + 5] : 0.0, lane & 8);  // row_mirror
#pragma unroll
    for (int i = 0; i < 3; ++i) d[i] = halve_dpp<0x141>(c[i], i < 2 ? c[i + 3] : 0.0, lane & 4);  // row_half_mirror
    e[0] = halve_dpp<0x4E>(d[0], d[2], lane & 2);  // quad_perm [2,3,0,1]
    e[1] = halve_dpp<0x4E>(d[1], 0.0, lane & 2);
    return halve_dpp<0xB1>(e[0], e[1], lane & 1);  // quad_perm [1,0,3,2]
}
__device__ __forceinline__ int wave_entry36(int lane) {
    const int t = (lane & 2) + (lane & 1);                 // of 3 (0, 1; 2)
    const int u = ((lane & 4) ? 3 : 0) + t;                // of 5 (0..2; 3, 4)
    const int w = ((lane & 8) ? 5 : 0) + u;                // of 9 (0..4; 5..8)
    if (t > 2 || ((lane & 4) && t > 1) || ((lane & 8) && u > 3)) return -1;
    return ((lane & 32) ? 18 : 0) + ((lane & 16) ? 9 : 0) + w;
}

// The same over the 8 lanes of a group: lane g of it gets entries g, g + 8, ...
// (five of them, or four where g > 3) in s.
__device__ __forceinline__ void octet_sum36(const double v[36], int lane, double s[5]) {
    double a[20], b[10];  // entries 8 m + (0..3 or 4..7), then 8 m + (0, 1 or 2, 3 of those)
#pragma unroll
    for (int i = 0; i < 20; ++i) {
        const int e = 8 * (i / 4) + i % 4;
        a[i] = halve_dpp<0x141>(v[e], e + 4 < 36 ? v[e + 4] : 0.0, lane & 4);  // row_half_mirror
    }
#pragma unroll
    for (int i = 0; i < 10; ++i) b[i] = halve_dpp<0x4E>(a[4 * (i / 2) + i % 2], a[4 * (i / 2) + i % 2 + 2], lane & 2);  // quad_perm [2,3,0,1]
#pragma unroll
    for (int m = 0; m < 5; ++m) s[m] = halve_dpp<0xB1>(b[2 * m], b[2 * m + 1], lane & 1);  // quad_perm [1,0,3,2]
}

// Block b of sum_l W_p V_l^-1 W_q^T over its term list (landmark l, edge of
// p, edge of q), W_p V_l^-1 W_q^T = [[C, -C K], [K C, -K C K]] with
// C = G_p V_l^-1 G_q and K = [X_l]x, by one wave: entry wave_entry36(lane)
// (row-major 6x6) in each lane. Lane t adds terms t, t + 64, ... in order.
//
// A term is a chain of two dependent gathers (its indices, then 168 bytes of
// blocks) and 126 FP64 operations, so what bounds the sum is how many terms
// are in flight: a whole wave per block, the next term's indices loaded with
// this term's blocks, 16-byte loads. Consecutive terms' landmarks and edges
// lie near one another in storage, so the lanes of a gather share lines.
// Eight lanes per block, each walking an eighth of the list, took 594 us for
// the 50-camera circle's 6.4M terms against 103 us here, 821 us for 64 stereo
// windows (longest list about 1,200 terms) against 158 us, and 840 us for
// the 3.5M-observation loop's 27.5M terms, lists in first-met order, against
// 492 us with the lists row by row: that one reads 4.6 GB of blocks through
// L1 and is bound there.
//
// With F32 the sum is of the mixed operator's blocks, its FP32-stored G and the
// V^-1 that it pairs with them: G rounded as it loads gives the same values.
template <bool F32>
__device__ __forceinline__ void schur_block_terms(const DevProblem& P, const DensePairs& D, int b, int lane, int lanes,
                                                  double acc[36]) {
    const double* const Vinv = F32 ? P.VinvM : P.Vinv64;
    auto stored = [](double2 v) { return F32 ? make_double2((float)v.x, (float)v.y) : v; };
#pragma unroll
    for (int i = 0; i < 36; ++i) acc[i] = 0.0;
    const int end = D.block_ptr[b + 1];
    int k = D.block_ptr[b] + lane;
    if (k < end) {
        const int32_t* t = D.terms + 3 * (size_t)k;
        int l = t[0], ep = t[1], eq = t[2];
        while (true) {
            const double2* v2 = (const double2*)(Vinv + 6 * (size_t)l);
            const double2* a2 = (const double2*)(P.Gl64 + 6 * (size_t)ep);
            const double2* b2 = (const double2*)(P.Gl64 + 6 * (size_t)eq);
            const double* X = P.lms + 3 * (size_t)l;
            const double2 v01 = v2[0], v23 = v2[1], v45 = v2[2];
            const double2 p01 = stored(a2[0]), p23 = stored(a2[1]), p45 = stored(a2[2]);
            const double2 q01 = stored(b2[0]), q23 = stored(b2[1]), q45 = stored(b2[2]);
            const double x0 = X[0], x1 = X[1], x2 = X[2];
            k += lanes;
            const int32_t* tn = D.terms + 3 * (size_t)min(k, end - 1);
            l = tn[0];
            ep = tn[1];
            eq = tn[2];
            const double vi[9] = {v01.x, v01.y, v23.x, v01.y, v23.y, v45.x, v23.x, v45.x, v45.y};
            const double gp[9] = {p01.x, p01.y, p23.x, p01.y, p23.y, p45.x, p23.x, p45.x, p45.y};
            const double gq[9] = {q01.x, q01.y, q23.x, q01.y, q23.y, q45.x, q23.x, q45.x, q45.y};
            double T[9], C[9], CK[9];
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int j = 0; j < 3; ++j)
                    T[3 * i + j] = fma(gp[3 * i + 2], vi[6 + j], fma(gp[3 * i + 1], vi[3 + j], gp[3 * i] * vi[j]));
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int j = 0; j < 3; ++j)
                    C[3 * i + j] = fma(T[3 * i + 2], gq[6 + j], fma(T[3 * i + 1], gq[3 + j], T[3 * i] * gq[j]));
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                CK[3 * i] = fma(C[3 * i + 1], x2, -(C[3 * i + 2] * x1));
                CK[3 * i + 1] = fma(C[3 * i + 2], x0, -(C[3 * i] * x2));
                CK[3 * i + 2] = fma(C[3 * i], x1, -(C[3 * i + 1] * x0));
            }
#pragma unroll
            for (int j = 0; j < 3; ++j) {
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    acc[6 * i + j] += C[3 * i + j];
                    acc[6 * i + 3 + j] -= CK[3 * i + j];
                }
                acc[18 + j] += fma(x1, C[6 + j], -(x2 * C[3 + j]));
                acc[24 + j] += fma(x2, C[j], -(x0 * C[6 + j]));
                acc[30 + j] += fma(x0, C[3 + j], -(x1 * C[j]));
                acc[21 + j] -= fma(x1, CK[6 + j], -(x2 * CK[3 + j]));
                acc[27 + j] -= fma(x2, CK[j], -(x0 * CK[6 + j]));
                acc[33 + j] -= fma(x0, CK[3 + j], -(x1 * CK[j]));
            }
            if (k >= end) break;
        }
    }
}

// The block's sum by one wave: entry wave_entry36(lane) (row-major 6x6) in
// each lane.
template <bool F32>
__device__ __forceinline__ double schur_block_wave(const DevProblem& P, const DensePairs& D, int b, int lane) {
    double acc[36];
    schur_block_terms<F32>(P, D, b, lane, 64, acc);
    return wave_sum36(acc, lane);
}

// The block of this wave of a kBlock launch over block_grid(num_blocks), one block per wave, neighbouring blocks
// (which share edges) on one XCD.
__device__ __forceinline__ int block_of_wave(int num_blocks) {
    constexpr int kWaves = kBlock / 64;
    const int wg = xcd_tile(blockIdx.x, (num_blocks + kWaves - 1) / kWaves);
    return __builtin_amdgcn_readfirstlane(wg * kWaves + (int)(threadIdx.x >> 6));
}
inline int block_grid(int num_blocks) { return xcd_grid(blocks_for(num_blocks, kBlock / 64)); }

// 6x6 Cholesky inverse; false for a non-positive or non-finite pivot.
// Every loop is unrolled, so that L and y stay in registers (dynamic
// indexing would put them in scratch memory).
__device__ inline bool cholesky_inverse6(double A[36], double out[36]) {
    double L[36];
#pragma unroll
    for (int i = 0; i < 36; ++i) L[i] = 0.0;
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        double d = A[6 * j + j];
#pragma unroll
        for (int k = 0; k < j; ++k) d -= L[6 * j + k] * L[6 * j + k];
        if (!(d > 0.0) || !isfinite(d)) return false;
        const double ljj = sqrt(d);
        L[6 * j + j] = ljj;
#pragma unroll
        for (int i = j + 1; i < 6; ++i) {
            double s = A[6 * i + j];
#pragma unroll
            for (int k = 0; k < j; ++k) s -= L[6 * i + k] * L[6 * j + k];
            L[6 * i + j] = s / ljj;
        }
    }
#pragma unroll
    for (int c = 0; c < 6; ++c) {
        double y[6];
#pragma unroll
        for (int i = 0; i < 6; ++i) {
            double s = (i == c) ? 1.0 : 0.0;
#pragma unroll
            for (int k = 0; k < i; ++k) s -= L[6 * i + k] * y[k];
            y[i] = s / L[6 * i + i];
        }
#pragma unroll
        for (int i = 5; i >= 0; --i) {
            double s = y[i];
#pragma unroll
            for (int k = i + 1; k < 6; ++k) s -= L[6 * k + i] * y[k];
            y[i] = s / L[6 * i + i];
        }
#pragma unroll
        for (int i = 0; i < 6; ++i) out[6 * i + c] = y[i];
    }
    bool finite = true;
#pragma unroll
    for (int i = 0; i < 36; ++i) finite = finite && isfinite(out[i]);
    return finite;
}

}  // namespace
}  // namespace vba

// explicit_schur.hip — the reduced camera matrix S = U + lambda I - W V^-1 W^T
// assembled explicitly as 6x6 blocks between variable poses that share a
// landmark, and the block-Jacobi PCG of implicit_schur.rs:522-761 run on it.
// The reference states this matrix in its operator tests
// (implicit_schur.rs:831-850, explicit_schur; compared with the implicit
// operator at :952-975 and :1190-1197); here it is a solver of its own: after
// one assembly per LM iteration each PCG product reads 36 values per stored
// block instead of streaming every edge's G.
//
// Assembly: one wave per upper block (an eighth of one where the lists are
// short) sums the block's term list (one term per landmark the two poses share,
// in landmark order) in a fixed order, then writes S_pq and its transpose S_qp.
// Products: four waves per block row, or one where there are many rows, 48 lanes
// of each as 6 rows x 8 column-block groups.
#include <hip/hip_runtime.h>

#include <cmath>

#include "device_common.hpp"
#include "pcg_device.hpp"

namespace vba {

namespace {

// ---------------------------------------------------------------------------
// Structure. Rows are bitmaps over the poses; a block's place in its row is
// the number of set bits before it, and the upper blocks are numbered row by
// row. The term lists come from each row's wave walking the row's edges 64 at
// a time (a lane per edge, its landmark's later poses one by one) and taking
// the next places of the blocks' lists from counters in LDS, the lanes of one
// list in lane order, so the lists have a fixed order. Once per prepared problem; the 26M terms of the 1,200-camera loop
// take 1.7 ms here (first solve 38 ms), against lists built on the host and
// sent (first solve 251 ms).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_explicit_lpose(DevProblem P, ExplicitBuild B) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < P.num_edges) B.lpose[i] = P.s_pose[P.lm_store[i]];
}

// The c-order edges of a pose.
__device__ __forceinline__ void pose_edges(const DevProblem& P, int p, int* begin, int* end) {
    const int t0 = P.cam_tile_ptr[p], t1 = P.cam_tile_ptr[p + 1];
    *begin = t0 < t1 ? P.cam_tiles[t0].begin : 0;
    *end = t0 < t1 ? P.cam_tiles[t1 - 1].end : 0;
}

__global__ __launch_bounds__(kBlock) void k_explicit_rows(DevProblem P, ExplicitBuild B) {
    extern __shared__ uint32_t row[];
    __shared__ int total, upper;
    const int p = blockIdx.x, tid = threadIdx.x;
    const bool var = P.pose_var[p] >= 0;
    for (int w = tid; w < B.nw; w += kBlock) row[w] = 0;
    if (tid == 0) total = upper = 0;
    __syncthreads();
    if (var) {
        if (tid == 0) atomicOr(&row[p >> 5], 1u << (p & 31));
        int begin, end;
        pose_edges(P, p, &begin, &end);
        for (int e = begin + tid; e < end; e += kBlock) {
            const int l = P.edge_lm[e];
            if (P.lm_var[l] < 0) continue;
            const int le = P.lm_edge_ptr[l + 1];
            for (int i = P.lm_edge_ptr[l]; i < le; ++i) {
                const int q = B.lpose[i];
                const uint32_t bit = 1u << (q & 31);
                if (P.pose_var[q] >= 0 && !(row[q >> 5] & bit)) atomicOr(&row[q >> 5], bit);
            }
        }
    }
    __syncthreads();
    for (int w = tid; w < B.nw; w += kBlock) {
        const uint32_t v = row[w];
        B.bits[(size_t)B.nw * p + w] = v;
        const uint32_t up = w > (p >> 5) ? v : w == (p >> 5) ? v >> (p & 31) : 0u;
        if (v) atomicAdd(&total, __popc(v));
        if (up) atomicAdd(&upper, __popc(up));
    }
    __syncthreads();
    if (tid == 0) {
        B.row_count[p] = total;
        B.up_count[p] = upper;
    }
}

// Exclusive sum of n values into out (n + 1), by one work-group.
__global__ __launch_bounds__(1024) void k_explicit_scan(const int32_t* in, int32_t* out, int n) {
    __shared__ int32_t part[1024];
    const int tid = threadIdx.x, per = (n + 1023) / 1024;
    const int b = min(n, tid * per), e = min(n, b + per);
    int32_t s = 0;
    for (int i = b; i < e; ++i) s += in[i];
    part[tid] = s;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        const int32_t v = tid >= off ? part[tid - off] : 0;
        __syncthreads();
        part[tid] += v;
        __syncthreads();
    }
    s = tid > 0 ? part[tid - 1] : 0;
    for (int i = b; i < e; ++i) {
        out[i] = s;
        s += in[i];
    }
    if (tid == 1023) out[n] = s;
}

// One wave per row: columns ascending, the diagonal's place, and for each
// upper block its pair and the full places of S_pq and S_qp.
__global__ __launch_bounds__(kBlock) void k_explicit_cols(DevProblem P, ExplicitBuild B) {
    const int p = blockIdx.x * (kBlock / 64) + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (p >= P.num_pose_slots) return;
    if (P.pose_var[p] < 0) {
        if (lane == 0) B.diag_pos[p] = -1;
        return;
    }
    const uint32_t* bits = B.bits + (size_t)B.nw * p;
    const int row0 = B.row_ptr[p], up0 = B.up_ptr[p], lower = (B.row_ptr[p + 1] - row0) - (B.up_ptr[p + 1] - up0);
    int base = 0;  // set bits before this round's words
    for (int w0 = 0; w0 < B.nw; w0 += 64) {
        const int w = w0 + lane;
        uint32_t v = w < B.nw ? bits[w] : 0u;
        int incl = __popc(v);
        for (int off = 1; off < 64; off <<= 1) {
            const int u = __shfl_up(incl, off, 64);
            if (lane >= off) incl += u;
        }
        int rank = base + incl - __popc(v);
        base += __shfl(incl, 63, 64);
        for (; v; v &= v - 1, ++rank) {
            const int q = 32 * w + __ffs(v) - 1;
            B.col[row0 + rank] = q;
            if (q < p) continue;
            const int ub = up0 + rank - lower;
            B.block_pq[2 * (size_t)ub] = p;
            B.block_pq[2 * (size_t)ub + 1] = q;
            B.block_pos[2 * (size_t)ub] = row0 + rank;
            if (q == p) {
                B.diag_pos[p] = row0 + rank;
                B.block_pos[2 * (size_t)ub + 1] = -1;
            } else {
                const uint32_t* other = B.bits + (size_t)B.nw * q;
                int before = __popc(other[p >> 5] & ((1u << (p & 31)) - 1u));
                for (int x = 0; x < (p >> 5); ++x) before += __popc(other[x]);
                B.block_pos[2 * (size_t)ub + 1] = B.row_ptr[q] + before;
            }
        }
    }
}

// LDS of the two list kernels: the row's words, the set bits before each
// word, and a counter per upper block.
struct RowIndex {
    uint32_t* words;
    int32_t* before;
    int32_t* count;
    int lower;  // columns below the diagonal
    __device__ __forceinline__ int upper_of(int q) const {
        const int w = q >> 5;
        return before[w] + __popc(words[w] & ((1u << (q & 31)) - 1u)) - lower;
    }
};
template <int NT>
__device__ __forceinline__ RowIndex load_row_index(const ExplicitBuild& B, int p, uint32_t* lds, int upper) {
    RowIndex r{lds, (int32_t*)lds + B.nw, (int32_t*)lds + 2 * B.nw, 0};
    for (int w = threadIdx.x; w < B.nw; w += NT) r.words[w] = B.bits[(size_t)B.nw * p + w];
    for (int j = threadIdx.x; j < upper; j += NT) r.count[j] = 0;
    __syncthreads();
    if (threadIdx.x < 64) {
        const int lane = threadIdx.x;
        int base = 0;
        for (int w0 = 0; w0 < B.nw; w0 += 64) {
            const int w = w0 + lane, c = w < B.nw ? __popc(r.words[w]) : 0;
            int incl = c;
            for (int off = 1; off < 64; off <<= 1) {
                const int u = __shfl_up(incl, off, 64);
                if (lane >= off) incl += u;
            }
            if (w < B.nw) r.before[w] = base + incl - c;
            base += __shfl(incl, 63, 64);
        }
    }
    __syncthreads();
    r.lower = r.before[p >> 5] + __popc(r.words[p >> 5] & ((1u << (p & 31)) - 1u));
    return r;
}

// Terms per upper block (into block_ptr) and per row.
__global__ __launch_bounds__(kBlock) void k_explicit_count(DevProblem P, ExplicitBuild B) {
    extern __shared__ uint32_t lds[];
    __shared__ int total;
    const int p = blockIdx.x, tid = threadIdx.x, up0 = B.up_ptr[p], upper = B.up_ptr[p + 1] - up0;
    if (tid == 0) total = 0;
    const RowIndex r = load_row_index<kBlock>(B, p, lds, upper);
    if (upper > 0) {
        int begin, end;
        pose_edges(P, p, &begin, &end);
        for (int e = begin + tid; e < end; e += kBlock) {
            const int l = P.edge_lm[e];
            if (P.lm_var[l] < 0) continue;
            const int le = P.lm_edge_ptr[l + 1];
            for (int i = P.lm_edge_ptr[l]; i < le; ++i) {
                const int q = B.lpose[i];
                if (q >= p && P.pose_var[q] >= 0) atomicAdd(&r.count[r.upper_of(q)], 1);
            }
        }
    }
    __syncthreads();
    for (int j = tid; j < upper; j += kBlock) {
        B.block_ptr[up0 + j] = r.count[j];
        atomicAdd(&total, r.count[j]);
    }
    __syncthreads();
    if (tid == 0) B.row_terms[p] = total;
}

// block_ptr from the counts, then the row's terms in list order. One wave.
__global__ __launch_bounds__(64) void k_explicit_fill(DevProblem P, ExplicitBuild B) {
    extern __shared__ uint32_t lds[];
    const int p = blockIdx.x, lane = threadIdx.x, up0 = B.up_ptr[p], upper = B.up_ptr[p + 1] - up0;
    if (p == P.num_pose_slots - 1 && lane == 0) B.block_ptr[B.up_ptr[p + 1]] = B.term_row[p + 1];
    const RowIndex r = load_row_index<64>(B, p, lds, upper);
    if (upper == 0) return;
    int base = B.term_row[p];
    for (int j0 = 0; j0 < upper; j0 += 64) {
        const int j = j0 + lane, c = j < upper ? B.block_ptr[up0 + j] : 0;
        int incl = c;
        for (int off = 1; off < 64; off <<= 1) {
            const int u = __shfl_up(incl, off, 64);
            if (lane >= off) incl += u;
        }
        if (j < upper) B.block_ptr[up0 + j] = r.count[j] = base + incl - c;
        base += __shfl(incl, 63, 64);
    }
    __syncthreads();
    int begin, end;
    pose_edges(P, p, &begin, &end);
    for (int e0 = begin; e0 < end; e0 += 64) {
        const int e = e0 + lane;
        const int l = e < end ? P.edge_lm[e] : 0;
        const bool on = e < end && P.lm_var[l] >= 0;
        const int ep = e < end ? P.perm_cl[e] : 0;
        const int le = on ? P.lm_edge_ptr[l + 1] : 0;
        int i = on ? P.lm_edge_ptr[l] : 0;
        while (i < le && B.lpose[i] < p) ++i;  // this edge's own place in its landmark
        for (; __any(i < le); ++i) {
            const int q = i < le ? B.lpose[i] : p;
            const bool term = i < le && P.pose_var[q] >= 0;
            const int j = term ? r.upper_of(q) : 0;
            // the lanes whose terms go to this lane's list, by the bits of j
            uint64_t same = __ballot(term);
            for (int bit = 1; bit < upper; bit <<= 1) {
                const uint64_t set = __ballot((j & bit) != 0);
                same &= j & bit ? set : ~set;
            }
            const int rank = __popcll(same & ((1ull << lane) - 1)), first = r.count[j];
            __builtin_amdgcn_wave_barrier();
            if (term && rank == 0) r.count[j] = first + __popcll(same);
            __builtin_amdgcn_wave_barrier();
            if (!term) continue;
            const int t = first + rank;
            B.terms[3 * (size_t)t] = l;
            B.terms[3 * (size_t)t + 1] = ep;
            B.terms[3 * (size_t)t + 2] = P.lm_store[i];
        }
    }
}

// One upper block per kLanes lanes (a wave, or an eighth of one): S_pq =
// [p == q](U_p + lambda I) - sum of its terms, stored row-major at
// block_pos[2b] and transposed at block_pos[2b + 1]. The diagonal block keeps
// its upper triangle and mirrors it, so that it is exactly symmetric.
template <bool F32, int kLanes>
__global__ __launch_bounds__(kBlock, 4) void k_explicit_assemble(DevProblem P, DensePairs D, ExplicitDev X,
                                                                 double lambda) {
    constexpr int kPer = 64 / kLanes;  // blocks a wave
    const int lane = threadIdx.x & 63, wave_block = kPer * block_of_wave((D.num_blocks + kPer - 1) / kPer);
    if (wave_block >= D.num_blocks) return;
    const int b = min(wave_block + lane / kLanes, D.num_blocks - 1);
    double s[5];  // (minus) the sums of entries first, first + 8, ...
    int first, count;
    if constexpr (kLanes == 64) {
        s[0] = -schur_block_wave<F32>(P, D, b, lane);
        first = wave_entry36(lane);
        count = first < 0 ? 0 : 1;
    } else {
        double acc[36];
        schur_block_terms<F32>(P, D, b, lane % kLanes, kLanes, acc);
        octet_sum36(acc, lane, s);
#pragma unroll
        for (int i = 0; i < 5; ++i) s[i] = -s[i];
        first = lane % kLanes;
        count = wave_block + lane / kLanes < D.num_blocks ? (first > 3 ? 4 : 5) : 0;
    }
    const int sp = D.block_pq[2 * b], sq = D.block_pq[2 * b + 1];
    const int pos = X.block_pos[2 * b], other = X.block_pos[2 * b + 1];
#pragma unroll
    for (int e = 0; e < (kLanes == 64 ? 1 : 5); ++e) {
        if (e >= count) break;
        const int idx = first + 8 * e, i = idx / 6, j = idx % 6, tidx = 6 * j + i;
        double v = s[e];
        int pos_t = other;
        if (sp == sq) {
            if (i > j) continue;
            v = P.U[21 * (size_t)sp + up6(i, j)] + (i == j && lambda > 0.0 ? lambda : 0.0) + v;
            pos_t = i < j ? pos : -1;
        }
        X.S64[36 * (size_t)pos + idx] = v;
        if (X.S32) X.S32[36 * (size_t)pos + idx] = (float)v;
        if (pos_t >= 0) {
            X.S64[36 * (size_t)pos_t + tidx] = v;
            if (X.S32) X.S32[36 * (size_t)pos_t + tidx] = (float)v;
        }
    }
}

// Block-Jacobi inverse of each variable pose's diagonal block.
__global__ __launch_bounds__(kBlock) void k_explicit_precond(DevProblem P, ExplicitDev X) {
    const int p = blockIdx.x * kBlock + threadIdx.x;
    if (p >= P.num_pose_slots) return;
    double* out = P.Minv + 36 * (size_t)p;
    const int pos = X.diag_pos[p];
    if (pos < 0) {
        for (int i = 0; i < 36; ++i) out[i] = 0.0;
        return;
    }
    double M[36], inv[36];
    for (int i = 0; i < 36; ++i) M[i] = X.S64[36 * (size_t)pos + i];
    if (!cholesky_inverse6(M, inv)) {
        P.scalars->precond_failed = 1;
        for (int i = 0; i < 36; ++i) out[i] = 0.0;
        return;
    }
    for (int i = 0; i < 36; ++i) out[i] = inv[i];
}

// A block row's product by kWaves waves. Lane 8i + g of wave w takes row i of
// the blocks 8 w + g, 8 (w + kWaves) + g, ... of the row, kBlocks of them at a
// time.
//
// Few rows (explicit_group_rows): the matrix is small (288 bytes a block; a
// loop's 60 blocks a row make 14 MB for 800 poses) and stays in the L2s, so the
// product is bound by its chain of dependent loads (row bounds, columns,
// vectors) and by the launch. Four waves a row and a block a lane and pass make
// two passes of a row of 64 blocks, and the inputs of the PCG scalars load with
// the first one. (Two blocks a lane: more registers and the same time; eight
// waves a row: 8 to 20 % slower.) One wave a row, four blocks at a time after
// the scalars, took 8.9 us at 210 poses (FP64 blocks) and 11.1 us at 800 (FP32
// blocks) by the trace; 5.6 and 8.7 us here.
//
// Many rows fill the device by themselves, and every wave derives the PCG
// scalars from all partials, so a row gets one wave, two blocks a lane, its
// scalars first (fewer registers), and a work-group four rows (half the
// partials that the step kernel's waves sum). Product and step with FP64
// blocks, four waves a row against this: 24.1 and 23.1 us at 2,000 poses, 28.0
// and 29.8 at 2,500, 30.6 and 30.1 at 3,000, 36.0 and 35.0 at 4,000, 58.3 and
// 53.7 at 8,000, 96 and 75 at 16,000 with 56 blocks a row.
template <int kWaves, int kBlocks, int kRows, bool kEarly>
struct RowSplit {
    static constexpr int waves = kWaves, blocks = kBlocks, rows = kRows, threads = 64 * kWaves * kRows;
    static constexpr bool early = kEarly;      // the PCG scalars before the row's loads
    static constexpr int stride = 8 * kWaves;  // blocks apart that a lane takes
};
using FewRows = RowSplit<4, 1, kExplicitFewRows, false>;
using ManyRows = RowSplit<1, 2, kExplicitManyRows, true>;

// Work-groups' rows: neighbouring rows on one XCD, whose L2 then holds their
// part of the matrix and of the vectors they share.
template <typename Split>
__device__ __forceinline__ int row_groups(const DevProblem& P) {
    return (P.num_pose_slots + Split::rows - 1) / Split::rows;
}

template <typename TS, int kBlocks>
struct RowLoads {
    int q[kBlocks];
    TS s[kBlocks][6];
};
// Blocks t, t + stride, ... of the row (clamped to its last block, whose
// product the caller drops) and their columns.
template <typename Split, typename TS>
__device__ __forceinline__ void load_row_blocks(const ExplicitDev& X, const TS* __restrict__ S, int t, int last, int i,
                                                RowLoads<TS, Split::blocks>* r) {
#pragma unroll
    for (int u = 0; u < Split::blocks; ++u) {
        const int tc = max(min(t + Split::stride * u, last), 0);
        r->q[u] = X.col[tc];
        load6(S + 36 * (size_t)tc + 6 * i, r->s[u]);
    }
}

// Sums over the 8 lanes of a group in every one of them.
__device__ __forceinline__ double group8_sum(double v) {
    v = v + dpp_partner<0xB1>(v);      // quad_perm [1,0,3,2]
    v = v + dpp_partner<0x4E>(v);      // quad_perm [2,3,0,1]
    return v + dpp_partner<0x141>(v);  // row_half_mirror
}

// (S v)_p for v = v1 + beta v2 (v2 may be null) over blocks t, t + stride, ...
// from the loaded ones on; `beta` is called once the vectors' loads are out
// and false ends the launch (the same in every wave). The row's sum of row
// component c is valid in lanes c < 6 of the row's wave 0.
template <typename Split, typename TS, typename Beta>
__device__ __forceinline__ bool row_product(const ExplicitDev& X, const TS* __restrict__ S, int begin, int end,
                                            const double* __restrict__ v1, const double* __restrict__ v2, Beta beta,
                                            int lane, int wave, double (*sum)[8], double* y) {
    const int i = min(lane >> 3, 5), g = lane & 7, last = end - 1;
    int base = begin + 8 * wave, t = base + g;
    RowLoads<TS, Split::blocks> r;
    double acc = 0.0, bt = 0.0;
    if (Split::early && !beta(&bt)) return false;
    load_row_blocks<Split>(X, S, t, last, i, &r);
    for (bool first = true;; first = false) {
        double v[Split::blocks][6], w[Split::blocks][6];
#pragma unroll
        for (int u = 0; u < Split::blocks; ++u) {
            load6(v1 + 6 * (size_t)r.q[u], v[u]);
            if (v2) load6(v2 + 6 * (size_t)r.q[u], w[u]);
        }
        if (!Split::early && first && !beta(&bt)) return false;
#pragma unroll
        for (int u = 0; u < Split::blocks; ++u)
            if (t + Split::stride * u < end)
#pragma unroll
                for (int j = 0; j < 6; ++j)
                    acc = fma((double)r.s[u][j], v2 ? fma(bt, w[u][j], v[u][j]) : v[u][j], acc);
        base += Split::stride * Split::blocks;
        t = base + g;
        if (base >= end) break;  // no lane of the wave has a block left
        load_row_blocks<Split>(X, S, t, last, i, &r);
    }
    acc = group8_sum(acc);
    if (lane < 48 && g == 0) sum[wave][i] = acc;
    __syncthreads();
    *y = 0.0;
    if (wave == 0 && lane < 6) {
        *y = sum[0][lane];
#pragma unroll
        for (int w = 1; w < Split::waves; ++w) *y += sum[w][lane];
    }
    return true;
}

// Sums (over lanes 0..5 of each row's wave 0, then over the work-group's
// rows) into the work-group's partial.
template <typename Split>
__device__ __forceinline__ void rows_to_partial(double v0, double v1, bool head, int row, double (*lds)[2],
                                                double* out) {
    if (head) {
        v0 = wave_sum(v0);
        v1 = wave_sum(v1);
        if ((threadIdx.x & 63) == 0) {
            lds[row][0] = v0;
            lds[row][1] = v1;
        }
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        double a = lds[0][threadIdx.x];
        for (int r = 1; r < Split::rows; ++r) a += lds[r][threadIdx.x];
        out[threadIdx.x] = a;
    }
}

// d_new = z + beta d_old and q = S d_new; d.q partials per work-group. The
// work-groups first derive the iteration's scalars.
template <typename TS, typename Split>
__global__ __launch_bounds__(Split::threads) void k_pcg_explicit(DevProblem P, ExplicitDev X, const TS* __restrict__ S,
                                                              const double* __restrict__ d_old,
                                                              double* __restrict__ d_new, int k, int fresh) {
    __shared__ double sum[Split::rows][Split::waves][8], lds[Split::rows][2];
    const PrologueIn pin = pcg_prologue_load(P, k);
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int row = wv / Split::waves, wave = wv % Split::waves;
    const int group = xcd_tile(blockIdx.x, row_groups<Split>(P)), p = group * Split::rows + row;
    if (group >= row_groups<Split>(P)) return;
    const int pc = min(p, P.num_pose_slots - 1);
    const bool var = p < P.num_pose_slots && P.pose_var[pc] >= 0;
    const size_t kk = 6 * (size_t)pc + (lane < 6 ? lane : 0);
    const double zc = P.z[kk], dc0 = d_old[kk];
    double beta = 0.0, y;
    // (the first product of a solve or restart has d = z and d_old = 0, so
    // the term that beta = 0 multiplies is finite)
    if (!row_product<Split, TS>(X, S, X.row_ptr[pc], X.row_ptr[pc + 1], P.z, d_old,
                         [&](double* b) {
                             const bool go = pcg_prologue_finish(P, k, fresh, pin, &beta);
                             *b = beta;
                             return go;
                         },
                         lane, wave, sum[row], &y))
        return;
    double dq = 0.0;
    if (var && wave == 0 && lane < 6) {
        const double dc = fma(beta, dc0, zc);
        d_new[kk] = dc;
        P.q[kk] = y;
        dq = dc * y;
    }
    rows_to_partial<Split>(dq, 0.0, wave == 0, row, lds, P.bpart + 2 * (size_t)group);
}

// r_t = b - S64 x; with restart r = r_t, z = M^-1 r_t, d = 0. Partials
// (r_t.r_t, r_t.z) per work-group, as the implicit operator's check.
template <typename Split>
__global__ __launch_bounds__(Split::threads) void k_explicit_true_pose(DevProblem P, ExplicitDev X, int restart) {
    __shared__ double sum[Split::rows][Split::waves][8], lds[Split::rows][2];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int row = wv / Split::waves, wave = wv % Split::waves;
    const int group = xcd_tile(blockIdx.x, row_groups<Split>(P)), p = group * Split::rows + row;
    if (group >= row_groups<Split>(P)) return;
    const int pc = min(p, P.num_pose_slots - 1);
    const bool var = p < P.num_pose_slots && P.pose_var[pc] >= 0;
    const int c = lane < 6 ? lane : 0;
    const size_t k = 6 * (size_t)pc + c;
    const double bc = P.b[k];
    double y;
    (void)row_product<Split, double>(X, X.S64, X.row_ptr[pc], X.row_ptr[pc + 1], P.x, nullptr, [](double*) { return true; },
                              lane, wave, sum[row], &y);
    double v[2] = {0.0, 0.0};
    if (var && wave == 0) {
        const double rt = bc - y;
        double zc = 0.0;
        if (restart) zc = pose_minv(P, p, c, 0, rt, lane < 6);
        if (lane < 6) {
            v[0] = rt * rt;
            if (restart) {
                P.r[k] = rt;
                P.z[k] = zc;
                P.d[k] = 0.0;
                v[1] = rt * zc;
            }
        }
    }
    rows_to_partial<Split>(v[0], v[1], wave == 0, row, lds, P.bpart + 2 * (size_t)group);
}

}  // namespace

void launch_explicit_rows(const DevProblem& P, const ExplicitBuild& B, hipStream_t s) {
    const int n = P.num_pose_slots;
    hipLaunchKernelGGL(k_explicit_lpose, dim3(blocks_for(P.num_edges, kBlock)), dim3(kBlock), 0, s, P, B);
    hipLaunchKernelGGL(k_explicit_rows, dim3(n), dim3(kBlock), (size_t)B.nw * sizeof(uint32_t), s, P, B);
    hipLaunchKernelGGL(k_explicit_scan, dim3(1), dim3(1024), 0, s, (const int32_t*)B.row_count, B.row_ptr, n);
    hipLaunchKernelGGL(k_explicit_scan, dim3(1), dim3(1024), 0, s, (const int32_t*)B.up_count, B.up_ptr, n);
}

void launch_explicit_lists(const DevProblem& P, const ExplicitBuild& B, int32_t max_upper, hipStream_t s) {
    const int n = P.num_pose_slots;
    const size_t lds = (2 * (size_t)B.nw + max_upper) * sizeof(int32_t);
    hipLaunchKernelGGL(k_explicit_cols, dim3(blocks_for(n, kBlock / 64)), dim3(kBlock), 0, s, P, B);
    hipLaunchKernelGGL(k_explicit_count, dim3(n), dim3(kBlock), lds, s, P, B);
    hipLaunchKernelGGL(k_explicit_scan, dim3(1), dim3(1024), 0, s, (const int32_t*)B.row_terms, B.term_row, n);
    hipLaunchKernelGGL(k_explicit_fill, dim3(n), dim3(64), lds, s, P, B);
}

void launch_explicit_assemble(const DevProblem& P, const DensePairs& D, const ExplicitDev& X, bool f32, double lambda,
                              hipStream_t s) {
    if (!D.num_blocks) return;
    const auto kernel = X.short_lists ? (f32 ? k_explicit_assemble<true, 8> : k_explicit_assemble<false, 8>)
                                      : (f32 ? k_explicit_assemble<true, 64> : k_explicit_assemble<false, 64>);
    const int waves = X.short_lists ? blocks_for(D.num_blocks, 8) : D.num_blocks;
    hipLaunchKernelGGL(kernel, dim3(block_grid(waves)), dim3(kBlock), 0, s, P, D, X, lambda);
}

void launch_explicit_precond(const DevProblem& P, const ExplicitDev& X, hipStream_t s) {
    hipLaunchKernelGGL(k_explicit_precond, dim3(blocks_for(P.num_pose_slots, kBlock)), dim3(kBlock), 0, s, P, X);
}

namespace {
template <typename TS>
void launch_product(const DevProblem& P, const ExplicitDev& X, const TS* S, const double* d_old, double* d_new,
                    int32_t pcg_iter, int32_t fresh, hipStream_t s) {
    const int rows = explicit_group_rows(P.num_pose_slots);
    const bool few = rows == FewRows::rows;
    const auto kernel = few ? k_pcg_explicit<TS, FewRows> : k_pcg_explicit<TS, ManyRows>;
    hipLaunchKernelGGL(kernel, dim3(xcd_grid(blocks_for(P.num_pose_slots, rows))),
                       dim3(few ? FewRows::threads : ManyRows::threads), 0, s, P, X, S, d_old, d_new, (int)pcg_iter,
                       (int)fresh);
}
}  // namespace

void launch_pcg_explicit(const DevProblem& P, const ExplicitDev& X, bool fp32, const double* d_old, double* d_new,
                         int32_t pcg_iter, int32_t fresh, hipStream_t s) {
    if (fp32) launch_product(P, X, (const float*)X.S32, d_old, d_new, pcg_iter, fresh, s);
    else launch_product(P, X, (const double*)X.S64, d_old, d_new, pcg_iter, fresh, s);
}

void launch_explicit_true_residual(const DevProblem& P, const ExplicitDev& X, int32_t restart,
                                   const Post<PcgState>& post, hipStream_t s) {
    const int rows = explicit_group_rows(P.num_pose_slots);
    const bool few = rows == FewRows::rows;
    const auto kernel = few ? k_explicit_true_pose<FewRows> : k_explicit_true_pose<ManyRows>;
    hipLaunchKernelGGL(kernel, dim3(xcd_grid(blocks_for(P.num_pose_slots, rows))),
                       dim3(few ? FewRows::threads : ManyRows::threads), 0, s, P, X, (int)restart);
    launch_pcg_true_finish(P, restart, post, s);
}

}  // namespace vba

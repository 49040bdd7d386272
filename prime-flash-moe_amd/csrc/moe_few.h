// bf16 kernels for a handful of (token, expert) pairs, gfx950: one token or a few through the layer.
//
// What bounds these calls is not a rate but a chain of latencies: launch, ids, weights, and what lies behind the last weight.
// The streaming kernels (moe_stream.h) put a ring of LDS stages, a barrier per slab and a sum over eight waves into that chain,
// a job of theirs is 131 KB (one token on 8 of 128 experts gives every other CU twice the bytes of its neighbour), and
// finalize is a launch of its own.  Here weights go straight into registers, no matrix instruction is involved, and the
// routing weights are applied where the output column is computed.  One token on 8 of 128 experts (K 2048, N 1536): up kernel
// 12.0 -> 9.4 us (5.4 TB/s), down kernel and finalize 11.3 -> 8.1.  A block's ids and expert are requested beside the length of
// the schedule instead of behind it, the routing weights at the start instead of one by one in the sum at the end: down kernel
// 7.8 -> 7.0 us, the layer 25.2 -> 24.2.
//
// Sixteen lanes share a weight row: a step of theirs is 128 elements, 256 contiguous bytes, of which a lane multiplies 8 with
// the matching 8 of one or two token rows, in fp32; the sums of the 16 lanes are added at the end.  A wave works on two sets of
// four weight rows at a time, and has the loads of eight steps (16 KB of weights) in flight.  (Two such
// batches by turns: 32 us for one token on 8 of 128 experts instead of 24, the compiler waits for the second with the first.)
//   up:   a wave per (block, 4 activation columns): 4 gate and the 4 matching up rows
//   down: a workgroup of 8 waves per 8 output columns, wave w the blocks w, w + 8, ...; of four blocks or fewer two waves or
//         more share the contraction of each.  The rows' results meet in LDS by pair id and are added up in pair order,
//         weighted, as finalize_kernel does
#pragma once
#include <type_traits>

#include "moe_pipeline.h"

namespace pmoe {
namespace few {

constexpr int kMaxPairs = 64;

__device__ __forceinline__ float lo_f32(uint32_t u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float hi_f32(uint32_t u) { return __uint_as_float(u & 0xffff0000u); }

// acc[q][r] += this lane's share of weight row w[q] x token row x[r], `n_steps` steps (the pointers include the lane's 16 bytes).
template <int NR>
__device__ __forceinline__ void dots(float (&acc)[2][NR], const char *const (&w)[2], const char *const (&x)[NR], int n_steps) {
    constexpr int S = 8;  // steps of a batch of loads
    for (int s0 = 0; s0 < n_steps; s0 += S) {
        uint4 wv[2][S], xv[NR][S];
#pragma unroll
        for (int s = 0; s < S; ++s)
            if (s0 + s < n_steps) {
#pragma unroll
                for (int q = 0; q < 2; ++q) wv[q][s] = load_once(w[q] + (int64_t)(s0 + s) * 256);
#pragma unroll
                for (int r = 0; r < NR; ++r) xv[r][s] = *reinterpret_cast<const uint4 *>(x[r] + (int64_t)(s0 + s) * 256);
            }
#pragma unroll
        for (int s = 0; s < S; ++s)
            if (s0 + s < n_steps) {
#pragma unroll
                for (int r = 0; r < NR; ++r) {
                    const uint32_t xu[4] = {xv[r][s].x, xv[r][s].y, xv[r][s].z, xv[r][s].w};
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        const uint32_t wu[4] = {wv[q][s].x, wv[q][s].y, wv[q][s].z, wv[q][s].w};
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            acc[q][r] = fmaf(lo_f32(wu[i]), lo_f32(xu[i]), acc[q][r]);
                            acc[q][r] = fmaf(hi_f32(wu[i]), hi_f32(xu[i]), acc[q][r]);
                        }
                    }
                }
            }
    }
}

// Sum over the 16 lanes of a row, in all of them.
__device__ __forceinline__ float row_sum(float v) {
#define PMOE_DPP_ADD(ctrl) v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, 0xf, 0xf, true))
    PMOE_DPP_ADD(0xb1);   // quad_perm [1, 0, 3, 2]
    PMOE_DPP_ADD(0x4e);   // quad_perm [2, 3, 0, 1]
    PMOE_DPP_ADD(0x141);  // row_half_mirror
    PMOE_DPP_ADD(0x140);  // row_mirror
#undef PMOE_DPP_ADD
    return v;
}

// A block of the schedule as one wave sees it: expert (-1: nothing to do), pair ids of rows lane and lane + 64, and the rows up
// to the last one that holds a pair.
struct Block {
    int e, id[2], n_rows;
};
// Rows of the schedule.
__device__ __forceinline__ int schedule_rows(const MoeArgs &a) { return min(a.ntpp[0], a.sorted_num); }
// In two steps: the loads do not wait for the length of the schedule, which is loaded beside them.
__device__ __forceinline__ Block request_block(const MoeArgs &a, int blk) {
    const int64_t at = (int64_t)blk * kBlockRows + (threadIdx.x & 63);
    Block b;
    b.id[0] = at < a.sorted_num ? a.sorted_ids[at] : -1;
    b.id[1] = at + 64 < a.sorted_num ? a.sorted_ids[at + 64] : -1;
    b.e = blk < a.n_blocks ? a.expert_ids[blk] : -1;
    b.n_rows = 0;
    return b;
}
__device__ __forceinline__ void settle_block(const MoeArgs &a, Block &b, int blk, int n_rows) {
    const int at = blk * kBlockRows + (threadIdx.x & 63);
    const unsigned n_pairs = (unsigned)(a.M * a.top_k);
    if (at >= n_rows) b.id[0] = -1;
    if (at + 64 >= n_rows) b.id[1] = -1;
    b.e = __builtin_amdgcn_readfirstlane(b.e);
    if (b.e < 0 || b.e >= a.E) b.e = -1;
    const uint64_t m0 = __ballot((unsigned)b.id[0] < n_pairs), m1 = __ballot((unsigned)b.id[1] < n_pairs);
    b.n_rows = m1 ? 128 - __builtin_clzll(m1) : m0 ? 64 - __builtin_clzll(m0) : 0;
}
// Pair id of row `row` (wave-uniform) of the block, -1: none.
__device__ __forceinline__ int pair_of(const MoeArgs &a, const Block &b, int row) {
    const int id = __builtin_amdgcn_readfirstlane(__shfl(row < 64 ? b.id[0] : b.id[1], row & 63, 64));
    return row < b.n_rows && (unsigned)id < (unsigned)(a.M * a.top_k) ? id : -1;
}

// The block's rows one or two at a time: group(integral NR, first row).  (More than two: a token that names an expert twice.)
template <typename Group>
__device__ __forceinline__ void by_rows(int n_rows, Group group) {
    if (n_rows == 1) group(std::integral_constant<int, 1>{}, 0);
    else
        for (int r = 0; r < n_rows; r += 2) group(std::integral_constant<int, 2>{}, r);
}

// act[rows, 4 columns from 4 tile] = swiglu(x W1^T).  The wave of a block's first columns also writes the sorted row of each of
// its pairs to `inv`: of a pair that blocks of two experts list one row stays there, and the down kernel, where several waves
// may share a contraction, takes that row alone.
__device__ __forceinline__ void up_job(const MoeArgs &a, Block b, int blk, int tile, int n_rows) {
    const int lane = threadIdx.x & 63, sub = lane >> 4, chunk = (lane & 15) * 16;
    const int K = a.K, H = a.H, col = 4 * tile + sub;
    settle_block(a, b, blk, n_rows);
    if (b.e < 0) return;
    if (tile == 0) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
            if ((unsigned)b.id[i] < (unsigned)(a.M * a.top_k)) a.inv[b.id[i]] = blk * kBlockRows + lane + 64 * i;
    }
    const char *const gate = a.w1 + ((int64_t)b.e * a.N + col) * K * 2 + chunk;
    const char *const w[2] = {gate, gate + (int64_t)H * K * 2};
    by_rows(b.n_rows, [&](auto n, int row0) {
        constexpr int NR = decltype(n)::value;
        const char *x[NR];
        bool live[NR];
        float acc[2][NR] = {};
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const int p = pair_of(a, b, row0 + r);
            live[r] = p >= 0;
            x[r] = a.x + (int64_t)(live[r] ? p / a.top_k : 0) * K * 2 + chunk;
        }
        dots<NR>(acc, w, x, K >> 7);
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const float g = row_sum(acc[0][r]), u = row_sum(acc[1][r]);
            if (live[r] && (lane & 15) == 0)
                reinterpret_cast<uint16_t *>(a.act)[((int64_t)blk * kBlockRows + row0 + r) * H + col] =
                    (uint16_t)pack2_bf16(swiglu(g, u), 0.f);
        }
    });
}

struct DownShared {
    float y[8][kMaxPairs][8];  // [part of the contraction][pair][column]
    float weight[kMaxPairs];
    int ok[kMaxPairs];
};
// Waves that share the contraction of a block when there are `n_live`.
__device__ __forceinline__ int parts_for(int n_live) { return n_live > 4 ? 1 : n_live > 2 ? 2 : n_live == 2 ? 4 : 8; }
// out[:, 8 columns from 8 tile] (+)= sum over the pairs, in their order, of weight x (act W2^T).  `blocks`: the live blocks the
// host expects; the wave's first block is requested as if they were as many, beside the schedule's length and the routing weights.
__device__ __forceinline__ void down_job(const MoeArgs &a, DownShared &sh, int tile, int blocks, char *out, bool accumulate) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int sub = lane >> 4, chunk = (lane & 15) * 16;
    const int K = a.K, H = a.H, n_pairs = a.M * a.top_k, n_steps = H >> 7;
    const int expected = wave / parts_for(blocks);
    Block ahead = request_block(a, expected);
    const float weight = tid < n_pairs ? a.topk_w[tid] : 0.f;
    const int n_rows = schedule_rows(a), n_live = (n_rows + kBlockRows - 1) / kBlockRows;
    const int parts = parts_for(n_live);
    const int part = wave & (parts - 1), s0 = part * n_steps / parts, s1 = (part + 1) * n_steps / parts;
    if (tid < n_pairs) {
        sh.ok[tid] = 0;
        sh.weight[tid] = weight;
    }
    __syncthreads();
    for (int blk = wave / parts; blk < n_live; blk += 8 / parts) {
        Block b = blk == expected ? ahead : request_block(a, blk);
        settle_block(a, b, blk, n_rows);
        if (b.e < 0) continue;
        const char *const first = a.w2 + ((int64_t)b.e * K + 8 * tile + sub) * H * 2 + chunk + s0 * 256;
        const char *const w[2] = {first, first + (int64_t)4 * H * 2};
        by_rows(b.n_rows, [&](auto n, int row0) {
            constexpr int NR = decltype(n)::value;
            const char *x[NR];
            int p[NR], stands[NR];  // the pair, the row that stands for it
            float acc[2][NR] = {};
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                p[r] = pair_of(a, b, row0 + r);
                stands[r] = a.inv[max(p[r], 0)];
                x[r] = a.act + ((int64_t)blk * kBlockRows + (p[r] >= 0 ? row0 + r : 0)) * H * 2 + chunk + s0 * 256;
            }
            dots<NR>(acc, w, x, s1 - s0);
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                const float lo = row_sum(acc[0][r]), hi = row_sum(acc[1][r]);
                if (p[r] >= 0 && stands[r] == blk * kBlockRows + row0 + r && (lane & 15) == 0) {
                    sh.y[part][p[r]][sub] = lo;
                    sh.y[part][p[r]][4 + sub] = hi;
                    sh.ok[p[r]] = 1;
                }
            }
        });
    }
    __syncthreads();
    for (int i = tid; i < a.M * 8; i += 512) {
        const int t = i >> 3, c = i & 7;
        uint16_t *dst = reinterpret_cast<uint16_t *>(out) + (int64_t)t * K + 8 * tile + c;
        float v = accumulate ? bf16_bits_to_f32(*dst) : 0.f;
        // (The reads of a few pairs are in flight together, eight words, four pairs at most: with four pairs whatever the parts, one behind
        // the other, a token of one expert waits for 32.  K 4096, N 2048, top 1: this kernel 8.0 us, 5.9 as it is.)
        auto add_pairs = [&](auto n) {
            constexpr int P = decltype(n)::value, G = P > 2 ? 8 / P : 4;
            for (int r0 = 0; r0 < a.top_k; r0 += G) {
                float y[G][P], wt[G];
                int ok[G];
#pragma unroll
                for (int r = 0; r < G; ++r) {
                    const int p = t * a.top_k + min(r0 + r, a.top_k - 1);
                    ok[r] = r0 + r < a.top_k ? sh.ok[p] : 0;
                    wt[r] = sh.weight[p];
#pragma unroll
                    for (int q = 0; q < P; ++q) y[r][q] = sh.y[q][p][c];
                }
#pragma unroll
                for (int r = 0; r < G; ++r) {
                    float sum = y[r][0];
#pragma unroll
                    for (int q = 1; q < P; ++q) sum += y[r][q];
                    if (ok[r]) v += wt[r] * sum;
                }
            }
        };
        if (parts == 8) add_pairs(std::integral_constant<int, 8>{});
        else if (parts == 4) add_pairs(std::integral_constant<int, 4>{});
        else if (parts == 2) add_pairs(std::integral_constant<int, 2>{});
        else add_pairs(std::integral_constant<int, 1>{});
        *dst = (uint16_t)pack2_bf16(v, 0.f);
    }
    __syncthreads();  // the table may be cleared again
}

}  // namespace few
}  // namespace pmoe

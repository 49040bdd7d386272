// Weight-streaming bf16 kernels for few rows per expert (decode batches), gfx950.
//
// What bounds these problems is the stream of the touched experts' weights from HBM, read once, and, for the
// smallest, how fast that stream starts and over how many CUs it is spread.  So a job is narrow: the live rows of
// one 128-row block x 32 U weight rows (U = 1, 2), a few hundred jobs even for a single token, and two
// workgroups per CU, one of which streams while the other starts or ends a job.  There is no schedule to build:
// job j is (block j / n_tiles, weight tile j % n_tiles), workgroup b takes jobs b, b + grid, ..., and the number
// of live rows is found when the block's ids are read.
//
// Workgroup: 8 waves, the contraction inside a slab split among them.  A slab is 256 B (128 elements) per row =
// eight 16-wide sub-steps, wave v takes sub-step v for every fragment of the tile, so each operand byte is read
// from LDS once; the eight partial sums meet in LDS when the contraction ends, added in wave order.
//
// Stage: [live token rows, rounded up to 4][32 U weight rows], 256 B each; as many stages as fit the LDS, at most
// 8, all but one in flight.  Rows are 16 chunks of 16 B, chunk c of row r in slot c ^ (r & 15): the operand
// reads of 16 consecutive rows cover the 64 banks once.  Token fragments read past the live rows into what lies
// behind them; that only reaches output columns nobody reads.
//
// Measured (kernel times): 8 experts of K 4096 x N 28672, 58 rows: up 338 -> 281 us (6.7 TB/s), down 219 -> 139 us
// (6.8 TB/s) against tiles of 256 weight rows with 128-byte slabs, which leave half of the CUs without a down job
// there; 8 of 128 experts of K 2048 x N 1536, one row each: up 21.4 -> 13.9, down 11.9 -> 7.9 us.  A flattened variant
// (the next job's first stages requested before the partial sums are added up) ran equal or 6 % slower.
#pragma once
#include "moe_ring.h"

namespace pmoe {
namespace stream {

constexpr int kRB = 256;                    // row bytes of a slab
constexpr int kUnitBytes = 32 * kRB;        // 32 weight rows of a slab
constexpr int kRing = 78 * 1024;
constexpr int kLdsBytes = 80 * 1024;        // two workgroups per CU
constexpr int kMaxStages = 8;
constexpr int kPassRows = 64;               // rows of a block that share one pass over its weights

struct Shared {
    char ring[kRing];
    int pair[kBlockRows];  // pair id of each row of the block, -1: none
    int last[2];           // 1 + index of the last live row among rows 0 .. 63 / 64 .. 127, 0: none
};
static_assert(sizeof(Shared) <= kLdsBytes, "two workgroups must fit a CU");

// A wave's copies of one stage: U instructions of 4 weight rows, and one of 4 token rows per 32-row fragment
// that has live rows among them.
template <int U>
struct Loader {
    const char *w_base[U];  // wave-uniform: first of the wave's rows of unit u
    const char *tok_base;   // wave-uniform
    uint32_t w_off;         // this lane's chunk of its weight row
    uint32_t tok_off[2];    // this lane's chunk of its token row
    bool tok_live[2];       // this lane's token row holds a token
    bool tok_any[2];        // wave-uniform: some lane's does
    int lps;                // instructions per stage
    bool w_once;            // wave-uniform: the weights are read by this pass only

    __device__ __forceinline__ void issue(char *stage, int tok_bytes, int wave, uint32_t koff) const {
#pragma unroll
        for (int q = 0; q < 2; ++q)
            if (tok_any[q]) {
                if (tok_live[q]) ring::copy16(tok_base, tok_off[q] + koff, stage + (32 * q + 4 * wave) * kRB);
            }
        char *w = stage + tok_bytes + 4 * wave * kRB;
        if (w_once) {
#pragma unroll
            for (int u = 0; u < U; ++u) ring::copy16_once(w_base[u], w_off + koff, w + u * kUnitBytes);
        } else {
#pragma unroll
            for (int u = 0; u < U; ++u) ring::copy16(w_base[u], w_off + koff, w + u * kUnitBytes);
        }
    }
};

// One pass over the contraction: acc[u][t] += weight rows of unit u x token fragment t, for this wave's sub-steps.
template <int U, int NF>
__device__ __forceinline__ void k_loop(f32x16 (&acc)[U][NF], const Loader<U> &ld, char *ring_lds, int tok_bytes,
                                       int n_slabs, int wave, int lane, int start) {
    const int stage_bytes = tok_bytes + U * kUnitBytes;
    const int ns = min(kMaxStages, kRing / stage_bytes);
    const int r = lane & 31;
    const int off = r * kRB + (((2 * wave + (lane >> 5)) ^ (r & 15)) << 4);
    int slab = start;  // next slab to issue (rotated order)
    auto issue_next = [&](int stage) {
        ld.issue(ring_lds + stage * stage_bytes, tok_bytes, wave, (uint32_t)slab * kRB);
        if (++slab == n_slabs) slab = 0;
    };
    for (int s = 0; s < ns - 1 && s < n_slabs; ++s) issue_next(s);
    int cur = 0;
    for (int kt = 0; kt < n_slabs; ++kt) {
        // slab kt has landed once at most the copies of the later slabs (up to ns - 2) are pending
        ring::wait_and_barrier_dyn(ld.lps * min(ns - 2, n_slabs - 1 - kt));
        // the stage slab kt - 1 used is free: everybody is past the barrier
        if (kt + ns - 1 < n_slabs) issue_next(cur == 0 ? ns - 1 : cur - 1);
        const char *st = ring_lds + cur * stage_bytes;
        bf16x8 a[U], b[NF];
#pragma unroll
        for (int u = 0; u < U; ++u) a[u] = *reinterpret_cast<const bf16x8 *>(st + tok_bytes + u * kUnitBytes + off);
#pragma unroll
        for (int t = 0; t < NF; ++t) b[t] = *reinterpret_cast<const bf16x8 *>(st + t * kUnitBytes + off);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int t = 0; t < NF; ++t) acc[u][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[u], b[t], acc[u][t], 0, 0, 0);
        if (++cur == ns) cur = 0;
    }
    __syncthreads();  // every stage has been read: the ring is scratch now
}

// Partial sums of the waves for one token fragment, [wave][unit][register / 4][lane] float4 in the ring.
template <int U>
__device__ __forceinline__ void put_partial(char *ring_lds, const f32x16 &v, int u, int wave, int lane) {
    float4 *dst = reinterpret_cast<float4 *>(ring_lds) + (wave * U + u) * 256 + lane;
#pragma unroll
    for (int i = 0; i < 4; ++i) dst[64 * i] = make_float4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
}
template <int U>
__device__ __forceinline__ float4 sum_partials(const char *ring_lds, int u, int i4, int lane) {
    const float4 *src = reinterpret_cast<const float4 *>(ring_lds) + u * 256 + 64 * i4 + lane;
    float4 s = src[0];
#pragma unroll
    for (int w = 1; w < 8; ++w) {
        const float4 v = src[w * U * 256];
        s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
    return s;
}

// One pass: contraction over the n rows the loader is set up for, then for each token fragment the partial sums
// in LDS handed to `finish(t)`.
template <int U, int NF, typename Finish>
__device__ __forceinline__ void run_pass(const Loader<U> &ld, char *ring_lds, int n, int n_slabs, int wave, int lane,
                                         int start, Finish finish) {
    f32x16 acc[U][NF];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (int t = 0; t < NF; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[u][t][i] = 0.f;
    k_loop<U, NF>(acc, ld, ring_lds, ((n + 3) & ~3) * kRB, n_slabs, wave, lane, start);
#pragma unroll
    for (int t = 0; t < NF; ++t) {
        if (t > 0) __syncthreads();
#pragma unroll
        for (int u = 0; u < U; ++u) put_partial<U>(ring_lds, acc[u][t], u, wave, lane);
        __syncthreads();
        finish(t);
    }
    __syncthreads();  // the ring may be filled again
}

// One job: block `blk` of expert `e`, weight tile `tile`; `id` = this thread's sorted id (threads 0 .. 127).
// UP: act[rows, 16 U columns] = swiglu(x W1^T), unit u = 16 gate rows and the 16 up rows that go with them, so that
// both operands of a SwiGLU element sit in registers i and i + 8 of one lane.  Otherwise y[pair, 32 U columns] =
// act W2^T.
template <bool UP, int U>
__device__ __forceinline__ void run_job(const MoeArgs &a, Shared &sh, int blk, int e, int tile, int id) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int K = a.K, H = a.H;
    if (tid < kBlockRows) {
        const bool ok = (unsigned)id < (unsigned)(a.M * a.top_k);
        sh.pair[tid] = ok ? id : -1;
        const uint64_t m = __ballot(ok);
        if (lane == 0) sh.last[wave] = m != 0 ? tid + 64 - __builtin_clzll(m) : 0;
    }
    __syncthreads();
    const int n_rows = __builtin_amdgcn_readfirstlane(sh.last[1] != 0 ? sh.last[1] : sh.last[0]);

    Loader<U> ld;
    const uint32_t row_bytes = (uint32_t)(UP ? K : H) * 2u;
    const int sub = lane >> 4;  // row of the lane inside an instruction
    const uint32_t chunk = (uint32_t)((lane & 15) ^ ((4 * wave + sub) & 15)) * 16u;
    ld.w_off = (uint32_t)sub * row_bytes + chunk;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        int64_t row;
        if (UP) row = (int64_t)e * a.N + (wave >= 4 ? H : 0) + (tile * U + u) * 16 + 4 * (wave & 3);
        else row = (int64_t)e * K + (tile * U + u) * 32 + 4 * wave;
        ld.w_base[u] = ring::uniform_ptr((UP ? a.w1 : a.w2) + row * row_bytes);
    }
    ld.tok_base = ring::uniform_ptr(UP ? a.x : a.act + (int64_t)blk * kBlockRows * row_bytes);
    ld.w_once = n_rows <= kPassRows;
    const int n_slabs = (int)(row_bytes / kRB);
    const int start = (blk + tile) % n_slabs;

    for (int row0 = 0; row0 < n_rows; row0 += kPassRows) {
        const int n = min(kPassRows, n_rows - row0);
        ld.lps = U;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int row = 32 * q + 4 * wave + sub;
            const int p = row < n ? sh.pair[row0 + row] : -1;
            ld.tok_live[q] = p >= 0;
            ld.tok_off[q] = (UP ? (uint32_t)max(p, 0) / (uint32_t)a.top_k : (uint32_t)(row0 + row)) * row_bytes + chunk;
            ld.tok_any[q] = __ballot(p >= 0) != 0;
            ld.lps += ld.tok_any[q] ? 1 : 0;
        }
        auto finish = [&](int t) {
            const int row = row0 + 32 * t + (lane & 31);
            const int p = row < row0 + n ? sh.pair[row] : -1;
            if (UP) {
                if (tid < U * 128) {
                    const int u = tid >> 7, q = (tid >> 6) & 1;
                    const float4 g = sum_partials<U>(sh.ring, u, q, lane), v = sum_partials<U>(sh.ring, u, q + 2, lane);
                    uint2 pk;
                    pk.x = pack2_bf16(swiglu(g.x, v.x), swiglu(g.y, v.y));
                    pk.y = pack2_bf16(swiglu(g.z, v.z), swiglu(g.w, v.w));
                    const int col = (tile * U + u) * 16 + 8 * q + 4 * (lane >> 5);
                    if (p >= 0) *reinterpret_cast<uint2 *>(a.act + (((int64_t)blk * kBlockRows + row) * H + col) * 2) = pk;
                }
            } else {
                if (tid < U * 256) {
                    const int u = tid >> 8, q = (tid >> 6) & 3;
                    const float4 v = sum_partials<U>(sh.ring, u, q, lane);
                    uint2 pk;
                    pk.x = pack2_bf16(v.x, v.y);
                    pk.y = pack2_bf16(v.z, v.w);
                    const int col = (tile * U + u) * 32 + 8 * q + 4 * (lane >> 5);
                    if (p >= 0) *reinterpret_cast<uint2 *>(a.y + ((int64_t)p * K + col) * 2) = pk;
                }
            }
        };
        if (n <= 32) run_pass<U, 1>(ld, sh.ring, n, n_slabs, wave, lane, start, finish);
        else run_pass<U, 2>(ld, sh.ring, n, n_slabs, wave, lane, start, finish);
    }
    __syncthreads();  // the table may be written again
}

// ---- Down GEMM with a short contraction (RB = 2 H = 256 or 512 bytes per row).
//
// A unit of 32 weight rows is then only 8 or 16 contiguous KB, and starting and ending a job for every one or two of
// them (a latency each, and eight partial sums to add) costs more than its stream.  Here every wave works alone:
// the token fragment sits in registers for the whole contraction, a unit is copied into the wave's own LDS, read into
// registers at once, and the next unit's copy runs under the matrix instructions, the store and, above all, the other
// waves.  No barrier, nothing to add up.
template <int RB>
struct Unit {
    static constexpr int kSteps = RB / 32;            // 16-wide sub-steps of the contraction
    static constexpr int kChunks = RB / 16;           // 16-byte chunks of a row
    static constexpr int kRowsPerCopy = 1024 / RB;
    static constexpr int kCopies = 32 / kRowsPerCopy;
    static constexpr int kBytes = 32 * RB;
};

// Units first, first + step, ... < last of block `blk` (expert e); id0 / id1 = sorted ids of rows lane / lane + 64.
// LDS: chunk c of row r in slot c ^ (r & 15) (16 consecutive rows cover the 64 banks once).
template <int RB>
__device__ __forceinline__ void down_short(const MoeArgs &a, char *buf, int blk, int e, int id0, int id1, int first,
                                           int step, int last) {
    using G = Unit<RB>;
    const int lane = threadIdx.x & 63, half = lane >> 5, r = lane & 31;
    const unsigned n_pairs = (unsigned)(a.M * a.top_k);
    const uint64_t m0 = __ballot((unsigned)id0 < n_pairs), m1 = __ballot((unsigned)id1 < n_pairs);
    const int n_rows = m1 ? 128 - __builtin_clzll(m1) : m0 ? 64 - __builtin_clzll(m0) : 0;
    if (n_rows == 0 || first >= last) return;
    // copy i moves rows kRowsPerCopy i ..: this lane's is row kRowsPerCopy i + sub, slot lane % kChunks
    const int sub = lane / G::kChunks;
    const uint32_t lane_off = (uint32_t)sub * RB + (uint32_t)((lane % G::kChunks) ^ sub) * 16u;
    const bool once = n_rows <= 32;
    const char *w_exp = a.w2 + (int64_t)e * a.K * RB;
    auto issue = [&](int u) {
        const char *w = ring::uniform_ptr(w_exp + (int64_t)u * G::kBytes);
#pragma unroll
        for (int i = 0; i < G::kCopies; ++i) {
            const uint32_t off = (lane_off ^ (uint32_t)(((i * G::kRowsPerCopy) & 15) << 4)) + i * 1024u;
            if (once) ring::copy16_once(w, off, buf + i * 1024);
            else ring::copy16(w, off, buf + i * 1024);
        }
    };
    const char *rd = buf + r * RB;

    for (int t = 0; t * 32 < n_rows; ++t) {
        issue(first);
        const int p = __shfl(t < 2 ? id0 : id1, 32 * (t & 1) + r, 64);
        const bool live = (unsigned)p < n_pairs;
        bf16x8 b[G::kSteps];
        const char *tok = a.act + ((int64_t)blk * kBlockRows + 32 * t + r) * RB + half * 16;
#pragma unroll
        for (int j = 0; j < G::kSteps; ++j) {
#pragma unroll
            for (int i = 0; i < 8; ++i) b[j][i] = (__bf16)0.f;
            if (live) b[j] = *reinterpret_cast<const bf16x8 *>(tok + j * 32);
        }
        char *dst = a.y + ((int64_t)(live ? p : 0) * a.K + 4 * half) * 2;
        for (int u = first; u < last; u += step) {
            asm volatile("s_waitcnt vmcnt(0)" : : : "memory");  // the unit has landed
            bf16x8 w[G::kSteps];
#pragma unroll
            for (int j = 0; j < G::kSteps; ++j)
                w[j] = *reinterpret_cast<const bf16x8 *>(rd + (((2 * j + half) ^ (r & 15)) << 4));
            asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");  // it is in registers: the buffer may be filled again
            if (u + step < last) issue(u + step);
            f32x16 acc[2];
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[0][i] = acc[1][i] = 0.f;
#pragma unroll
            for (int j = 0; j < G::kSteps; ++j) acc[j & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[j], b[j], acc[j & 1], 0, 0, 0);
            if (live) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    float v[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[i] = acc[0][4 * q + i] + acc[1][4 * q + i];
                    uint2 pk;
                    pk.x = pack2_bf16(v[0], v[1]);
                    pk.y = pack2_bf16(v[2], v[3]);
                    *reinterpret_cast<uint2 *>(dst + (32 * u + 8 * q) * 2) = pk;
                }
            }
        }
    }
}

}  // namespace stream
}  // namespace pmoe

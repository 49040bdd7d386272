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
#include <type_traits>

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
    bool w_once;            // wave-uniform: the block reads the weights in one pass (other blocks of the expert, rare where
                            // these kernels run, are not looked for)

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

// Inverts the sorted order for finalize: inv[pair id] = sorted row (entries of pairs that are not in the schedule keep
// what the buffer held; the reader validates them).  The workgroups of the grid from `first` on, `threads` threads each.
__device__ __forceinline__ void invert(const MoeArgs &a, int threads, int first = 0) {
    const int n_rows = min(a.ntpp[0], a.sorted_num), n_pairs = a.M * a.top_k;
    for (int s = ((int)blockIdx.x - first) * threads + (int)threadIdx.x; s < n_rows; s += ((int)gridDim.x - first) * threads) {
        const int p = a.sorted_ids[s], es = a.expert_ids[s >> 7];
        if (p >= 0 && p < n_pairs && es >= 0 && es < a.E) a.inv[p] = s;
    }
}

// The jobs of this workgroup: job(block, expert, weight tile, sorted id of this thread's row), none if skip(length of
// the schedule).  The up kernel also inverts the sorted order.
template <bool UP, typename Skip, typename Job>
__device__ __forceinline__ void for_each_job(const MoeArgs &a, int n_tiles, Skip skip, Job job) {
    const int tid = threadIdx.x, grid = (int)gridDim.x;
    // sorted id (threads 0 .. 127) and expert of a job's block, fetched under the job before; for the first job
    // without waiting for the length of the schedule
    auto fetch = [&](int j, int &id, int &e) {
        id = e = -1;
        const int blk = n_tiles > 0 ? j / n_tiles : a.n_blocks;
        if (blk < a.n_blocks) {
            const int s = blk * kBlockRows + tid;
            if (tid < kBlockRows && s < a.sorted_num) id = a.sorted_ids[s];
            e = a.expert_ids[blk];
        }
    };
    int id, e;
    fetch((int)blockIdx.x, id, e);
    const int ntpp = a.ntpp[0];
    const int n_jobs = min((ntpp + kBlockRows - 1) / kBlockRows, a.n_blocks) * n_tiles;
    if (UP) invert(a, 512);
    if (skip(ntpp)) return;
    for (int j = (int)blockIdx.x; j < n_jobs; j += grid) {
        const int blk = j / n_tiles;
        int next_id, next_e;
        fetch(j + grid, next_id, next_e);
        if (e >= 0 && e < a.E) job(blk, __builtin_amdgcn_readfirstlane(e), j - blk * n_tiles, id);
        id = next_id;
        e = next_e;
    }
}

// ---- Down GEMM with a short contraction (at most 512 bytes per weight row).
//
// A unit of 32 weight rows is then only a few contiguous KB, and starting and ending a job for every one or two of
// them (a latency each, and eight partial sums to add) costs more than its stream.  Here every wave works alone: it
// copies a turn (up to 16 KB of one expert's rows) into its own LDS, reads it into registers at once, and runs the
// block's token fragments past it; the next turn's copy and its first token fragment are under way meanwhile.  No
// barrier, nothing to add up, and no weight row is read twice.  A workgroup's four waves take neighbouring turns, and
// neighbouring workgroups neighbouring jobs: what the chip reads at one time is one narrow window that moves through
// W2, which the HBM channels serve evenly (257 experts, K 7168, H 256 in bf16: 158 us; with 14 turns in a row per wave
// 188, with 28 of its own per wave 239; the general kernel 219).
//
// Engine: request() starts the copy of a turn, request_tokens() the loads of the block's first token fragment (`pair`:
// pair id of the lane's row of it), wait() makes both land in registers, compute() does the work of the turn.
template <typename Engine>
__device__ __forceinline__ void for_each_turn(const MoeArgs &a, int n_turns, Engine &eng) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int n_live = min((a.ntpp[0] + kBlockRows - 1) / kBlockRows, a.n_blocks);
    const int n_jobs = (n_turns + 3) / 4, total = n_live * n_jobs;
    const unsigned n_pairs = (unsigned)(a.M * a.top_k);
    struct Job {
        int blk, turn, e, id0, id1, n_rows;
    };
    // job j of this wave; its sorted ids (rows lane and lane + 64) and expert
    auto fetch = [&](int j, Job &job) {
        job.n_rows = -1;
        job.e = job.id0 = job.id1 = -1;
        job.blk = job.turn = 0;
        if (j < total) {
            job.blk = j / n_jobs;
            job.turn = (j - job.blk * n_jobs) * 4 + wave;
            const int s0 = job.blk * kBlockRows + lane;
            if (s0 < a.sorted_num) job.id0 = a.sorted_ids[s0];
            if (s0 + 64 < a.sorted_num) job.id1 = a.sorted_ids[s0 + 64];
            job.e = a.expert_ids[job.blk];
        }
    };
    auto count = [&](Job &job) {  // n_rows = 0: nothing to do
        const bool ok = job.turn < n_turns && (unsigned)__builtin_amdgcn_readfirstlane(job.e) < (unsigned)a.E;
        const uint64_t m0 = __ballot((unsigned)job.id0 < n_pairs), m1 = __ballot((unsigned)job.id1 < n_pairs);
        job.n_rows = !ok ? 0 : m1 ? 128 - __builtin_clzll(m1) : m0 ? 64 - __builtin_clzll(m0) : 0;
    };
    int j = (int)blockIdx.x;
    Job cur, next;
    fetch(j, cur);
    count(cur);
    auto request = [&](const Job &job) {
        if (job.n_rows > 0) eng.request(__builtin_amdgcn_readfirstlane(job.e), job.turn);
    };
    auto request_tokens = [&](const Job &job) {
        if (job.n_rows > 0) eng.request_tokens(job.blk, __shfl(job.id0, lane & 31, 64));
    };
    request(cur);
    request_tokens(cur);
    for (; j < total; j += (int)gridDim.x) {
        fetch(j + (int)gridDim.x, next);
        if (cur.n_rows > 0) eng.wait();
        count(next);
        request(next);
        if (cur.n_rows > 0) eng.compute(cur.blk, cur.turn, cur.id0, cur.id1, cur.n_rows);
        request_tokens(next);
        cur = next;
    }
}

// bf16, RB = 2 H = 256 or 512 bytes per row; a turn is one unit of 32 weight rows (output columns).
// LDS: chunk c of row r in slot c ^ (r & 15) (16 consecutive rows cover the 64 banks once).
template <int RB>
struct ShortDown {
    static constexpr int kSteps = RB / 32;   // 16-wide sub-steps of the contraction
    static constexpr int kChunks = RB / 16;  // 16-byte chunks of a row
    static constexpr int kRowsPerCopy = 1024 / RB;
    static constexpr int kBytes = 32 * RB;
    static constexpr int kTurnCols = 32;

    const MoeArgs &a;
    char *buf;
    bf16x8 w[kSteps], b[kSteps] = {};  // the turn's rows, a token fragment

    __device__ __forceinline__ ShortDown(const MoeArgs &args, char *lds) : a(args), buf(lds) {}
    // Token fragment from row row0 on.  Rows without a pair are not loaded: their lanes keep what they hold, which only
    // reaches output rows nobody stores (loading them too: 216 us instead of 158 with 3 rows in 32).
    __device__ __forceinline__ void load_tokens(bf16x8 (&dst)[kSteps], int blk, int row0, int pair) const {
        const int lane = threadIdx.x & 63;
        if ((unsigned)pair >= (unsigned)(a.M * a.top_k)) return;
        const char *tok = a.act + ((int64_t)blk * kBlockRows + row0 + (lane & 31)) * RB + (lane >> 5) * 16;
#pragma unroll
        for (int j = 0; j < kSteps; ++j) dst[j] = *reinterpret_cast<const bf16x8 *>(tok + j * 32);
    }
    __device__ __forceinline__ void request(int e, int turn) {
        const int lane = threadIdx.x & 63, sub = lane / kChunks;
        const uint32_t lane_off = (uint32_t)sub * RB + (uint32_t)((lane % kChunks) ^ sub) * 16u;
        const char *src = ring::uniform_ptr(a.w2 + ((int64_t)e * a.K + turn * 32) * RB);
#pragma unroll
        for (int i = 0; i < 32 / kRowsPerCopy; ++i)
            ring::copy16_once(src, (lane_off ^ (uint32_t)(((i * kRowsPerCopy) & 15) << 4)) + i * 1024u, buf + i * 1024);
    }
    __device__ __forceinline__ void request_tokens(int blk, int pair) { load_tokens(b, blk, 0, pair); }
    __device__ __forceinline__ void wait() {
        const int lane = threadIdx.x & 63, r = lane & 31, half = lane >> 5;
        asm volatile("s_waitcnt vmcnt(0)" : : : "memory");  // the turn has landed
#pragma unroll
        for (int j = 0; j < kSteps; ++j) {
            // (taken over here: the compiler's wait for them, placed behind the next copies, would wait for those too)
            asm volatile("" : "+v"(b[j]));
            w[j] = *reinterpret_cast<const bf16x8 *>(buf + r * RB + (((2 * j + half) ^ (r & 15)) << 4));
        }
        asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");  // it is in registers: the buffer may be filled again
    }
    __device__ __forceinline__ void compute(int blk, int turn, int id0, int id1, int n_rows) {
        const int lane = threadIdx.x & 63, r = lane & 31, half = lane >> 5;
        int p = __shfl(id0, r, 64);
        for (int row0 = 0;;) {
            f32x16 acc;
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
            for (int j = 0; j < kSteps; ++j) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[j], b[j], acc, 0, 0, 0);
            asm volatile("" : "+v"(acc));  // (kept out of the branch: every lane takes part)
            if ((unsigned)p < (unsigned)(a.M * a.top_k)) {
                char *dst = a.y + ((int64_t)p * a.K + 32 * turn + 4 * half) * 2;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    uint2 pk;
                    pk.x = pack2_bf16(acc[4 * q], acc[4 * q + 1]);
                    pk.y = pack2_bf16(acc[4 * q + 2], acc[4 * q + 3]);
                    *reinterpret_cast<uint2 *>(dst + 16 * q) = pk;
                }
            }
            row0 += 32;
            if (row0 >= n_rows) break;
            p = __shfl(row0 < 64 ? id0 : id1, (row0 & 32) + r, 64);
            load_tokens(b, blk, row0, p);
        }
    }
};

}  // namespace stream
}  // namespace pmoe

// bf16 kernels of the fused MoE forward for gfx950, on tall tiles (moe_tall.h): prologue (row tiles cut by
// 32-row fragments, plan of the two kernels), gate/up GEMM + SwiGLU, down GEMM.
//
// Replaces the bf16 launcher and kernels of the reference's
// prime_moe/csrc/kernels/fused_moe_bf16_kernel.cu:21-733 (gather :21-47, gate/up GEMM + SwiGLU :196-229,
// down GEMM :496-542).
//
// No work list: a workgroup derives its job from its id and a plan that workgroup 0 of the prologue writes
// (see TallPlan), so the prologue only builds the table of row tiles.  Problems of few up jobs have no prologue: the
// workgroups of moe_deep_up_kernel plan for themselves.  One token or two: the kernels of moe_few.h.  No value is
// accumulated with atomics and every sum has a fixed order: the result is a pure function of the inputs.
#include <algorithm>

#include "align_sort.h"
#include "moe_few.h"
#include "moe_pipeline.h"
#include "moe_stream.h"
#include "moe_tall.h"

namespace pmoe {

// Crowded schedules.  Whether the streaming kernels (moe_stream.h) are the faster ones is a matter of the rows per
// block, and the host, which enqueues them when there are few rows per expert on average, does not know how the
// tokens are spread: with all of them on a few experts a block is full, its weights are read once per 64 rows, and the
// short down kernel reads the activation once per 32 columns.  The length of the schedule tells: `pairs` rows on
// n_live blocks.  So where crowding can matter (crowding_possible), both kinds of kernels are enqueued and decide by
// this function, the same in all of them, which of them works: bit 0 the up kernel, bit 1 the down kernel is a tall one.
//  * up, and down with H > 256: more than 64 rows per live block, that is, more than one pass over most weights, and enough
//    bytes in a pass that the prologue (8 us) is small against it;
//  * down with H <= 256: the fragments of 32 rows beyond the first of a block cost a pass over its rows of W2 each.
// Streaming / tall / as decided here, us, whole op.  K 2048, N 1536, 512 tokens x top 8 on 85 of 128 experts (48 rows per
// block): 188 / 199 / 194, on 64: 168 / 163 / 175, on 51: 188 / 152 / 155, on 21: 138 / 85 / 91; K 4096, N 28672, 128 x 2 on
// 4 of 8 (64 rows): 400 / 419 / 406, on 3: 423 / 342 / 348; K 7168, N 512, 900 x 9 on all 257 (31 rows): 662 / 659 / 630,
// on 63: 532 / 246 / 233, 256 x 9 on 57 (40 rows): 169 / 199 / 162.
// The kernels that are enqueued and find nothing to do cost 2 us each, so they are enqueued where crowding would cost more:
// an expert has at most M rows (more only if a token names it twice, which is not looked for), M <= 64 is one pass.  The
// tall up kernel comes with the prologue and the tall down kernel, unless these are there already.  Crowded, without / with it,
// and spread out, without / with it, us: K 2048, N 1536 top 8: 200 tokens on 16 experts 70 / 66, on all 128 216 / 222 (157 MB:
// not enqueued), 256 on 16 103 / 74, on 128 220 / 227; K = N = 2048, 256 x 4 on 6 of 32 experts 71 / 63, on 4 54 / 63, on 32 91 / 96
// (134 MB: not enqueued); K 7168, N 512, 160 x 9 on 9 of 257 130 / 101, on all 481 / 485.
constexpr float kCrowdedUpBytes = 64e6f, kCrowdedDownBytes = 96e6f;
__device__ __forceinline__ int crowding(const MoeArgs &a, int ntpp) {
    if (!a.crowd) return 0;
    const float n_live = (float)min((ntpp + kBlockRows - 1) / kBlockRows, a.n_blocks);
    if (n_live < 1.f) return 0;
    const float rows = (float)(a.M * a.top_k) / n_live, w2_bytes = 2.f * (float)a.K * (float)a.H;
    int tall = rows > 64.f && n_live * 2.f * w2_bytes >= kCrowdedUpBytes ? 3 : 0;
    if (a.H <= 256) {
        // rows of a block spread round the mean: the second fragment appears from 24 rows on
        const float extra = fminf((rows - 24.f) * (1.f / 16.f), rows * (1.f / 32.f) - 0.5f);
        if (n_live * extra * w2_bytes >= kCrowdedDownBytes) tall |= 2;
    }
    return tall & a.crowd;
}
// The tall kernels to enqueue (bits as in crowding()).
static int crowding_possible(const MoeArgs &a) {
    const double pairs = (double)a.M * a.top_k, w2_bytes = 2.0 * a.K * a.H;
    int tall = a.H <= 256 && a.M > 24 && 0.75 * pairs / 32 * w2_bytes >= kCrowdedDownBytes ? 2 : 0;
    if (a.M > 64 && pairs / 64 * 2 * w2_bytes >= (tall ? 2 : 3) * kCrowdedUpBytes) tall = 3;
    return tall;
}

constexpr int kPrologueThreads = 1024;
// Inclusive scan of one int per thread over the workgroup of the prologue; `s_part` holds an int per wave.
__device__ __forceinline__ int block_scan(int v, int *s_part) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int t = __shfl_up(v, d, 64);
        if (lane >= d) v += t;
    }
    __syncthreads();  // s_part may still be read from the previous call
    if (lane == 63) s_part[wave] = v;
    __syncthreads();
    for (int w = 0; w < wave; ++w) v += s_part[w];
    return v;
}

// Estimated time of a kernel (in units of a third of a microsecond) whose `f2` pairs of fragments are cut into
// `n_tiles` row tiles: whole rounds of the chip's CUs at the cost of a mean tile, plus a last round whose jobs
// are shared by rows.  A tile of g pairs costs (0.6 + g) per slab of its K loop (measured on operands that stay in
// L2: 0.18 + 0.34 g us on tiles of 2 to 6 pairs; inside a full kernel the fixed part is larger, which only
// strengthens the preference for few, tall tiles) and 3 + 2.5 g for set-up and epilogue; a round of nothing but shared jobs costs 1.3
// times what its small tiles would among large ones (measured on the Mixtral-like down kernel: every weight row
// is then read twice as often).
__device__ __forceinline__ float estimate_kernel(int n_tiles, int f2, int n_wt, int n_slabs, int n_cus, int &parts,
                                                 int &tail) {
    parts = 1;
    tail = 0;
    if (n_tiles <= 0) return 0.f;
    const float g = (float)f2 / (float)n_tiles;
    auto cost = [&](float pairs) { return (float)n_slabs * (0.6f + pairs) + 3.f + 2.5f * pairs; };
    const int jobs = n_tiles * n_wt, rounds = jobs / n_cus, rest = jobs % n_cus;
    float t = (float)rounds * cost(g);
    if (rest > 0) {
        // (the walk is dealt in whole rounds of kWalkRound jobs, and a split takes all that is left behind them: only where that
        // is what the chip has left over, too, always on as many CUs)
        const int p = rounds >= 16 || rest != jobs % kWalkRound ? 1 : min(min(4, n_cus / rest), max(1, (int)g));
        t += p > 1 ? 1.3f * cost(g / (float)p) : cost(g);
        if (p > 1) {
            parts = p;
            tail = rest;
        }
    }
    return t;
}
// Number of row tiles for a kernel with n_wt weight tiles: the fewest there can be (t_min, tiles of up to 6
// pairs), or, if the estimate likes it better, the next number that fills whole rounds of the CUs (smaller
// tiles, nothing left over), as long as that is at most half as many again and fits the tables (t_cap).
__device__ __forceinline__ int choose_tiles(int t_min, int t_cap, int f2, int n_wt, int n_slabs, int n_cus) {
    if (t_min <= 0) return 0;
    int g = n_cus, r = n_wt;  // gcd
    while (r) {
        const int x = g % r;
        g = r;
        r = x;
    }
    const int step = n_cus / g;  // tiles x n_wt is a multiple of n_cus for every multiple of step
    const int t_full = (t_min + step - 1) / step * step;
    if (t_full == t_min || t_full > t_cap || 2 * t_full > 3 * t_min || t_full > f2) return t_min;
    int parts, tail;
    const float e_min = estimate_kernel(t_min, f2, n_wt, n_slabs, n_cus, parts, tail);
    const float e_full = estimate_kernel(t_full, f2, n_wt, n_slabs, n_cus, parts, tail);
    return e_full < 0.98f * e_min ? t_full : t_min;
}

// Prologue of a bf16 call.  Workgroup 0 builds the row tiles and the plan:
//  1. runs of blocks with one expert (a thread per block, block-wide scans per 1024 blocks); the thread of a run's
//     last block reads that block's 128 ids for the last row that holds a pair: the run has f2 pairs of fragments;
//  2. per kernel the number of row tiles (see choose_tiles);
//  3. the runs in the order of falling f2, runs of one size in their own order (a stable counting sort: a job's place in
//     the walk sets where its K loop starts, so places given in order of arrival would change the last bits of
//     the result from call to call): the walk of a kernel then ends with the small tiles, and what is left over
//     when the CUs run out of jobs is short;
//  4. the tiles of the two cuts (a run gets the tiles it needs at 6 pairs a tile, and the largest runs one more
//     each until the chosen number is reached), then the plans with the split of the tails.
// The list of runs lives in LDS (in the workspace when there are more than kLdsRuns blocks).
// All workgroups invert the sorted order: inv[pair id] = sorted row.  Entries of pairs that are not in the
// schedule keep whatever the buffer held; the reader validates an entry against sorted_ids.
constexpr int kLdsRuns = 2048;
constexpr int kSizeKeyBits = 7, kSizeKeys = 1 << kSizeKeyBits;  // runs are ordered by min(f2, kSizeKeys - 1)
__global__ __launch_bounds__(kPrologueThreads) void moe_prologue_kernel_bf16(MoeArgs a, int n_wt_up, int n_wt_down, int n_cus,
                                                                int do_invert) {
    if (a.crowd && crowding(a, a.ntpp[0]) == 0) return;
    const int n_pairs = a.M * a.top_k;
    if (blockIdx.x == 0) {
        __shared__ int4 s_runs[kLdsRuns];  // {first block, f2, expert, 0}
        __shared__ int s_order[kLdsRuns];
        __shared__ int s_part[kPrologueThreads / 64], s_carry[2], s_want[2], s_tiles[2];
        __shared__ int s_sum[8];            // [0]: tiles of up to 6 pairs the runs need; [4]: pairs of fragments
        __shared__ int s_hist[kSizeKeys];   // runs per size key, then the next place of each key in the order
        const int tid = threadIdx.x;
        const int n_live = min((a.ntpp[0] + kBlockRows - 1) / kBlockRows, a.n_blocks);
        int4 *runs = n_live <= kLdsRuns ? s_runs : a.runs;
        int *order = n_live <= kLdsRuns ? s_order : reinterpret_cast<int *>(a.runs + n_live);
        if (tid < 2) s_carry[tid] = tid == 0 ? -1 : 0;
        if (tid < 8) s_sum[tid] = 0;
        if (tid < kSizeKeys) s_hist[tid] = 0;
        if (tid < 16) a.plan->counters[tid] = n_cus / 8;  // the first slots are taken without asking (see ask_slot)
        __syncthreads();
        // 1. runs
        for (int base = 0; base < n_live; base += kPrologueThreads) {
            const int b = base + tid;
            const bool live = b < n_live;
            const int e = live ? a.expert_ids[b] : -1;
            const bool is_start = live && (b == 0 || a.expert_ids[b - 1] != e);
            const bool is_last = live && (b + 1 == n_live || a.expert_ids[b + 1] != e);
            // start of this block's run: the largest start at or before it
            int v = is_start ? b : -1;
            {
                const int lane = tid & 63, wave = tid >> 6;
#pragma unroll
                for (int d = 1; d < 64; d <<= 1) {
                    const int t = __shfl_up(v, d, 64);
                    if (lane >= d) v = max(v, t);
                }
                __syncthreads();
                if (lane == 63) s_part[wave] = v;
                __syncthreads();
                for (int w = 0; w < wave; ++w) v = max(v, s_part[w]);
                v = max(v, s_carry[0]);
            }
            const int run_start = v;
            int f2 = 0;
            if (is_last && e >= 0 && e < a.E) {
                const int s0 = b * kBlockRows;
                int last = -1;
                if (s0 + kBlockRows <= a.sorted_num && (reinterpret_cast<uintptr_t>(a.sorted_ids) & 15) == 0) {
                    // all 32 loads in flight together
                    const int4 *src = reinterpret_cast<const int4 *>(a.sorted_ids + s0);
                    int4 v[kBlockRows / 4];
#pragma unroll
                    for (int r = 0; r < kBlockRows / 4; ++r) v[r] = src[r];
#pragma unroll
                    for (int r = 0; r < kBlockRows / 4; ++r) {
                        if ((unsigned)v[r].x < (unsigned)n_pairs) last = 4 * r;
                        if ((unsigned)v[r].y < (unsigned)n_pairs) last = 4 * r + 1;
                        if ((unsigned)v[r].z < (unsigned)n_pairs) last = 4 * r + 2;
                        if ((unsigned)v[r].w < (unsigned)n_pairs) last = 4 * r + 3;
                    }
                } else {
                    for (int r = 0; r < kBlockRows; ++r) {
                        const int p = s0 + r < a.sorted_num ? a.sorted_ids[s0 + r] : -1;
                        if ((unsigned)p < (unsigned)n_pairs) last = r;
                    }
                }
                f2 = ((b - run_start) * kBlockRows + last + 1 + 63) >> 6;
            }
            const int incl = block_scan(f2 > 0 ? 1 : 0, s_part);
            const int carry = s_carry[1];
            if (f2 > 0) {
                runs[carry + incl - 1] = make_int4(run_start, f2, e, 0);
                atomicAdd(&s_hist[min(f2, kSizeKeys - 1)], 1);
                atomicAdd(&s_sum[4], f2);
                atomicAdd(&s_sum[0], (f2 + 5) / 6);
            }
            __syncthreads();
            if (tid == kPrologueThreads - 1) {
                s_carry[0] = run_start;
                s_carry[1] = carry + incl;
            }
            __syncthreads();
        }
        const int n_runs = s_carry[1];
        __threadfence_block();
        // 2. the number of row tiles of each kernel: thread 64 the up kernel's, thread 65 the down kernel's (a wave
        // that has no part in step 3)
        if ((tid & ~1) == 64) {
            const int down = tid & 1;
            const int n_wt = down ? n_wt_down : n_wt_up, n_slabs = (down ? a.H : a.K) * 2 / tall::kRB;
            s_want[down] = choose_tiles(s_sum[0], a.n_blocks, s_sum[4], n_wt, n_slabs, n_cus);
        }
        // 3. order of the runs, by one wave: the first place of each key, then every run takes the next place of its key
        if (tid < 64) {
            // (key k's place = runs with a larger key; two keys per lane, largest keys first)
            const int k_hi = kSizeKeys - 1 - 2 * tid, k_lo = k_hi - 1;
            const int c_hi = s_hist[k_hi], c_lo = s_hist[k_lo];
            int incl = c_hi + c_lo;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int t = __shfl_up(incl, d, 64);
                if (tid >= d) incl += t;
            }
            s_hist[k_hi] = incl - c_hi - c_lo;
            s_hist[k_lo] = incl - c_lo;
            for (int base = 0; base < n_runs; base += 64) {
                const int i = base + tid;
                const int key[1] = {i < n_runs ? min(runs[i].y, kSizeKeys - 1) : -1};
                int place[1];
                align::rank_ids<1>(key, place, s_hist, kSizeKeys, kSizeKeyBits, tid);
                if (i < n_runs) order[place[0]] = i;
            }
        }
        __syncthreads();
        __threadfence_block();
        // 4. the tiles of the two cuts (one pass when both kernels use the same cut), and the plans
        const int t_min = s_sum[0];
        const bool same = s_want[0] == s_want[1];
        for (int k = 0; k < (same ? 1 : 2); ++k) {
            const int extra = max(s_want[k] - t_min, 0);
            if (tid == 0) s_carry[0] = 0;
            __syncthreads();
            for (int base = 0; base < n_runs; base += kPrologueThreads) {
                const int i = base + tid;  // place in the order: the largest runs come first
                int4 r = make_int4(0, 0, 0, 0);
                if (i < n_runs) r = runs[order[i]];
                const int f2 = r.y;
                int n = (f2 + 5) / 6;
                if (i < n_runs) n = min(f2, n + extra / n_runs + (i < extra % n_runs ? 1 : 0));
                const int incl = block_scan(n, s_part);
                const int carry = s_carry[0];
                int t = carry + incl - n, frag = 4 * r.x;
                for (int q = 0; q < n; ++q) {
                    const int fg = f2 / n + (q < f2 % n ? 1 : 0);
                    const int4 tl = make_int4(frag, fg, r.z, 0);
                    if (k == 0) a.tiles[t + q] = tl;
                    if (k == 1 || same) a.tiles_down[t + q] = tl;
                    frag += 2 * fg;
                }
                __syncthreads();
                if (tid == kPrologueThreads - 1) s_carry[0] = carry + incl;
                __syncthreads();
            }
            if (tid == 0) s_tiles[k] = s_carry[0];
            if (tid == 0 && same) s_tiles[1] = s_carry[0];
            __syncthreads();
        }
        if (tid < 2) {
            const int n_wt = tid ? n_wt_down : n_wt_up, n_slabs = (tid ? a.H : a.K) * 2 / tall::kRB;
            KernelPlan kp{};
            kp.n_tiles = s_tiles[tid];
            estimate_kernel(kp.n_tiles, s_sum[4], n_wt, n_slabs, n_cus, kp.parts, kp.tail);
            if (tid == 0) a.plan->up = kp;
            else a.plan->down = kp;
        }
    }
    if (do_invert) {
        const int n_rows = min(a.ntpp[0], a.sorted_num);
        const int stride = (int)(gridDim.x * blockDim.x);
        for (int s = (int)(blockIdx.x * blockDim.x + threadIdx.x); s < n_rows; s += stride) {
            const int p = a.sorted_ids[s];
            const int e = a.expert_ids[s >> 7];  // rows of a block without an expert are not computed
            if (p >= 0 && p < n_pairs && e >= 0 && e < a.E) a.inv[p] = s;
        }
    }
}

template <int FG>
__device__ __forceinline__ void zero_acc(f32x16 (&acc)[2][FG]) {
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int t = 0; t < FG; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[f][t][i] = 0.f;
}

// The part of a tile (first fragment f0, FG pairs of fragments) that part `part` of `parts` takes when a
// tail job is shared by rows: pairs [part FG / parts, (part + 1) FG / parts).  Returns its number of pairs.
__device__ __forceinline__ int row_split(int &f0, int fg, int part, int parts) {
    const int lo = part * fg / parts, hi = (part + 1) * fg / parts;
    f0 += 2 * lo;
    return hi - lo;
}

// Where the partial sums of (part of `parts`, fragment, weight tile) live: 2048 float4 = the two accumulators
// (gate, up) of the four waves that own the fragment, [f][q][wave % 4][lane].  Fragments are numbered through the tiles.
__device__ __forceinline__ float4 *partial_block(const MoeArgs &a, int part, int parts, int frag, int wt) {
    return reinterpret_cast<float4 *>(a.up_partials) + (((int64_t)frag * a.n_wtiles + wt) * parts + part) * 2048;
}

// The queue of an XCD: its workgroups (workgroup w is number w / 8 of XCD w mod 8) start with the slot of their own
// number and take further slots from the XCD's counter, which the prologue sets to the number of workgroups
// per XCD.  Thread 0 asks for the next slot before the last slab but one of a tile (asked much earlier, a busy
// workgroup would hold a job that an idle one could run); `pass` hands it to every thread.
__device__ __forceinline__ int ask_slot(int *counter) { return threadIdx.x == 0 ? atomicAdd(counter, 1) : 0; }
__device__ __forceinline__ int pass_slot(int asked, char *lds) {
    int *word = reinterpret_cast<int *>(lds + tall::kWordOff);
    if (threadIdx.x == 0) *word = asked;
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(*word);
}

// One job of a resident kernel.
struct Work {
    int state;  // 1: a job; 0: the slot is empty; -1: the queue has ended
    int pos, tile, part, parts, wt;
    int e, f0, fg;                  // expert, first token fragment, pairs of fragments (from the row tile)
    int slab0, n_slabs, deep_part;  // its share of the contraction; deep_part < 0: not shared
};
__device__ __forceinline__ Work slot_work(int pos, int n_wt, const KernelPlan &kp) {
    Work w;
    TallJob j;
    w.pos = pos;
    w.state = resolve_tall_job(8 * pos + (int)(blockIdx.x & 7), n_wt, kp, j);
    w.tile = j.tile;
    w.part = j.part;
    w.parts = j.parts;
    w.wt = j.wt;
    return w;
}
// Completes a job with its row tile's entry `tl`.  Only moe_deep_up_kernel takes the branches on kp.deep, here and in
// resolve_tall_job.  In the resident kernels they stand for the sake of the register allocation: with the deep kernel's jobs set
// up by code of its own, and no such branch, the compiler spills 33 registers of the resident up kernel and 3 of the down
// kernel instead of none, and the layers take longer: 4096 tokens on 8 experts of K 4096 x N 28672 2424 -> 2977 us, 8192 on 128 of
// K 2048 x N 1536 729 -> 772, 131072 on 32 of K = N = 2048 5832 -> 7782 (the README layer at 400 to 3000 tokens: the same).
__device__ __forceinline__ void tile_work(Work &w, const int4 &tl, const KernelPlan &kp, int n_slabs) {
    w.f0 = __builtin_amdgcn_readfirstlane(tl.x);
    w.fg = __builtin_amdgcn_readfirstlane(tl.y);
    w.e = __builtin_amdgcn_readfirstlane(tl.z);
    w.slab0 = 0;
    w.n_slabs = n_slabs;
    w.deep_part = -1;
    if (kp.deep) {
        w.slab0 = w.part * n_slabs / w.parts;
        w.n_slabs = (w.part + 1) * n_slabs / w.parts - w.slab0;
        w.deep_part = w.part;
    } else if (w.parts > 1) {
        w.fg = row_split(w.f0, w.fg, w.part, w.parts);
        if (w.fg == 0) w.state = 0;
    }
}
// Workgroups that run side by side start their K walks at different slabs.
__device__ __forceinline__ int k_start(const Work &w) { return (w.pos & 7) % w.n_slabs; }

// Hand-over from tile to tile.  A workgroup fills the LDS of its CU, so nothing else runs while a tile is set up,
// waits for its first slab and stores its results.  The next job is therefore looked up, and the copies of its first
// slabs are issued, under the epilogue of the current one, whose waves transpose through a few KB of their own
// (no barriers) behind the stages that are being filled.  The lookup is a chain (slot -> row tile entry -> row
// ids of the gather -> copies) whose links are spread over the first fragments of the epilogue:
//   epilogue(q): fragment q of the wave's FG;  link(0) .. link(kLinks - 1): the links, in order.
template <int FG, int kLinks, typename Epilogue, typename Link>
__device__ __forceinline__ void epilogue_with_links(Epilogue epilogue, Link link) {
    link(0);
#pragma unroll
    for (int t = 0; t < FG; ++t) {
        epilogue(t);
        PMOE_TALL_FENCE();
        if (t + 1 < kLinks) link(t + 1);
    }
#pragma unroll
    for (int l = FG + 1; l < kLinks; ++l) link(l);
}

// LDS written by some lanes of a wave is read by others of the same wave: LDS operations of a wave are executed in
// order, only the compiler has to keep them so.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Up kernel tile: token fragments f0 .. f0 + 2 FG - 1 x activation columns [128 wt, 128 wt + 128) of expert e,
// contraction slabs [slab0, slab0 + n_slabs).  LDS weight rows 0..127 are gate rows, 128..255 the matching up
// rows; wave v of a group owns gate/up rows 32v..32v+31, so gate and up of one activation element sit in the
// same lane and register: SwiGLU in registers, the 2H-wide tensor never leaves the chip.
// QUEUE = false (deep mode): the workgroup has this one job, whose contraction is shared; the fp32 sums go to up_partials
// instead, from fragment number `deep_frag` on.
// `pre`: the first slabs are on their way (tok_ahead: the offsets of their token rows); `next` returns the
// job after this one, with `pre` and tok_ahead for it.
struct UpTile {
    const char *x, *w_gate, *w_up;
    uint32_t row_bytes;
};
__device__ __forceinline__ UpTile up_operands(const MoeArgs &a, const Work &w) {
    UpTile u;
    u.row_bytes = (uint32_t)a.K * 2u;
    u.x = a.x + w.slab0 * tall::kRB;
    u.w_gate = a.w1 + ((int64_t)w.e * a.N + w.wt * 128) * a.K * 2 + w.slab0 * tall::kRB;
    u.w_up = u.w_gate + (int64_t)a.H * a.K * 2;
    return u;
}
// Byte offset in x of the token of pair id `p`, and of that of sorted row `s`; dead rows read token 0.
__device__ __forceinline__ uint32_t token_off(const MoeArgs &a, int p, uint32_t row_bytes) {
    return ((uint32_t)p < (uint32_t)(a.M * a.top_k) ? (uint32_t)p / (uint32_t)a.top_k : 0u) * row_bytes;
}
__device__ __forceinline__ uint32_t gather_off(const MoeArgs &a, int64_t s, uint32_t row_bytes) {
    return token_off(a, s < a.sorted_num ? a.sorted_ids[s] : -1, row_bytes);
}
template <int FG, bool QUEUE = true>
__device__ __forceinline__ void up_tile_tall(const MoeArgs &a, const KernelPlan &kp, const Work &w, int *counter, char *lds,
                                             bool &pre, uint32_t (&tok_ahead)[tall::kMaxFrags / 2], Work &next,
                                             int deep_frag = 0) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = wave >> 2, w4 = wave & 3;
    const int H = a.H;
    const int h0 = w.wt * 128;
    const int64_t row0 = (int64_t)w.f0 * 32;
    const UpTile u = up_operands(a, w);
    tall::Loader<FG, true> ld;
    ld.setup(tid, u.x, u.w_gate, u.w_up, u.row_bytes, u.row_bytes,
             [&](int row) { return gather_off(a, row0 + row, u.row_bytes); }, pre || !QUEUE ? tok_ahead : nullptr);
    const int wrow[2] = {32 * w4, 128 + 32 * w4};
    f32x16 acc[2][FG];
    zero_acc<FG>(acc);
    int asked = 0;
    tall::main_loop<FG>(acc, ld, lds, w.n_slabs, wrow, grp * FG, lane, k_start(w), pre,
                        [&] {
                            if constexpr (QUEUE) asked = ask_slot(counter);
                        },
                        [] {});

    int lane_e = lane;
    asm volatile("" : "+v"(lane_e));
    const int r = lane_e & 31, half = lane_e >> 5;
    if constexpr (!QUEUE) {
#pragma unroll
        for (int t = 0; t < FG; ++t) {
            float4 *dst = partial_block(a, w.deep_part, w.parts, deep_frag + grp * FG + t, w.wt);
#pragma unroll
            for (int f = 0; f < 2; ++f)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    dst[((f * 4 + q) * 4 + w4) * 64 + lane_e] =
                        make_float4(acc[f][t][4 * q], acc[f][t][4 * q + 1], acc[f][t][4 * q + 2], acc[f][t][4 * q + 3]);
        }
        return;
    }
    char *scratch = lds + tall::kScratchOff + wave * tall::kScratchBytes;
    constexpr int kPitch = 80;  // 32 activation columns + 16 B pad
    int4 tl = make_int4(0, 0, 0, 0);
    pre = false;
    epilogue_with_links<FG, 3>(
        [&](int t) {
            // register i of lane_e l = activation column 32 w4 + 8(i/4) + 4(l/32) + i%4 of token row 32 t + l%32
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                uint2 pk;
                pk.x = pack2_bf16(swiglu(acc[0][t][4 * g], acc[1][t][4 * g]), swiglu(acc[0][t][4 * g + 1], acc[1][t][4 * g + 1]));
                pk.y = pack2_bf16(swiglu(acc[0][t][4 * g + 2], acc[1][t][4 * g + 2]),
                                  swiglu(acc[0][t][4 * g + 3], acc[1][t][4 * g + 3]));
                *reinterpret_cast<uint2 *>(scratch + r * kPitch + 16 * g + 8 * half) = pk;
            }
            wave_lds_order();
            // 64 bytes of a row by 4 lanes, to the activation rows (by sorted row)
            char *dst = a.act + ((row0 + (grp * FG + t) * 32) * H + h0 + 32 * w4) * 2 + (lane_e & 3) * 16;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int row = (lane_e >> 2) + 16 * i;
                const uint4 v = *reinterpret_cast<const uint4 *>(scratch + row * kPitch + (lane_e & 3) * 16);
                *reinterpret_cast<uint4 *>(dst + (int64_t)row * H * 2) = v;
            }
            wave_lds_order();
        },
        [&](int link) {
            if (link == 0) {
                next = slot_work(pass_slot(asked, lds), a.n_wtiles, kp);
                if (next.state > 0) tl = a.tiles[next.tile];
            } else if (link == 1) {
                if (next.state > 0) tile_work(next, tl, kp, a.K * 2 / tall::kRB);
                if (next.state > 0) {
                    const int row = 8 * wave + (lane_e >> 3);
                    const uint32_t chunk = (uint32_t)((lane_e & 7) ^ ((row >> 1) & 7)) * 16u;
#pragma unroll
                    for (int q = 0; q < tall::kMaxFrags / 2; ++q)
                        if (q < next.fg) tok_ahead[q] = gather_off(a, (int64_t)next.f0 * 32 + row + 64 * q, u.row_bytes) + chunk;
                    pre = true;
                }
            } else if (next.state > 0) {
                const UpTile n = up_operands(a, next);
                tall::pre_issue<true>(next.fg, lds, wave, lane_e, n.x, n.w_gate, n.w_up, n.row_bytes, n.row_bytes, tok_ahead,
                                      next.n_slabs, k_start(next));
            }
        });
}

// The walk of a resident kernel over its queue; tile<FG>() runs a tile and finds the next job.
template <typename Run>
__device__ __forceinline__ void walk_queue(const KernelPlan &kp, const int4 *tiles, int n_wt, int n_slabs, int *counter,
                                           char *lds, Run run) {
    Work w = slot_work((int)(blockIdx.x >> 3), n_wt, kp);
    if (w.state > 0) tile_work(w, tiles[w.tile], kp, n_slabs);
    while (w.state >= 0) {
        if (w.state == 0) {
            __syncthreads();  // the word may still be read
            w = slot_work(pass_slot(ask_slot(counter), lds), n_wt, kp);
            if (w.state > 0) tile_work(w, tiles[w.tile], kp, n_slabs);
            continue;
        }
        Work next;
        run(w, next);
        w = next;
    }
}

__global__ __launch_bounds__(512) void moe_up_kernel_bf16(MoeArgs a) {
    __shared__ __attribute__((aligned(1024))) char lds[tall::kLdsBytes];
    if (a.crowd && !(crowding(a, a.ntpp[0]) & 1)) return;
    const KernelPlan kp = a.plan->up;
    int *counter = &a.plan->counters[blockIdx.x & 7];
    bool pre = false;
    uint32_t tok_ahead[tall::kMaxFrags / 2] = {};
    walk_queue(kp, a.tiles, a.n_wtiles, a.K * 2 / tall::kRB, counter, lds, [&](const Work &w, Work &next) {
        switch (w.fg) {
            case 1: up_tile_tall<1>(a, kp, w, counter, lds, pre, tok_ahead, next); break;
            case 2: up_tile_tall<2>(a, kp, w, counter, lds, pre, tok_ahead, next); break;
            case 3: up_tile_tall<3>(a, kp, w, counter, lds, pre, tok_ahead, next); break;
            case 4: up_tile_tall<4>(a, kp, w, counter, lds, pre, tok_ahead, next); break;
            case 5: up_tile_tall<5>(a, kp, w, counter, lds, pre, tok_ahead, next); break;
            default: up_tile_tall<6>(a, kp, w, counter, lds, pre, tok_ahead, next); break;
        }
    });
}

// Few up jobs (at most kDeepJobs (block, weight tile) pairs, K >= 2048).  All of them together leave most CUs idle, so every
// job's contraction is shared among up to kDeepParts workgroups, which store fp32 partial sums; moe_up_join_kernel adds them in
// part order and applies SwiGLU.  There are at most 64 blocks: a wave of every workgroup works out the row tiles (a lane per
// block) while the last workgroup writes what the kernels behind need, and no prologue runs in front.
// What bounds a workgroup is a chain: 1.4 us until it has the last rows of the blocks, 0.9 to cut them, 1.3 to its first
// copies, 2 - 3 until these land, 0.7 - 1 per slab of its share of K, 1 for the sums.  So the tiles are small, one
// pair of fragments or two: there are more busy CUs than with tiles of up to six pairs, a slab takes 0.72 instead of 1.0
// us, and fewer sums leave through each CU (a run of blocks has at most twice as many pairs as blocks, so tiles of two
// leave the jobs of 32 (block, weight tile) pairs their eight parts on 256 CUs, those of 128 two).  Of eight parts, part p of every
// job runs on XCD p, and the weight rows that two tiles of a run share come from one L2.  The token rows are gathered by the ids
// read for the plan.  8 experts of K 4096, N 512, top 4, the layer at 256 tokens 41.7 -> 39.8 us (this kernel 18.6 -> 17.4),
// with up to six / up to two pairs a tile.  With 12 and 16 parts the K
// loop is shorter by what the sums are longer: 25.1 and 25.2 us with the join instead of 23.6 (six pairs a tile).
struct DeepTiles {
    int4 tile[kDeepBlocks];  // {first fragment, pairs of fragments, expert, first fragment's number}
    int rows[kDeepBlocks];   // of every block: 1 + its last live row
    int ids[kDeepBlocks * kBlockRows];  // sorted ids: the rows of a tile are gathered by them
    KernelPlan plan;
};
__global__ __launch_bounds__(512) void moe_deep_up_kernel(MoeArgs a, int n_wt_down, int n_cus, int plan_only) {
    __shared__ __attribute__((aligned(1024))) char lds[tall::kLdsBytes];
    DeepTiles &s = *reinterpret_cast<DeepTiles *>(lds);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned n_pairs = (unsigned)(a.M * a.top_k);
    const int n_slabs = a.K * 2 / tall::kRB;
    const int ntpp = a.ntpp[0], e_all = lane < a.n_blocks ? a.expert_ids[lane] : -1;
    // the last live row of every block: four blocks of a wave in flight
    for (int b0 = wave; b0 < a.n_blocks; b0 += 32) {
        int id[4][2];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t at = (int64_t)(b0 + 8 * u) * kBlockRows + lane;
            id[u][0] = at < a.sorted_num ? a.sorted_ids[at] : -1;
            id[u][1] = at + 64 < a.sorted_num ? a.sorted_ids[at + 64] : -1;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int blk = b0 + 8 * u;
            if (blk >= a.n_blocks) break;
            const uint64_t m0 = __ballot((unsigned)id[u][0] < n_pairs), m1 = __ballot((unsigned)id[u][1] < n_pairs);
            s.ids[blk * kBlockRows + lane] = id[u][0];
            s.ids[blk * kBlockRows + 64 + lane] = id[u][1];
            if (lane == 0) s.rows[blk] = m1 ? 128 - __builtin_clzll(m1) : m0 ? 64 - __builtin_clzll(m0) : 0;
        }
    }
    __syncthreads();
    if (wave == 0) {
        const int n_live = min((ntpp + kBlockRows - 1) / kBlockRows, a.n_blocks);
        const bool live = lane < n_live;
        const int e = live ? e_all : -1;
        const int before = __shfl_up(e, 1, 64);  // (with all lanes active: a lane that is switched off hands out 0)
        const uint64_t starts = __ballot(live && (lane == 0 || before != e));
        const bool last = live && (lane + 1 == n_live || ((starts >> (lane + 1)) & 1));
        const int run = 63 - __builtin_clzll((starts & ((2ull << lane) - 1)) | 1);  // first block of the lane's run
        const int f2 = last && e >= 0 && e < a.E ? ((lane - run) * kBlockRows + s.rows[lane] + 63) >> 6 : 0;
        const int n = (f2 + 5) / 6;
        const int halves = (f2 + 1) / 2;  // tiles of two pairs
        // tiles, runs, pairs of fragments and tiles of two pairs (at most 64, 64, 128 and 64) up to and including this lane,
        // added up together
        auto up_to = [&](int v) {
#pragma unroll
            for (int d = 1; d < kDeepBlocks; d <<= 1) {
                const int t = __shfl_up(v, d, 64);
                if (lane >= d) v += t;
            }
            return v;
        };
        const int sums = up_to(n | (f2 > 0 ? 1 << 8 : 0) | f2 << 16 | halves << 24), all = __shfl(sums, kDeepBlocks - 1, 64);
        const int tiles = sums & 0xff, runs = (sums >> 8) & 0xff, pairs = (sums >> 16) & 0xff;
        const int n_tiles = all & 0xff, n_runs = (all >> 8) & 0xff, n_f2 = (all >> 16) & 0xff;
        auto cut = [&](int4 *dst, int at, int count) {  // this lane's run in `count` tiles
            int frag = 4 * run, number = 2 * (pairs - f2);
            for (int q = 0; q < count; ++q) {
                const int fg = f2 / count + (q < f2 % count ? 1 : 0);
                dst[at + q] = make_int4(frag, fg, e, number);
                frag += 2 * fg;
                number += 2 * fg;
            }
        };
        // The up kernel's tiles: one pair of fragments where that leaves a workgroup for every part of every job, or two (of
        // which there are never more than blocks; more than 64 of one pair would take 520 CUs, and have no room in the table).
        const bool single = n_f2 <= kDeepBlocks && n_f2 * a.n_wtiles * kDeepParts <= (int)gridDim.x;
        const int n_up = single ? f2 : halves, n_up_tiles = single ? n_f2 : all >> 24;
        cut(s.tile, (single ? pairs : sums >> 24) - n_up, n_up);
        KernelPlan kp{};
        kp.n_tiles = n_up_tiles;
        kp.deep = 1;
        kp.parts = min(min(kDeepParts, n_slabs / 4), (int)gridDim.x / max(n_up_tiles * a.n_wtiles, 1));
        kp.parts = max(1, min(kp.parts, kDeepSums / max(2 * n_f2 * a.n_wtiles, 1)));
        if (lane == 0) s.plan = kp;
        if (blockIdx.x == gridDim.x - 1) {
            // for the kernels behind: the down kernel's tiles and queues, the plans, the sorted numbers of the fragments
            const int want = choose_tiles(n_tiles, a.n_blocks, n_f2, n_wt_down, a.H * 2 / tall::kRB, n_cus), extra = max(want - n_tiles, 0);
            const int mine = f2 > 0 ? min(f2, n + extra / n_runs + (runs <= extra % n_runs ? 1 : 0)) : 0;
            const int at = up_to(mine), n_down = __shfl(at, kDeepBlocks - 1, 64);
            cut(a.tiles_down, at - mine, mine);
            int *numbers = reinterpret_cast<int *>(a.runs);
            for (int q = 0; q < 2 * f2; ++q) numbers[2 * (pairs - f2) + q] = 4 * run + q;
            if (lane < 8) a.plan->counters[8 + lane] = n_cus / 8;
            if (lane == 0) {
                KernelPlan down{};
                down.n_tiles = n_down;
                estimate_kernel(n_down, n_f2, n_wt_down, a.H * 2 / tall::kRB, n_cus, down.parts, down.tail);
                a.plan->up = kp;
                a.plan->down = down;
                a.plan->deep_frags = 2 * n_f2;
            }
        }
    }
    __syncthreads();
    KernelPlan kp{};
    kp.n_tiles = __builtin_amdgcn_readfirstlane(s.plan.n_tiles);
    kp.parts = __builtin_amdgcn_readfirstlane(s.plan.parts);
    kp.deep = 1;
    Work w = slot_work((int)(blockIdx.x >> 3), a.n_wtiles, kp);
    // The sorted order is inverted by the workgroups without a job, or by all of them at the end.
    const int busy = kp.n_tiles * a.n_wtiles * kp.parts, first = !plan_only && (int)gridDim.x - busy >= 16 ? busy : 0;
    if (plan_only || w.state <= 0) {
        if ((int)blockIdx.x >= first) stream::invert(a, 512, first);
        return;
    }
    const int4 tl = s.tile[w.tile];
    const int deep_frag = __builtin_amdgcn_readfirstlane(tl.w);
    tile_work(w, tl, kp, n_slabs);
    bool pre = false;
    uint32_t tok_ahead[tall::kMaxFrags / 2] = {};
    {
        const int row = 8 * wave + (lane >> 3);
        const uint32_t chunk = (uint32_t)((lane & 7) ^ ((row >> 1) & 7)) * 16u;
#pragma unroll
        for (int q = 0; q < 2; ++q)
            if (q < w.fg) tok_ahead[q] = token_off(a, s.ids[w.f0 * 32 + row + 64 * q], (uint32_t)a.K * 2u) + chunk;
    }
    __syncthreads();  // the tiles and ids have been read: the ring may be filled
    Work next;
    if (w.fg == 1) up_tile_tall<1, false>(a, kp, w, nullptr, lds, pre, tok_ahead, next, deep_frag);
    else up_tile_tall<2, false>(a, kp, w, nullptr, lds, pre, tok_ahead, next, deep_frag);
    if (first == 0) stream::invert(a, 512);
}

// Adds the partial sums the parts of every up job left in memory and finishes the tiles.  One
// workgroup of 4 waves per (fragment, weight tile, quarter of the accumulator registers):
// thread (v, lane) takes over registers 4q .. 4q + 3 of what thread (v, lane) of the fragment's group held, gate
// and up sums, adds the parts in part order, applies SwiGLU and writes its 4 activation values.  All loads of
// a thread are in flight together: the kernel is one memory latency long.
__global__ __launch_bounds__(256) void moe_up_join_kernel(MoeArgs a) {
    const int q = blockIdx.x & 3, b = (int)blockIdx.x >> 2;
    const int number = b / a.n_wtiles, wt = b - number * a.n_wtiles;
    const int parts = a.plan->up.parts;
    const int frag = reinterpret_cast<const int *>(a.runs)[number];
    if (number >= a.plan->deep_frags) return;
    const int tid = threadIdx.x, lane = tid & 63, v = tid >> 6;
    float4 vg[kDeepParts], vu[kDeepParts];
    const float4 *src = partial_block(a, 0, parts, number, wt) + (q * 4 + v) * 64 + lane;
#pragma unroll
    for (int p = 0; p < kDeepParts; ++p)
        if (p < parts) {
            vg[p] = src[p * 2048];
            vu[p] = src[p * 2048 + 1024];
        }
    float g[4] = {0.f, 0.f, 0.f, 0.f}, u[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int p = 0; p < kDeepParts; ++p)
        if (p < parts) {
            g[0] += vg[p].x; g[1] += vg[p].y; g[2] += vg[p].z; g[3] += vg[p].w;
            u[0] += vu[p].x; u[1] += vu[p].y; u[2] += vu[p].z; u[3] += vu[p].w;
        }
    const int hl = 32 * v + 8 * q + 4 * (lane >> 5);  // tile-local activation column, as in up_tile_tall
    uint2 pk;
    pk.x = pack2_bf16(swiglu(g[0], u[0]), swiglu(g[1], u[1]));
    pk.y = pack2_bf16(swiglu(g[2], u[2]), swiglu(g[3], u[3]));
    *reinterpret_cast<uint2 *>(a.act + (((int64_t)frag * 32 + (lane & 31)) * a.H + wt * 128 + hl) * 2) = pk;
}

// Down kernel tile: y[pairs of the tile's rows, 256 columns of K from 256 wt] = act[rows, :H] . W2[e][cols, :H]^T,
// the whole reduction over H inside the workgroup; the routing weights are applied later, by finalize_kernel.
// Weight rows (output columns) sit on the MFMA M side: register i of lane l = output column
// 64 w4 + 32 f + 8(i/4) + 4(l/32) + i%4 of tile row 32 t + l%32.  A wave rounds a fragment of its 64 columns to
// bf16, transposes it through its LDS scratch and stores whole 128-byte lines to y[pair id]; rows without a pair
// are skipped.
struct DownTile {
    const char *act, *w_lo, *w_hi;
    uint32_t row_bytes;
};
__device__ __forceinline__ DownTile down_operands(const MoeArgs &a, const Work &w) {
    DownTile d;
    d.row_bytes = (uint32_t)a.H * 2u;
    d.act = a.act + (int64_t)w.f0 * 32 * d.row_bytes;
    // weight rows (output columns) k0 .. k0 + 255 of the expert; the last tile of a K that is not a multiple
    // of 256 has 128 of them and reads the first half twice
    const int k0 = w.wt * kWRows;
    d.w_lo = a.w2 + ((int64_t)w.e * a.K + k0) * d.row_bytes;
    d.w_hi = (k0 + 128 < a.K) ? d.w_lo + (int64_t)128 * d.row_bytes : d.w_lo;
    return d;
}
template <int FG>
__device__ __forceinline__ void down_tile_tall(const MoeArgs &a, const KernelPlan &kp, const Work &w, int *counter, char *lds,
                                               bool &pre, Work &next) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = wave >> 2, w4 = wave & 3;
    const int K = a.K;
    const int k0 = w.wt * kWRows;
    const DownTile d = down_operands(a, w);
    tall::Loader<FG, false> ld;
    ld.setup(tid, d.act, d.w_lo, d.w_hi, d.row_bytes, d.row_bytes, [&](int row) { return (uint32_t)row * d.row_bytes; });
    const int wrow[2] = {64 * w4, 64 * w4 + 32};
    f32x16 acc[2][FG];
    zero_acc<FG>(acc);
    int asked = 0;
    // pair ids of the wave's 32 FG rows, one per lane; fetched before the last slab, in the registers its loader no
    // longer needs
    constexpr int NP = (FG + 1) / 2;
    int pairs[NP];
    tall::main_loop<FG>(acc, ld, lds, w.n_slabs, wrow, grp * FG, lane, k_start(w), pre, [&] { asked = ask_slot(counter); },
                        [&] {
#pragma unroll
                            for (int q = 0; q < NP; ++q) {
                                const int64_t s = (int64_t)w.f0 * 32 + grp * 32 * FG + 64 * q + lane;
                                pairs[q] = (64 * q + lane < 32 * FG && s < a.sorted_num) ? a.sorted_ids[s] : -1;
                            }
                        });
    // (they are here before the copies of the next tile queue up behind them)
#pragma unroll
    for (int q = 0; q < NP; ++q) asm volatile("" : "+v"(pairs[q]));

    // (the epilogue's addresses are computed from a lane number that the compiler knows nothing about: it would keep
    // them in registers across the K loop, that is spill them, and a reload here waits for the copies in flight)
    int lane_e = lane;
    asm volatile("" : "+v"(lane_e));
    const int r = lane_e & 31, half = lane_e >> 5;
    const bool in_cols = k0 + 64 * w4 < K;  // (K is a multiple of 128: a wave's 64 columns are inside or outside)
    const uint32_t n_pairs = (uint32_t)(a.M * a.top_k);
    char *scratch = lds + tall::kScratchOff + wave * tall::kScratchBytes;
    constexpr int kPitch = 144;  // 64 columns + 16 B pad
    char *dst = a.y + (int64_t)(k0 + 64 * w4) * 2 + (lane_e & 7) * 16;
    int4 tl = make_int4(0, 0, 0, 0);
    pre = false;
    epilogue_with_links<FG, 2>(
        [&](int t) {
#pragma unroll
            for (int f = 0; f < 2; ++f)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    uint2 pk;
                    pk.x = pack2_bf16(acc[f][t][4 * q], acc[f][t][4 * q + 1]);
                    pk.y = pack2_bf16(acc[f][t][4 * q + 2], acc[f][t][4 * q + 3]);
                    *reinterpret_cast<uint2 *>(scratch + r * kPitch + 64 * f + 16 * q + 8 * half) = pk;
                }
            wave_lds_order();
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = (lane_e >> 3) + 8 * i;
                const int p = __shfl(pairs[t / 2], 32 * (t & 1) + row, 64);
                const uint4 v = *reinterpret_cast<const uint4 *>(scratch + row * kPitch + (lane_e & 7) * 16);
                if (in_cols && (uint32_t)p < n_pairs) store_once(dst + (int64_t)p * K * 2, v);
            }
            wave_lds_order();
        },
        [&](int link) {
            if (link == 0) {
                next = slot_work(pass_slot(asked, lds), a.n_wtiles, kp);
                if (next.state > 0) tl = a.tiles_down[next.tile];
            } else {
                if (next.state > 0) tile_work(next, tl, kp, a.H * 2 / tall::kRB);
                if (next.state > 0) {
                    const DownTile n = down_operands(a, next);
                    const int row = 8 * wave + (lane_e >> 3);
                    const uint32_t off = (uint32_t)row * n.row_bytes + (uint32_t)((lane_e & 7) ^ ((row >> 1) & 7)) * 16u;
                    tall::pre_issue<false>(next.fg, lds, wave, lane_e, n.act, n.w_lo, n.w_hi, n.row_bytes, n.row_bytes, &off,
                                           next.n_slabs, k_start(next));
                    pre = true;
                }
            }
        });
}

__global__ __launch_bounds__(512) void moe_down_kernel_bf16(MoeArgs a) {
    __shared__ __attribute__((aligned(1024))) char lds[tall::kLdsBytes];
    if (a.crowd && !(crowding(a, a.ntpp[0]) & 2)) return;
    const KernelPlan kp = a.plan->down;
    int *counter = &a.plan->counters[8 + (blockIdx.x & 7)];
    bool pre = false;
    walk_queue(kp, a.tiles_down, a.n_wtiles, a.H * 2 / tall::kRB, counter, lds, [&](const Work &w, Work &next) {
        switch (w.fg) {
            case 1: down_tile_tall<1>(a, kp, w, counter, lds, pre, next); break;
            case 2: down_tile_tall<2>(a, kp, w, counter, lds, pre, next); break;
            case 3: down_tile_tall<3>(a, kp, w, counter, lds, pre, next); break;
            case 4: down_tile_tall<4>(a, kp, w, counter, lds, pre, next); break;
            case 5: down_tile_tall<5>(a, kp, w, counter, lds, pre, next); break;
            default: down_tile_tall<6>(a, kp, w, counter, lds, pre, next); break;
        }
    });
}

// Weight-streaming kernels (moe_stream.h).  n_tiles: weight tiles per block (0: the up kernel only inverts).  CROWD: tall
// kernels are enqueued too.  (An instantiation of its own: with the test in both, the calls without tall kernels took up to 2 us
// longer, 97 tokens x top 9 on 257 experts of K 7168 x N 512 455.8 us instead of 454.1.)
template <bool UP, int U, bool CROWD>
__global__ __launch_bounds__(512, 4) void moe_stream_kernel(MoeArgs a, int n_tiles) {
    __shared__ __attribute__((aligned(1024))) stream::Shared sh;
    stream::for_each_job<UP>(a, n_tiles, [&](int ntpp) { return CROWD && (crowding(a, ntpp) & (UP ? 1 : 2)) != 0; },
                             [&](int blk, int e, int tile, int id) { stream::run_job<UP, U>(a, sh, blk, e, tile, id); });
}

// Down GEMM of the streaming path for H = RB / 2 (see stream::for_each_turn).
template <int RB>
__global__ __launch_bounds__(256, RB == 256 ? 4 : 2) void moe_stream_down_short_kernel(MoeArgs a) {
    __shared__ __attribute__((aligned(1024))) char bufs[4][stream::ShortDown<RB>::kBytes];
    if (a.crowd && (crowding(a, a.ntpp[0]) & 2)) return;
    stream::ShortDown<RB> eng(a, bufs[__builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6)]);
    stream::for_each_turn(a, a.K / 32, eng);
}

// A handful of pairs (moe_few.h).  The down kernel ends the pipeline, nothing is left for finalize.
__global__ __launch_bounds__(64) void moe_few_up_kernel(MoeArgs a) {
    const int n_tiles = a.H / 4;
    int j = (int)blockIdx.x, blk = j / n_tiles;
    few::Block b = few::request_block(a, blk);
    const int n_rows = few::schedule_rows(a), n_live = (n_rows + kBlockRows - 1) / kBlockRows;
    while (j < n_live * n_tiles) {
        few::up_job(a, b, blk, j - blk * n_tiles, n_rows);
        j += (int)gridDim.x;
        blk = j / n_tiles;
        b = few::request_block(a, blk);
    }
}
__global__ __launch_bounds__(512) void moe_few_down_kernel(MoeArgs a, char *out, int blocks, int accumulate) {
    __shared__ few::DownShared sh;
    for (int j = (int)blockIdx.x; j < a.K / 8; j += (int)gridDim.x) few::down_job(a, sh, j, blocks, out, accumulate != 0);
}

// ------------------------------------------------------------------------------------------ host

// One token or two: weights straight into registers.  Whole layer, streaming kernels / these, us: K 2048, N 1536, 8 of 128
// experts 29.7 / 23.7 at 1 token, 39.2 / 36.0 at 2; K 4096, N 512, 4 of 8 24.3 / 16.6, 25.4 / 21.0; K 4096, N 28672, 2 of 8 121.8 /
// 115.9, 193.7 / 171.9.  The op alone: K 4096, N 4096, 2 of 64 at 2 tokens 41.5 / 38.3, both on the same two experts 26.3 / 27.5.
// From three tokens on blocks have more rows than are multiplied at a time, and the weights are read again: 53.4 / 47.6 at
// 3 tokens on 128 experts, but all on the same 8 21.8 / 30.0.  With K beyond 4096 a CU has more than two workgroups' worth of
// output columns, whose latencies add up: K 7168, N 4096, 1 token 116 / 124 (down kernel 41 / 50), N 512, 2 tokens 38 / 44.
// What a call gains is a fixed 5 to 7 us of latency; what it loses grows with the pairs.  The op on weights that are not in the
// caches, streaming / these, us:
//  * up to four pairs these are faster nearly everywhere: K 2048, N 1536 17.1 / 13.9 at 4, K 512, N 512 11.3 / 7.6; at worst
//    K 2048, N 8192 41.8 / 43.0 at 4;
//  * a workgroup of the down kernel has 8 output columns, and with fewer workgroups than CUs the others idle while it reads
//    pairs x N x 8 bytes: kFewIdle is what that may cost.  K 512, N 1536 18.6 / 17.9 at 16 pairs, 26.9 / 31.1 at 32; K 512, N 4096
//    20.6 / 20.1 at 8, 29.1 / 34.2 at 16; K 1024, N 2048 27.7 / 27.1 at 16, 43.5 / 45.9 at 32; K 1024, N 4096 26.6 / 27.0 at 8,
//    42.6 / 45.4 at 16;
//  * with more workgroups than CUs every step of a workgroup is paid twice: K 4096, N 512 22.5 / 21.2 at 8 pairs, 29.1 / 31.4 at 16,
//    N 1536 38.0 / 34.3 at 8, 59.2 / 59.9 at 16; N 2048 43.0 / 42.8 at 8, and 26.3 / 27.9 where two tokens share their four experts;
//  * of more than eight blocks a wave takes several, one behind the other, and each has to be long: K 2048, N 512 20.1 / 19.7 at 16
//    pairs, 30.1 / 30.9 at 32, N 1024 28.6 / 26.9 and 45.6 / 43.6; K 512, N 512 14.3 / 13.0 and 17.5 / 19.7; K 1024, N 1024
//    20.6 / 18.6 and 29.3 / 30.8 (with less room for idle CUs, too);
//  * large experts stream at the rate of memory either way: K 2048, N 4096 42.8 / 40.9 at 8 pairs, N 8192 73.8 / 74.0 (40.4 / 44.1
//    where two tokens share their four experts), 140 / 135 at 16.
constexpr int64_t kFewIdle = 50 << 20;
static bool use_few(const MoeArgs &a) {
    if (a.M > 2 || a.K > 4096 || a.n_blocks == 0) return false;
    const int64_t pairs = (int64_t)a.M * a.top_k, idle = 8 * resident_grid() - a.K;  // output columns the CUs have room for beside K
    if (pairs <= 4) return true;
    if (idle < 0) return pairs <= 8 && a.N <= 1536;
    if (pairs <= 16) return pairs * a.N * idle <= kFewIdle;
    return pairs <= few::kMaxPairs && a.N >= 1024 && pairs * a.N * idle <= kFewIdle / 4;
}
static int launch_few_pipeline(const MoeArgs &a, void *out, int split, hipStream_t s) {
    const int mask = phase_mask();
    const int64_t blocks = std::min<int64_t>(a.n_blocks, std::min<int64_t>(a.E, (int64_t)a.M * a.top_k));
    if (mask & PMOE_PHASE_UP)
        hipLaunchKernelGGL(moe_few_up_kernel, dim3((unsigned)std::min<int64_t>(blocks * (a.H / 4), 1 << 16)), dim3(64), 0, s, a);
    if (mask & PMOE_PHASE_DOWN)
        hipLaunchKernelGGL(moe_few_down_kernel, dim3(a.K / 8), dim3(512), 0, s, a, static_cast<char *>(out), (int)blocks, split ? 0 : 1);
    return check_launch("fused_moe_bf16 launch");
}

// A workgroup of moe_deep_up_kernel has one job and comes back for no other: the grid holds every job, however the blocks
// fall into tiles, and shares it between two workgroups at least.  Prologue and resident kernel / deep mode, whole layer, us: 8
// experts of K 4096, N 512, top 4: 63.2 / 43.7 at 280 tokens (17 blocks), 75.3 / 46.8 at 400, 78.9 / 57.9 at 600, 88.7 / 57.8 at 770, 89.0 /
// 72.1 at 1000, 98.4 / 82.4 at 1400, 111.8 / 95.3 at 1790 (64 blocks); one of N 2048 82.9 / 62.3 at 1000 tokens; 2 of N 4096 73.7 / 62.8 at
// 300; 4 of K 2048, N 1024, top 2 58.3 / 50.5 at 1000; 4 of K 7168, N 2048 121.3 / 86.1 at 500.
static bool use_deep(const MoeArgs &a) { return a.deep_ok && a.n_blocks > 0 && 2 * a.n_blocks * (a.H / 128) <= resident_grid(); }

// Few rows per expert on average: what the problem costs is the stream of the weights (moe_stream.h).  Whole op,
// stream against tall tiles, us (graph replays): 8 large experts (K 4096, N 28672, top 2) 117 / 300 at 1 token, 424 /
// 567 at 32, 487 / 570 at 128 (32 rows per expert), 576 / 573 at 192; 128 small experts (K 2048, N 1536, top 8) 24 /
// 45 at 1 token, 163 / 232 at 64, 251 / 264 at 384, 285 / 282 at 512 (32 rows per expert), 343 / 293 at 768.
// With few jobs of tall tiles and no deep mode to share them it pays longer (37 experts, K 4096, N 256, top 9: 74 / 121
// at 256 tokens, 62 rows per expert).  With the deep mode for up to 32 (block, weight tile) pairs it ends at 32 rows; beyond, the
// deep mode is the faster one where the contraction is long and the weight tiles are one or two.  How early depends on the bytes of
// the weights, which streaming reads once per 32 or 64 rows: from 34 rows per expert on with 112 MB or more, behind 48 with less.  Stream /
// deep at 35, 44 and 58 rows, whole layer, us: K 4096, 16 experts of N 512 (101 MB) 39.4 / 41.7, 41.5 / 42.0 and 51.0 / 43.5, 28 of N 256 (88
// MB) 43.2 / 44.7, 46.5 / 44.7 and 61.9 / 50.4, 24 of N 256 (75 MB) 40.8 / 41.8 at 44 and 53.9 / 44.3, 18 of N 512 (113 MB) 49.1 / 46.6, 54.4 /
// 47.8 and 72.2 / 51.3, 37 of N 256 (116 MB) 53.4 / 49.2, 57.3 / 50.7 and 67.6 / 53.4; K 5120, 14 of N 512 (110 MB) 43.3 / 45.4, 48.3 / 46.0 and
// 60.5 / 48.5; K 6144, 13 of N 512 (123 MB) 47.3 / 45.7, 52.5 / 46.8 and 67.2 / 48.9; K 16384, 37 of N 256 183 / 137, 188 / 143 and 209 / 149.
// With a shorter contraction or more weight tiles, at 34 and 62 rows: K 2048, 37 of N 256 35.9 / 40.4 and 47.8 / 44.3, 24 of N 512 36.1 / 38.2
// and 45.4 / 42.1, 8 of N 2048 33.8 / 42.9 and 44.2 / 47.6; K 4096, 8 of N 1024 33.1 / 40.1 and 48.4 / 44.2: these stream up to 64.
// One expert named by all of 180 tokens, 37 of K 4096, N 256: 72.2 / 54.0.
constexpr float kStreamBytes = 112e6f;
constexpr int64_t kStreamRows = 32;  // the fewest rows per expert up to which any call streams
static bool always_streams(const MoeArgs &a) { return (int64_t)a.M * a.top_k <= kStreamRows * a.E; }
static bool use_stream(const MoeArgs &a) {
    const int64_t tall_jobs = std::min<int64_t>(a.n_blocks, a.E) * (a.H / 128);
    const int n_wt = a.H / 128;
    const bool few_jobs = tall_jobs < resident_grid() / 2;
    int64_t rows = few_jobs ? 64 : kStreamRows;
    if (few_jobs && use_deep(a)) {
        const bool heavy = 3.f * (float)a.E * (float)a.N * (float)a.K >= kStreamBytes;
        rows = a.n_blocks * n_wt <= 32 ? kStreamRows : a.K >= 4096 && n_wt <= 2 ? (heavy ? 34 : 48) : 64;
    }
    return (int64_t)a.M * a.top_k <= rows * a.E;
}

static int launch_stream_pipeline(MoeArgs a, void *out, int split, hipStream_t s) {
    const int mask = phase_mask(), n_cus = resident_grid();
    const int n_wgs = 2 * n_cus;
    const int n_wt_up = a.H / 128, n_wt_down = (a.K + kWRows - 1) / kWRows;
    const int tall = a.n_blocks > 0 ? crowding_possible(a) : 0;
    a.crowd = tall;
    // units of 32 weight rows a job takes: two when that still leaves a job for every workgroup
    const int64_t blocks = std::min<int64_t>(a.n_blocks, std::min<int64_t>(a.E, (int64_t)a.M * a.top_k));
    auto launch = [&](auto one, auto two, int units) {
        const bool wide = blocks * units >= 2 * (int64_t)n_wgs && units % 2 == 0;
        const int n_tiles = wide ? units / 2 : units;
        const int grid = (int)std::min<int64_t>((int64_t)a.n_blocks * std::max(n_tiles, 1), n_wgs);
        if (grid > 0) hipLaunchKernelGGL(wide ? two : one, dim3(grid), dim3(512), 0, s, a, n_tiles);
    };
    if (mask & (PMOE_PHASE_UP | PMOE_PHASE_PROLOGUE)) {
        const int units = (mask & PMOE_PHASE_UP) ? a.H / 16 : 0;
        if (tall) launch(moe_stream_kernel<true, 1, true>, moe_stream_kernel<true, 2, true>, units);
        else launch(moe_stream_kernel<true, 1, false>, moe_stream_kernel<true, 2, false>, units);
    }
    if (tall) {
        MoeArgs t = a;
        hipLaunchKernelGGL(moe_prologue_kernel_bf16, dim3(1), dim3(kPrologueThreads), 0, s, t, n_wt_up, n_wt_down, n_cus, 0);
        t.n_wtiles = n_wt_up;
        if ((tall & 1) && (mask & PMOE_PHASE_UP)) hipLaunchKernelGGL(moe_up_kernel_bf16, dim3(n_cus), dim3(512), 0, s, t);
        t.n_wtiles = n_wt_down;
        if (mask & PMOE_PHASE_DOWN) hipLaunchKernelGGL(moe_down_kernel_bf16, dim3(n_cus), dim3(512), 0, s, t);
    }
    if ((mask & PMOE_PHASE_DOWN) && a.H <= 256 && a.n_blocks > 0) {
        const int grid = (int)std::min<int64_t>((int64_t)a.n_blocks * (a.K / 128), (a.H == 128 ? 4 : 2) * n_cus);
        if (a.H == 128) hipLaunchKernelGGL(moe_stream_down_short_kernel<256>, dim3(grid), dim3(256), 0, s, a);
        else hipLaunchKernelGGL(moe_stream_down_short_kernel<512>, dim3(grid), dim3(256), 0, s, a);
    } else if (mask & PMOE_PHASE_DOWN) {
        if (tall) launch(moe_stream_kernel<false, 1, true>, moe_stream_kernel<false, 2, true>, a.K / 32);
        else launch(moe_stream_kernel<false, 1, false>, moe_stream_kernel<false, 2, false>, a.K / 32);
    }
    if (mask & PMOE_PHASE_FINALIZE) launch_finalize(a, out, split, n_wt_down, s);
    return check_launch("fused_moe_bf16 launch");
}

size_t bf16_workspace(MoeArgs &a, char *ws) {
    const size_t H = (size_t)a.H;
    const size_t rows = align_up((size_t)a.sorted_num, kBlockRows);
    const size_t blocks = rows / kBlockRows;
    const size_t n_wt_up = H / 128;
    size_t off = 0;
    auto take = [&](size_t bytes) {
        const size_t at = off;
        off = align_up(off + bytes, 256);
        return ws != nullptr ? ws + at : nullptr;
    };
    a.plan = reinterpret_cast<TallPlan *>(take(sizeof(TallPlan)));
    // (run list and its order, used when they do not fit the LDS of the prologue)
    a.runs = reinterpret_cast<int4 *>(take((blocks + 1) * (sizeof(int4) + sizeof(int))));
    // (a cut has at most one tile per block: choose_tiles)
    a.tiles = reinterpret_cast<int4 *>(take((blocks + 1) * sizeof(int4)));
    a.tiles_down = reinterpret_cast<int4 *>(take((blocks + 1) * sizeof(int4)));
    // few up jobs for the chip and a contraction long enough to share (whether the chip has room is seen at the launch: the
    // size does not depend on the device), and not so few rows that the streaming kernels run whatever the device
    a.deep_ok = (blocks <= (size_t)kDeepBlocks && blocks * n_wt_up <= (size_t)kDeepJobs && a.K >= 2048 && !always_streams(a)) ? 1 : 0;
    a.up_partials = reinterpret_cast<float *>(
        take(a.deep_ok ? std::min<size_t>(kDeepParts * 4 * blocks * n_wt_up, kDeepSums) * 2048 * sizeof(float4) : 0));
    const size_t pairs = (size_t)a.M * (size_t)std::max(a.top_k, 1);
    a.inv = reinterpret_cast<int32_t *>(take(pairs * sizeof(int32_t)));
    a.y = take(pairs * a.K * 2);  // one row per pair id
    a.act = take(rows * H * 2);
    return off;
}

int launch_bf16_pipeline(MoeArgs a, void *out, int split, hipStream_t s) {
    const int mask = phase_mask();
    a.n_blocks = (a.sorted_num + kBlockRows - 1) / kBlockRows;
    if (use_few(a)) return launch_few_pipeline(a, out, split, s);
    if (use_stream(a)) return launch_stream_pipeline(a, out, split, s);
    const int n_wt_up = a.H / 128, n_wt_down = (a.K + kWRows - 1) / kWRows;
    const int n_cus = resident_grid();
    a.n_wtiles = n_wt_up;
    if (use_deep(a)) {
        // (the plan is part of the up kernel, and a launch of its own only where the down kernel runs without it)
        if (mask & (PMOE_PHASE_UP | PMOE_PHASE_DOWN | PMOE_PHASE_PROLOGUE))
            hipLaunchKernelGGL(moe_deep_up_kernel, dim3(n_cus), dim3(512), 0, s, a, n_wt_down, n_cus,
                               (mask & PMOE_PHASE_UP) ? 0 : 1);
        if (mask & PMOE_PHASE_UP) hipLaunchKernelGGL(moe_up_join_kernel, dim3(a.n_blocks * 4 * n_wt_up * 4), dim3(256), 0, s, a);
    } else {
        // the plan is needed by the two kernels even when the rest of the prologue is masked off
        const int do_invert = (mask & PMOE_PHASE_PROLOGUE) ? 1 : 0;
        const int blocks = do_invert ? std::max(1, std::min((a.sorted_num + kPrologueThreads - 1) / kPrologueThreads, 512)) : 1;
        hipLaunchKernelGGL(moe_prologue_kernel_bf16, dim3(blocks), dim3(kPrologueThreads), 0, s, a, n_wt_up, n_wt_down, n_cus,
                           do_invert);
        // resident kernels: a workgroup per CU (their 160 KB of LDS leave room for one)
        if (a.n_blocks > 0 && (mask & PMOE_PHASE_UP)) hipLaunchKernelGGL(moe_up_kernel_bf16, dim3(n_cus), dim3(512), 0, s, a);
    }
    if (a.n_blocks > 0) {
        MoeArgs d = a;
        d.n_wtiles = n_wt_down;
        if (mask & PMOE_PHASE_DOWN) hipLaunchKernelGGL(moe_down_kernel_bf16, dim3(n_cus), dim3(512), 0, s, d);
    }
    if (mask & PMOE_PHASE_FINALIZE) launch_finalize(a, out, split, n_wt_down, s);
    return check_launch("fused_moe_bf16 launch");
}

}  // namespace pmoe

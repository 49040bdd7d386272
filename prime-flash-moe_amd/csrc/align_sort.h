// Device side of the counting sort behind moe_align (moe_align.hip) and the router (route.hip): ids held in registers,
// ranked within their wave by ballots, then within the workgroup through a table of per-wave counts in LDS.
//
// What bounds these kernels is latency, so every id is loaded once, all loads of a thread in flight together (a loop
// that loads, ranks and loads again waits a memory latency per 64 ids of a wave: 11.5 us for 8192 ids, 417 us for
// 524288 in one workgroup), and ranked once.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pmoe {
namespace align {

constexpr int kMaxExperts = 1024;

// Ranks of a wave's ids: id[i] of lane l is number 64 i + l of the wave's run.  ord[i] = how many ids before it in
// the run name the same expert; counts[e] (LDS, the wave's own row) grows by the run's count of e.  Lanes that hold
// the same expert find each other with one ballot per id bit.  Ids outside [0, E) are skipped.
template <int PER>
__device__ __forceinline__ void rank_ids(const int (&id)[PER], int (&ord)[PER], int32_t *counts, int E, int id_bits, int lane) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = id[i];
        const bool valid = (unsigned)e < (unsigned)E;
        unsigned long long peers = __ballot(valid);
        for (int b = 0; b < id_bits; ++b) {
            const bool bit = (e >> b) & 1;
            const unsigned long long set = __ballot(bit);
            peers &= bit ? set : ~set;
        }
        ord[i] = 0;
        if (valid) {
            const int rank = __popcll(peers & ((1ull << lane) - 1ull)), cnt = __popcll(peers);
            const int before = counts[e];
            ord[i] = before + rank;
            if (rank == cnt - 1) counts[e] = before + cnt;  // one writer per expert, after all reads
        }
    }
}

// Loads a workgroup's run of NW * 64 * PER ids starting at `base`; entries at or past `end` become -1.
template <int NW, int PER>
__device__ __forceinline__ void load_ids(int (&id)[PER], const int32_t *ids, int64_t base, int64_t end) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int64_t at = base + (int64_t)(wave * PER + i) * 64 + lane;
        id[i] = at < end ? ids[at] : -1;
    }
}

// Exclusive prefix of padc[0 .. E) into offs[0 .. E], by wave 0: serial inside a lane's chunk, shuffle scan across.
__device__ __forceinline__ void scan_experts(const int32_t *padc, int32_t *offs, int E) {
    if (threadIdx.x >= 64) return;
    const int lane = threadIdx.x, chunk = (E + 63) >> 6, b = lane * chunk;
    int local = 0;
    for (int j = 0; j < chunk; ++j)
        if (b + j < E) local += padc[b + j];
    int incl = local;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int v = __shfl_up(incl, d, 64);
        if (lane >= d) incl += v;
    }
    int run = incl - local;
    for (int j = 0; j < chunk; ++j)
        if (b + j < E) {
            offs[b + j] = run;
            run += padc[b + j];
        }
    if (lane == 63) offs[E] = incl;  // lane 63's inclusive sum is the grand total
}

// Expert whose padded range holds `row` (the last one that starts at or before it); E - 1 past the total.
__device__ __forceinline__ int owner_of(const int32_t *offs, int E, int row) {
    if (row >= offs[E]) return E - 1;
    int lo = 0, hi = E - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (offs[mid] <= row) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

struct Outputs {
    int32_t *sorted_token_ids, *expert_ids, *num_tokens_post_padded;
    int block_m, pad_to, max_padded, max_blocks;
};

// Thread `me` of `n_threads` that fill `count` words.
__device__ __forceinline__ void fill_minus_one(int32_t *out, int count, int me, int n_threads) {
    if ((reinterpret_cast<uintptr_t>(out) & 15) == 0) {
        int4 *dst = reinterpret_cast<int4 *>(out);
        for (int i = me; i < count / 4; i += n_threads) dst[i] = make_int4(-1, -1, -1, -1);
        for (int64_t i = (count & ~3) + (int64_t)me; i < count; i += n_threads) out[i] = -1;
    } else {
        for (int64_t i = me; i < count; i += n_threads) out[i] = -1;
    }
}

__device__ __forceinline__ void write_expert_ids(const Outputs &o, const int32_t *offs, int E, int n_threads) {
    for (int64_t j = threadIdx.x; j < o.max_blocks; j += n_threads) o.expert_ids[j] = owner_of(offs, E, (int)j * o.block_m);
}

// LDS words of sort_in_workgroup.
__host__ __device__ constexpr int sort_words(int n_waves, int E) { return 2 * E + 1 + n_waves * E; }

// The whole sort by one workgroup of NW waves whose ids are in registers (load_ids from 0; n <= NW * 64 * PER), in two steps
// with a barrier between them.  What does not need the ids, by thread `me` of `n_threads`:
template <int NW>
__device__ __forceinline__ void begin_sort(const Outputs &o, int E, int32_t *smem, int me, int n_threads) {
    fill_minus_one(o.sorted_token_ids, o.max_padded, me, n_threads);  // complete before any pair id lands on top of it: barriers follow
    for (int i = me; i < NW * E; i += n_threads) smem[2 * E + 1 + i] = 0;
}
template <int NW, int PER>
__device__ __forceinline__ void finish_sort(const int (&id)[PER], const Outputs &o, int E, int id_bits, int32_t *smem) {
    constexpr int NT = NW * 64;
    int32_t *offs = smem, *padc = smem + E + 1, *table = smem + 2 * E + 1;  // table: [NW][E] counts, then bases
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int ord[PER];
    rank_ids<PER>(id, ord, table + wave * E, E, id_bits, lane);
    __syncthreads();
    for (int e = tid; e < E; e += NT) {
        int run = 0;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const int c = table[w * E + e];
            table[w * E + e] = run;
            run += c;
        }
        padc[e] = (run + o.pad_to - 1) / o.pad_to * o.pad_to;
    }
    __syncthreads();
    scan_experts(padc, offs, E);
    __syncthreads();
    if (tid == 0) o.num_tokens_post_padded[0] = offs[E];
    write_expert_ids(o, offs, E, NT);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = id[i];
        if ((unsigned)e < (unsigned)E)
            o.sorted_token_ids[offs[e] + table[wave * E + e] + ord[i]] = (wave * PER + i) * 64 + lane;
    }
}
template <int NW, int PER>
__device__ __forceinline__ void sort_in_workgroup(const int (&id)[PER], const Outputs &o, int E, int id_bits, int32_t *smem) {
    begin_sort<NW>(o, E, smem, threadIdx.x, NW * 64);
    __syncthreads();
    finish_sort<NW, PER>(id, o, E, id_bits, smem);
}

inline int id_bits_for(int num_experts) {
    int id_bits = 1;
    while ((1 << id_bits) < num_experts) ++id_bits;
    return id_bits;
}

}  // namespace align
}  // namespace pmoe

// moe_align for gfx950: stable counting sort of pair ids by expert, padded per expert.
//
// Semantics follow the reference kernel (prime_moe/csrc/kernels/fused_moe_bf16_kernel.cu:853-907)
// except that the within-expert order is made unique (ascending pair id) instead of being
// left to an atomic race.  Up to kFewIds ids, or any number without scratch memory, one workgroup does it (align_sort.h):
// ranks inside the waves, per-expert counts of the waves -> bases, padded totals -> prefix, scatter.  More ids spread over
// workgroups if the caller gives scratch (pmoe_moe_align_static, which has its own, does so above kSingleMaxIds).
// Ids, positions and sizes are int32 (loops that step past a size near 2^31 count in int64), and the output is a pure function of the input.
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "align_sort.h"
#include "pmoe_common.h"

namespace pmoe {
using align::kMaxExperts;

int moe_align_validate(const int32_t *topk_ids, const int32_t *sorted_token_ids, const int32_t *expert_ids,
             const int32_t *num_tokens_post_padded, int n, int num_experts, int block_m, int pad_to, int max_padded,
             int max_blocks) {
    PMOE_REQUIRE(num_experts > 0 && block_m > 0 && pad_to > 0, "moe_align: block_m, bpc and num_experts must be positive");
    PMOE_REQUIRE(num_experts <= kMaxExperts, "moe_align supports at most 1024 experts, got %d", num_experts);
    PMOE_REQUIRE(n >= 0 && max_padded >= 0 && max_blocks >= 0, "moe_align: negative size");
    PMOE_REQUIRE(pad_to % block_m == 0, "moe_align: pad_to must be a multiple of block_m");
    const long long need = ((long long)n + (long long)num_experts * (pad_to - 1) + pad_to - 1) / pad_to * pad_to;
    PMOE_REQUIRE(max_padded >= need, "moe_align: max_padded %d is smaller than the worst case %lld", max_padded, need);
    PMOE_REQUIRE((long long)max_blocks * block_m <= (long long)max_padded + block_m - 1,
                 "moe_align: max_blocks %d does not match max_padded %d", max_blocks, max_padded);
    PMOE_REQUIRE(sorted_token_ids && expert_ids && num_tokens_post_padded && (topk_ids || n == 0), "moe_align: null pointer");
    return PMOE_OK;
}

}  // namespace pmoe

namespace {

using namespace pmoe::align;

// One workgroup, n <= NW * 64 * PER (8192 ids of 8 experts: 11.5 -> 6 us against loading and ranking 64 ids at a time).
template <int NW, int PER>
__global__ __launch_bounds__(NW * 64) void moe_align_kernel(const int32_t *__restrict__ topk_ids, Outputs o, int n, int E,
                                                            int id_bits) {
    extern __shared__ int32_t smem[];
    int id[PER];
    load_ids<NW, PER>(id, topk_ids, 0, n);
    sort_in_workgroup<NW, PER>(id, o, E, id_bits, smem);
}

// ---- many ids: the same sort spread over workgroups, two launches (three for very many).
//   count:   workgroup g counts ids [g S, (g + 1) S) per expert -> counts[g][e]
//   scatter: every workgroup sums counts[.][e] itself (all slices: totals and the padded prefix; the slices before
//            its own: its bases), ranks its slice as above and writes pair id i to offs[e] + base + rank; it also
//            writes its share of the padding slots (those at or behind an expert's count, and past the total) and of
//            expert_ids.  No slot is written twice and no order between workgroups is needed.
// Slices are contiguous and ascending in g, waves inside a slice likewise: the order inside an expert is
// ascending pair id, bit for bit what the single workgroup produces.
// That reading of all counts by every workgroup grows with the square of the number of slices: above kSelfScanWords
// a kernel between the two turns counts[.][e] into bases and totals (align_bases_kernel).
// Ranking is what a slice costs (ballots, a few hundred instructions per 64 ids of a wave), so slices are as small as
// the scratch allows, from 1024 ids on, up to 64 of them: 65536 ids of 128 experts take 20 us in 8 slices.
constexpr int kMinSliceIds = 1024, kMaxSliceIds = 8192;
constexpr int kFewIds = 8192;         // up to here one workgroup is as fast (8192 ids: 8.7 us; 16384: 19.6)
constexpr int kSingleMaxIds = 16384;  // up to here the small scratch of pmoe_moe_align_workspace_bytes is nothing

int slice_ids(int n) {
    int s = kMinSliceIds;
    while (s < kMaxSliceIds && (int64_t)s * 64 < n) s *= 2;
    return s;
}
int n_slices(int n, int slice) { return (int)(((int64_t)n + slice - 1) / slice); }

template <int NW, int PER>
__global__ __launch_bounds__(NW * 64) void align_count_kernel(const int32_t *__restrict__ topk_ids, int n, int E, int id_bits,
                                                              int32_t *__restrict__ counts) {
    extern __shared__ int32_t smem[];  // [NW][E]
    constexpr int NT = NW * 64;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = blockIdx.x;
    int id[PER], ord[PER];
    load_ids<NW, PER>(id, topk_ids, (int64_t)g * NT * PER, n);
    for (int i = tid; i < NW * E; i += NT) smem[i] = 0;
    __syncthreads();
    rank_ids<PER>(id, ord, smem + wave * E, E, id_bits, lane);
    __syncthreads();
    for (int e = tid; e < E; e += NT) {
        int c = 0;
#pragma unroll
        for (int w = 0; w < NW; ++w) c += smem[w * E + e];
        counts[(size_t)g * E + e] = c;
    }
}

// counts[g][e] -> ids of e in the slices before g, for 1 << bits experts per workgroup; their totals -> totals[e].  A
// thread sums a run of slices, the runs before it come from LDS, and a second pass over its run writes the bases.
__global__ __launch_bounds__(1024) void align_bases_kernel(int32_t *counts, int32_t *totals, int G, int E, int bits) {
    __shared__ int32_t sums[1024];
    constexpr int kBatch = 16;  // loads in flight
    const int tid = threadIdx.x, cols = 1 << bits, parts = 1024 >> bits, col = tid & (cols - 1), part = tid >> bits;
    const int e = blockIdx.x * cols + col, per = (G + parts - 1) / parts, end = min((part + 1) * per, G);
    int sum = 0;
    if (e < E) {
#pragma unroll 16
        for (int s = part * per; s < end; ++s) sum += counts[(size_t)s * E + e];
    }
    sums[tid] = sum;
    __syncthreads();
    int run = 0, all = 0;
    for (int p = 0; p < parts; ++p) {
        const int v = sums[p * cols + col];
        run += p < part ? v : 0;
        all += v;
    }
    if (e >= E) return;
    if (part == 0) totals[e] = all;
    for (int s = part * per; s < end; s += kBatch) {
        int c[kBatch];
#pragma unroll
        for (int i = 0; i < kBatch; ++i) c[i] = s + i < end ? counts[(size_t)(s + i) * E + e] : 0;
#pragma unroll
        for (int i = 0; i < kBatch; ++i) {
            if (s + i < end) counts[(size_t)(s + i) * E + e] = run;
            run += c[i];
        }
    }
}

// `totals`: counts holds the bases already (align_bases_kernel); null: it holds the counts.
template <int NW, int PER>
__global__ __launch_bounds__(NW * 64) void align_scatter_kernel(const int32_t *__restrict__ topk_ids, const int32_t *__restrict__ counts,
                                                                const int32_t *__restrict__ totals, Outputs o, int n, int E, int id_bits) {
    extern __shared__ int32_t smem[];
    constexpr int NT = NW * 64;
    int32_t *offs = smem, *padc = smem + E + 1, *table = smem + 2 * E + 1;  // table: [NW][E]
    int32_t *tot = table + NW * E, *before = tot + E;                       // all ids of e; those in earlier slices
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = blockIdx.x, G = gridDim.x;
    int id[PER], ord[PER];
    load_ids<NW, PER>(id, topk_ids, (int64_t)g * NT * PER, n);
    for (int i = tid; i < (NW + 2) * E; i += NT) table[i] = 0;
    __syncthreads();
    if (totals != nullptr) {
        for (int e = tid; e < E; e += NT) {
            tot[e] = totals[e];
            before[e] = counts[(size_t)g * E + e];
        }
    } else {
        // thread (part, e) sums every parts-th slice
        const int bits = 32 - __builtin_clz(max(E - 1, 1)), pitch = 1 << bits, parts = max(1, NT >> bits);
        for (int i = tid; i < pitch * parts; i += NT) {
            const int e = i & (pitch - 1), part = i >> bits;
            if (e >= E) continue;
            int all = 0, mine = 0;
#pragma unroll 8
            for (int s = part; s < G; s += parts) {
                const int c = counts[(size_t)s * E + e];
                all += c;
                mine += s < g ? c : 0;
            }
            atomicAdd(tot + e, all);
            atomicAdd(before + e, mine);
        }
    }
    rank_ids<PER>(id, ord, table + wave * E, E, id_bits, lane);
    __syncthreads();
    for (int e = tid; e < E; e += NT) {
        int run = before[e];
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const int c = table[w * E + e];
            table[w * E + e] = run;
            run += c;
        }
        padc[e] = (tot[e] + o.pad_to - 1) / o.pad_to * o.pad_to;
    }
    __syncthreads();
    scan_experts(padc, offs, E);
    __syncthreads();
    const int total = offs[E];
    if (g == 0 && tid == 0) o.num_tokens_post_padded[0] = total;
    for (int64_t j = g * NT + tid; j < o.max_blocks; j += G * NT) o.expert_ids[j] = owner_of(offs, E, (int)j * o.block_m);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = id[i];
        if ((unsigned)e < (unsigned)E)
            o.sorted_token_ids[offs[e] + table[wave * E + e] + ord[i]] = (g * NW * PER + wave * PER + i) * 64 + lane;
    }
    // padding: an expert's by one wave, the slots past the total by everybody
    for (int e = g * NW + wave; e < E; e += G * NW)
        for (int64_t pos = (int64_t)offs[e] + tot[e] + lane; pos < offs[e + 1]; pos += 64) o.sorted_token_ids[pos] = -1;
    for (int64_t pos = (int64_t)total + g * NT + tid; pos < o.max_padded; pos += (int64_t)G * NT) o.sorted_token_ids[pos] = -1;
}

// Any number of ids by one workgroup, for callers without scratch memory: a pass that counts, then the sort run by
// run with the experts' bases carried on.
template <int NW>
__global__ __launch_bounds__(NW * 64) void align_runs_kernel(const int32_t *__restrict__ topk_ids, Outputs o, int n, int E, int id_bits) {
    extern __shared__ int32_t smem[];
    constexpr int NT = NW * 64, PER = 16, RUN = NT * PER;
    int32_t *offs = smem, *padc = smem + E + 1, *table = smem + 2 * E + 1, *base = table + NW * E;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    fill_minus_one(o.sorted_token_ids, o.max_padded, tid, NT);
    for (int i = tid; i < (NW + 1) * E; i += NT) table[i] = 0;
    __syncthreads();
    int id[PER], ord[PER];
    for (int64_t r = 0; r < n; r += RUN) {
        load_ids<NW, PER>(id, topk_ids, r, n);
        rank_ids<PER>(id, ord, table + wave * E, E, id_bits, lane);
    }
    __syncthreads();
    for (int e = tid; e < E; e += NT) {
        int c = 0;
        for (int w = 0; w < NW; ++w) c += table[w * E + e];
        padc[e] = (c + o.pad_to - 1) / o.pad_to * o.pad_to;
    }
    __syncthreads();
    scan_experts(padc, offs, E);
    __syncthreads();
    if (tid == 0) o.num_tokens_post_padded[0] = offs[E];
    write_expert_ids(o, offs, E, NT);
    for (int64_t r = 0; r < n; r += RUN) {
        load_ids<NW, PER>(id, topk_ids, r, n);
        for (int i = tid; i < NW * E; i += NT) table[i] = 0;
        __syncthreads();
        rank_ids<PER>(id, ord, table + wave * E, E, id_bits, lane);
        __syncthreads();
        for (int e = tid; e < E; e += NT) {
            int run = base[e];
            for (int w = 0; w < NW; ++w) {
                const int c = table[w * E + e];
                table[w * E + e] = run;
                run += c;
            }
            base[e] = run;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = id[i];
            if ((unsigned)e < (unsigned)E)
                o.sorted_token_ids[offs[e] + table[wave * E + e] + ord[i]] = (int)r + (wave * PER + i) * 64 + lane;
        }
        __syncthreads();
    }
}

// Scratch of the entry point that allocates nothing (pmoe_moe_align_static): what the first query asks for, that is
// 2 E + 1 words more than the counts[G][E] in use, for the multi-workgroup sort of up to kStaticMaxIds ids and kMaxExperts
// experts: 520 KB held by every device the library runs on until the process ends.  In host code this name is only a
// handle for hipGetSymbolAddress; kernels get the address that call returns.
constexpr int kStaticMaxIds = PMOE_ALIGN_STATIC_MAX_IDS;
constexpr size_t kStaticWords = (size_t)(kStaticMaxIds / kMaxSliceIds) * kMaxExperts + 2 * kMaxExperts + 1;
static __device__ __align__(256) int32_t scratch[kStaticWords];

// One workgroup sorts everything.  (16 waves; 8 above 512 experts, whose tables would not fit the LDS otherwise.)
int launch_single(const int32_t *topk_ids, const Outputs &o, int n, int E, hipStream_t s) {
    const int id_bits = id_bits_for(E);
    auto launch = [&](auto nw) {
        constexpr int NW = decltype(nw)::value;
        const size_t smem = sizeof(int32_t) * (size_t)sort_words(NW, E);
        const int per = (n + NW * 64 - 1) / (NW * 64);
        auto go = [&](auto kernel, size_t bytes) { hipLaunchKernelGGL(kernel, dim3(1), dim3(NW * 64), bytes, s, topk_ids, o, n, E, id_bits); };
        if (per <= 1) go(moe_align_kernel<NW, 1>, smem);
        else if (per <= 2) go(moe_align_kernel<NW, 2>, smem);
        else if (per <= 4) go(moe_align_kernel<NW, 4>, smem);
        else if (per <= 8) go(moe_align_kernel<NW, 8>, smem);
        else if (per <= 16) go(moe_align_kernel<NW, 16>, smem);
        else go(align_runs_kernel<NW>, smem + sizeof(int32_t) * E);
    };
    if (E <= 512) launch(std::integral_constant<int, 16>{});
    else launch(std::integral_constant<int, 8>{});
    return pmoe::check_launch("moe_align launch");
}

// The launches of the multi-workgroup sort in slices of `slice` ids; `words` holds n_slices * E int32 of device
// scratch, or E more (n_words), every one of which is written before it is read.
// What the scatter kernel reads if it adds up the counts itself, in words of all its workgroups, against one launch more:
// equal at 1 << 20 ids of 1024 experts (48 us, 16.8 M words) and 1 << 21 of 128 (27 / 29 us, 8.4 M); 21 / 28 us at 1 << 22 of 8
// (2.1 M), 140 / 72 at 1 << 22 of 1024 (268 M), 247 / 139 at 1 << 24 of 128, 1144 / 219 at 1 << 24 of 1024, 15097 / 731 at 1 << 26.
constexpr int64_t kSelfScanWords = 1 << 24;
int launch_multi(const int32_t *topk_ids, const Outputs &o, int n, int E, int slice, int32_t *words, size_t n_words, hipStream_t s) {
    const int id_bits = id_bits_for(E);
    const int G = n_slices(n, slice);
    int32_t *totals = (int64_t)G * G * E > kSelfScanWords && n_words >= (size_t)(G + 1) * E ? words + (size_t)G * E : nullptr;
    auto launch = [&](auto nw, auto p) {
        constexpr int NW = decltype(nw)::value, PER = decltype(p)::value;
        hipLaunchKernelGGL((align_count_kernel<NW, PER>), dim3(G), dim3(NW * 64), sizeof(int32_t) * (size_t)NW * E, s, topk_ids, n, E,
                           id_bits, words);
        const int bits = std::min(id_bits, 6);
        if (totals != nullptr)
            hipLaunchKernelGGL(align_bases_kernel, dim3((E + (1 << bits) - 1) >> bits), dim3(1024), 0, s, words, totals, G, E, bits);
        hipLaunchKernelGGL((align_scatter_kernel<NW, PER>), dim3(G), dim3(NW * 64), sizeof(int32_t) * (size_t)(sort_words(NW, E) + 2 * E), s,
                           topk_ids, words, totals, o, n, E, id_bits);
    };
    auto with_per = [&](auto nw) {
        constexpr int NW = decltype(nw)::value;
        if (slice <= 1024) launch(nw, std::integral_constant<int, 1024 / (NW * 64)>{});
        else if (slice <= 2048) launch(nw, std::integral_constant<int, 2048 / (NW * 64)>{});
        else if (slice <= 4096) launch(nw, std::integral_constant<int, 4096 / (NW * 64)>{});
        else launch(nw, std::integral_constant<int, 8192 / (NW * 64)>{});
    };
    if (E <= 512) with_per(std::integral_constant<int, 16>{});
    else with_per(std::integral_constant<int, 8>{});
    return pmoe::check_launch("moe_align launch");
}

// Device address of `scratch` on the current device: every device holds its own copy of the array at
// its own address, looked up once per device (with that device current) and kept.  `data` is one of the
// call's device pointers: the current device must be the one that holds it (the kernels run where the data
// is, and another device's copy of the array has another address), otherwise the call is rejected.
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
int32_t *g_scratch_ptr[kMaxDevices] = {nullptr};

int static_scratch(const void *data, int32_t **out) {
    int dev = 0;
    hipError_t err = hipGetDevice(&dev);
    if (err != hipSuccess) return pmoe::fail(PMOE_ERR_HIP, "moe_align_static: hipGetDevice: %s", hipGetErrorString(err));
    PMOE_REQUIRE(dev >= 0 && dev < kMaxDevices, "moe_align_static: device index %d out of range", dev);
    hipPointerAttribute_t attr;
    if (hipPointerGetAttributes(&attr, data) == hipSuccess)
        PMOE_REQUIRE(attr.device == dev, "moe_align_static: the data lives on device %d but device %d is current", attr.device, dev);
    else
        (void)hipGetLastError();  // (a pointer the runtime does not know: nothing to compare)
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[dev] == nullptr) {
        void *p = nullptr;
        err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (err != hipSuccess || p == nullptr)
            return pmoe::fail(PMOE_ERR_HIP, "moe_align_static: hipGetSymbolAddress: %s", hipGetErrorString(err));
        g_scratch_ptr[dev] = static_cast<int32_t *>(p);
    }
    *out = g_scratch_ptr[dev];
    return PMOE_OK;
}

}  // namespace

extern "C" size_t pmoe_moe_align_workspace_bytes(int n, int num_experts) {
    if (n <= kSingleMaxIds || num_experts <= 0 || num_experts > kMaxExperts) return 0;
    const size_t G = (size_t)n_slices(n, kMaxSliceIds);  // counts, totals; E + 1 words more than are used, as callers know it
    return sizeof(int32_t) * (G * (size_t)num_experts + 2 * (size_t)num_experts + 1);
}

extern "C" size_t pmoe_moe_align_workspace_bytes_fast(int n, int num_experts) {
    if (n <= kFewIds || num_experts <= 0 || num_experts > kMaxExperts) return 0;
    return std::max(sizeof(int32_t) * (size_t)n_slices(n, slice_ids(n)) * (size_t)num_experts,
                    pmoe_moe_align_workspace_bytes(n, num_experts));
}

extern "C" int pmoe_moe_align(const int32_t *topk_ids, int32_t *sorted_token_ids,
                              int32_t *expert_ids, int32_t *num_tokens_post_padded, int n,
                              int num_experts, int block_m, int pad_to, int max_padded,
                              int max_blocks, void *stream) {
    return pmoe_moe_align_ws(topk_ids, sorted_token_ids, expert_ids, num_tokens_post_padded, n, num_experts, block_m,
                             pad_to, max_padded, max_blocks, nullptr, 0, stream);
}

extern "C" int pmoe_moe_align_ws(const int32_t *topk_ids, int32_t *sorted_token_ids, int32_t *expert_ids,
                                 int32_t *num_tokens_post_padded, int n, int num_experts, int block_m, int pad_to,
                                 int max_padded, int max_blocks, void *workspace, size_t workspace_bytes,
                                 void *stream) {
    if (int rc = pmoe::moe_align_validate(topk_ids, sorted_token_ids, expert_ids, num_tokens_post_padded, n, num_experts, block_m,
                          pad_to, max_padded, max_blocks))
        return rc;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const Outputs o{sorted_token_ids, expert_ids, num_tokens_post_padded, block_m, pad_to, max_padded, max_blocks};
    if (n > kFewIds && workspace != nullptr) {
        // A misaligned pointer is an error only where the call cannot do without the scratch it was given for; where the
        // first query asks for none, or for more than this, it is not looked at.
        const bool aligned = (reinterpret_cast<uintptr_t>(workspace) & 3) == 0;
        PMOE_REQUIRE(aligned || n <= kSingleMaxIds || workspace_bytes < pmoe_moe_align_workspace_bytes(n, num_experts),
                     "moe_align: workspace must be 4-byte aligned");
        // the finest slices whose counts fit the scratch
        for (int slice = slice_ids(n); aligned && slice <= kMaxSliceIds; slice *= 2)
            if (sizeof(int32_t) * (size_t)n_slices(n, slice) * num_experts <= workspace_bytes)
                return launch_multi(topk_ids, o, n, num_experts, slice, static_cast<int32_t *>(workspace), workspace_bytes / sizeof(int32_t), s);
    }
    return launch_single(topk_ids, o, n, num_experts, s);
}

extern "C" int pmoe_moe_align_static(const int32_t *topk_ids, int32_t *sorted_token_ids, int32_t *expert_ids,
                                     int32_t *num_tokens_post_padded, int n, int num_experts, int block_m,
                                     int pad_to, int max_padded, int max_blocks, void *stream) {
    if (int rc = pmoe::moe_align_validate(topk_ids, sorted_token_ids, expert_ids, num_tokens_post_padded, n, num_experts, block_m,
                          pad_to, max_padded, max_blocks))
        return rc;
    PMOE_REQUIRE(n <= kStaticMaxIds, "moe_align_static: at most %d ids fit the built-in scratch, got %d", kStaticMaxIds, n);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const Outputs o{sorted_token_ids, expert_ids, num_tokens_post_padded, block_m, pad_to, max_padded, max_blocks};
    if (n <= kSingleMaxIds)  // one workgroup sorts these in its LDS: no device scratch involved
        return launch_single(topk_ids, o, n, num_experts, s);
    int32_t *words = nullptr;
    if (int rc = static_scratch(topk_ids, &words)) return rc;
    // the finest slices whose counts fit the array
    int slice = slice_ids(n);
    while (slice < kMaxSliceIds && (size_t)n_slices(n, slice) * num_experts > kStaticWords) slice *= 2;
    return launch_multi(topk_ids, o, n, num_experts, slice, words, kStaticWords, s);
}

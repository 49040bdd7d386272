// Router front-end for gfx950: gate logits -> top-k expert ids + softmax weights, followed by moe_align.
//
// The reference leaves routing to the caller ("routing comes from your gate", README.md:147-149; its
// benchmark draws ids directly, benchmark/benchmark.py:124-166) and starts at moe_align.  This is the
// step in front of it, on the same stream, without a host synchronisation:
//   topk_ids[t, r]     = index of the r-th largest of logits[t, :] (+ bias), ties to the lower index,
//                        NaN above every number (the order torch.topk documents);
//   topk_weights[t, :] = softmax over the top_k selected values, fp32
//   then the moe_align sort of the T * top_k ids (same kernels, same bits as pmoe_moe_align_ws).
//
// One wave per token.  Lane l holds experts l, l + 64, l + 128, ... (EPL of them) as order-preserving 32-bit keys.
// A round takes the largest key (a maximum over the lane's keys, then over the wave by DPP moves: register to
// register, where shuffles through LDS cost ten times the latency), finds the lowest expert that holds it with a ballot
// per key register, and retires it.  The softmax of the top_k winners is computed by the lanes that keep them.
//
// Few tokens (one workgroup's work, see fits_small): top-k and sort in one kernel, the ids handed over in LDS
// (align_sort.h).
#include <algorithm>
#include <type_traits>

#include "align_sort.h"
#include "pmoe_common.h"

namespace pmoe {
// Argument checks of moe_align (moe_align.hip).
int moe_align_validate(const int32_t *topk_ids, const int32_t *sorted_token_ids, const int32_t *expert_ids,
                       const int32_t *num_tokens_post_padded, int n, int num_experts, int block_m, int pad_to, int max_padded,
                       int max_blocks);
}  // namespace pmoe

namespace {

constexpr int kMaxTopK = 32;

__device__ __forceinline__ float load_logit(const float *p, int64_t i) { return p[i]; }
__device__ __forceinline__ float load_logit(const uint16_t *p, int64_t i) { return __uint_as_float((uint32_t)p[i] << 16); }

// Monotone map float -> uint32 (a < b <=> key(a) < key(b)); -0 counts as +0, NaN lands above +inf.
__device__ __forceinline__ uint32_t order_key(float v) {
    v += 0.0f;  // -0 -> +0
    uint32_t u = __float_as_uint(v);
    if (v != v) u = 0x7fffffffu;  // every NaN: the largest positive pattern
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float key_value(uint32_t k) {
    const uint32_t u = (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k;
    return __uint_as_float(u);
}

// Maximum over the wave, in every lane.  Row shifts by 1, 2, 4, 8 and the two row broadcasts leave it in lane 63.
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
#define PMOE_DPP_MAX(ctrl, rows) v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, rows, 0xf, false))
    PMOE_DPP_MAX(0x111, 0xf);  // row_shr:1
    PMOE_DPP_MAX(0x112, 0xf);  // row_shr:2
    PMOE_DPP_MAX(0x114, 0xf);  // row_shr:4
    PMOE_DPP_MAX(0x118, 0xf);  // row_shr:8
    PMOE_DPP_MAX(0x142, 0xa);  // row_bcast:15
    PMOE_DPP_MAX(0x143, 0xc);  // row_bcast:31
#undef PMOE_DPP_MAX
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// Top-k and softmax of token t; lane r < top_k returns winner r (id, weight).
template <int EPL, typename T>
__device__ __forceinline__ void topk_of_token(const T *__restrict__ logits, const float *__restrict__ bias, int64_t t, int E, int top_k,
                                              int lane, int &my_id, float &my_weight) {
    uint32_t key[EPL];
#pragma unroll
    for (int j = 0; j < EPL; ++j) {
        const int e = lane + 64 * j;
        key[j] = 0u;  // below every real key: never selected before a real element
        if (e < E) {
            float v = load_logit(logits, t * E + e);
            if (bias != nullptr) v += bias[e];
            key[j] = order_key(v);
        }
    }
    float my_val = 0.f;  // lane r keeps the value of winner r
    my_id = 0;
    for (int r = 0; r < top_k; ++r) {
        uint32_t best = key[0];
#pragma unroll
        for (int j = 1; j < EPL; ++j) best = max(best, key[j]);
        best = wave_max(best);
        int win = -1;
#pragma unroll
        for (int j = EPL - 1; j >= 0; --j) {
            const uint64_t m = __ballot(key[j] == best);
            if (m != 0) win = 64 * j + __builtin_ctzll(m);
        }
#pragma unroll
        for (int j = 0; j < EPL; ++j)
            if (lane + 64 * j == win) key[j] = 0u;
        if (lane == r) {
            my_val = key_value(best);
            my_id = win;
        }
    }
    // softmax over the winners: lanes 0 .. top_k - 1 hold them, winner 0 is the maximum
    const float vmax = __shfl(my_val, 0, 64);
    const float ex = lane < top_k ? expf(my_val - vmax) : 0.f;
    float sum = ex;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) sum += __shfl_xor(sum, d, 64);
    my_weight = ex / sum;
}

template <int EPL, typename T>
__global__ __launch_bounds__(256) void route_topk_kernel(const T *__restrict__ logits, const float *__restrict__ bias,
                                                         int32_t *__restrict__ topk_ids,
                                                         float *__restrict__ topk_weights, int n_tokens, int E,
                                                         int top_k) {
    const int lane = threadIdx.x & 63;
    const int64_t t = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6;
    if (t >= n_tokens) return;
    int id;
    float w;
    topk_of_token<EPL, T>(logits, bias, t, E, top_k, lane, id, w);
    if (lane < top_k) {
        topk_ids[t * top_k + lane] = id;
        topk_weights[t * top_k + lane] = w;
    }
}

// Top-k of all tokens (wave w: tokens w, w + NW, ...) and the sort of their ids: n_tokens * top_k <= NW * 64.  Workgroup 0 does
// that for the rows that the pairs can reach (`reach`, a multiple of block_m or max_padded: every pair in an expert of its own);
// the others write what is known of the rest, -1 and the last expert.  (A token of 128 experts has room for 16264 rows and
// reaches 1024, five of 256 experts 32552 and 5120; one CU takes 0.5 and 1 us to fill them.)  Workgroup 0 fills its rows with the waves that
// have no token, beside the top-k, or with all of them behind it: stores in front of its logits are waited for with them.  The whole
// kernel, all rows by one workgroup behind the top-k / as it is, us: one token, top 1 of 3 3.7 / 3.6, top 8 of 64, 128, 256 and 512 5.0 / 4.7, 6.0 /
// 5.4, 7.6 / 6.4 and 10.5 / 8.3; 16 tokens, top 1 of 3 4.0 / 4.0, top 8 of 64, 256 and 512 5.7 / 5.7, 8.6 / 7.8 and 12.2 / 10.7.
template <int NW, int EPL, typename T>
__global__ __launch_bounds__(NW * 64) void route_small_kernel(const T *__restrict__ logits, const float *__restrict__ bias,
                                                              int32_t *__restrict__ topk_ids, float *__restrict__ topk_weights,
                                                              pmoe::align::Outputs o, int reach, int reach_blocks, int n_tokens, int E, int top_k, int id_bits) {
    extern __shared__ int32_t smem[];
    __shared__ int32_t ids[NW * 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (blockIdx.x > 0) {
        const int n = (int)(gridDim.x - 1) * NW * 64, me = (int)(blockIdx.x - 1) * NW * 64 + tid;
        pmoe::align::fill_minus_one(o.sorted_token_ids + reach, o.max_padded - reach, me, n);
        for (int64_t j = reach_blocks + (int64_t)me; j < o.max_blocks; j += n) o.expert_ids[j] = E - 1;
        return;
    }
    o.max_padded = reach;
    o.max_blocks = reach_blocks;
    const int busy = n_tokens <= NW - 2 ? n_tokens : 0;  // (one wave alone would be the last to arrive)
    if (busy > 0 && wave >= busy) pmoe::align::begin_sort<NW>(o, E, smem, tid - 64 * busy, 64 * (NW - busy));
    for (int t = wave; t < n_tokens; t += NW) {
        int id;
        float w;
        topk_of_token<EPL, T>(logits, bias, t, E, top_k, lane, id, w);
        if (lane < top_k) {
            ids[t * top_k + lane] = id;
            topk_ids[t * top_k + lane] = id;
            topk_weights[t * top_k + lane] = w;
        }
    }
    if (busy == 0) pmoe::align::begin_sort<NW>(o, E, smem, tid, 64 * NW);
    __syncthreads();
    const int id[1] = {tid < n_tokens * top_k ? ids[tid] : -1};
    pmoe::align::finish_sort<NW, 1>(id, o, E, id_bits, smem);
}

// Tokens that one workgroup routes and sorts faster than two launches do: a token per wave, or as many as take a wave four rounds
// of the top-k (one launch / two, us: 1 token, top 8 of 128 5.9 / 9.8, four per wave 16.8 / 10.3; top 2 of 8, two per wave 4.6 /
// 6.2, four 6.9 / 6.3; top 4 of 64, two per wave 6.6 / 6.9).
bool fits_small(int n_tokens, int E, int top_k) {
    const int nw = E <= 512 ? 16 : 8;
    return n_tokens * top_k <= nw * 64 && (n_tokens <= nw || (n_tokens + nw - 1) / nw * top_k <= 4);
}

template <typename T>
int launch_topk(const T *logits, const float *bias, int32_t *topk_ids, float *topk_weights, const pmoe::align::Outputs *o,
                int n_tokens, int E, int top_k, hipStream_t s) {
    auto with_epl = [&](auto go) {
        const int epl = (E + 63) / 64;
        if (epl <= 1) go(std::integral_constant<int, 1>{});
        else if (epl <= 2) go(std::integral_constant<int, 2>{});
        else if (epl <= 4) go(std::integral_constant<int, 4>{});
        else if (epl <= 8) go(std::integral_constant<int, 8>{});
        else go(std::integral_constant<int, 16>{});
    };
    if (o != nullptr) {
        with_epl([&](auto e) {
            constexpr int EPL = decltype(e)::value, NW = EPL <= 8 ? 16 : 8;
            const int n = n_tokens * top_k;
            const int64_t rows = n + (int64_t)std::min(n, E) * (o->pad_to - 1);
            const int reach = (int)std::min<int64_t>(o->max_padded, (rows + o->block_m - 1) / o->block_m * o->block_m);
            const int reach_blocks = (int)std::min<int64_t>(((int64_t)reach + o->block_m - 1) / o->block_m, o->max_blocks);
            const int64_t rest = std::max<int64_t>(o->max_padded - reach, 4 * ((int64_t)o->max_blocks - reach / o->block_m));
            const int fillers = (int)std::min<int64_t>((rest + NW * 256 - 1) / (NW * 256), 15);  // 16 bytes a thread and turn
            hipLaunchKernelGGL((route_small_kernel<NW, EPL, T>), dim3(1 + fillers), dim3(NW * 64), sizeof(int32_t) * (size_t)pmoe::align::sort_words(NW, E),
                               s, logits, bias, topk_ids, topk_weights, *o, reach, reach_blocks, n_tokens, E, top_k, pmoe::align::id_bits_for(E));
        });
        return pmoe::check_launch("route launch");
    }
    const dim3 grid((unsigned)((n_tokens + 3) / 4)), block(256);  // four tokens (waves) per workgroup
    with_epl([&](auto e) {
        hipLaunchKernelGGL((route_topk_kernel<decltype(e)::value, T>), grid, block, 0, s, logits, bias, topk_ids, topk_weights, n_tokens,
                           E, top_k);
    });
    return pmoe::check_launch("route_topk launch");
}

}  // namespace

extern "C" int pmoe_route(const void *logits, int logits_dtype, const float *bias, int32_t *topk_ids,
                          float *topk_weights, int32_t *sorted_token_ids, int32_t *expert_ids,
                          int32_t *num_tokens_post_padded, int n_tokens, int num_experts, int top_k, int block_m,
                          int pad_to, int max_padded, int max_blocks, void *workspace, size_t workspace_bytes,
                          void *stream) {
    PMOE_REQUIRE(n_tokens >= 0, "route: negative token count");
    PMOE_REQUIRE(num_experts > 0 && num_experts <= 1024, "route supports 1..1024 experts, got %d", num_experts);
    PMOE_REQUIRE(top_k > 0 && top_k <= kMaxTopK && top_k <= num_experts,
                 "route: top_k must be in 1..min(%d, num_experts), got %d", kMaxTopK, top_k);
    PMOE_REQUIRE(logits_dtype == PMOE_DTYPE_F32 || logits_dtype == PMOE_DTYPE_BF16, "route: logits must be fp32 or bf16");
    PMOE_REQUIRE((int64_t)n_tokens * top_k < (1ll << 31), "route: too many (token, slot) pairs");
    PMOE_REQUIRE(topk_ids && topk_weights && (logits || n_tokens == 0), "route: null pointer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool small = sorted_token_ids != nullptr && n_tokens > 0 && fits_small(n_tokens, num_experts, top_k);
    pmoe::align::Outputs o{sorted_token_ids, expert_ids, num_tokens_post_padded, block_m, pad_to, max_padded, max_blocks};
    if (small) {
        if (int rc = pmoe::moe_align_validate(topk_ids, sorted_token_ids, expert_ids, num_tokens_post_padded, n_tokens * top_k,
                                          num_experts, block_m, pad_to, max_padded, max_blocks))
            return rc;
    }
    if (n_tokens > 0) {
        const pmoe::align::Outputs *sort = small ? &o : nullptr;
        const int rc = logits_dtype == PMOE_DTYPE_F32
                           ? launch_topk(static_cast<const float *>(logits), bias, topk_ids, topk_weights, sort, n_tokens,
                                         num_experts, top_k, s)
                           : launch_topk(static_cast<const uint16_t *>(logits), bias, topk_ids, topk_weights, sort, n_tokens,
                                         num_experts, top_k, s);
        if (rc != PMOE_OK || small) return rc;
    }
    if (sorted_token_ids == nullptr) return PMOE_OK;  // top-k and weights only
    return pmoe_moe_align_ws(topk_ids, sorted_token_ids, expert_ids, num_tokens_post_padded, n_tokens * top_k,
                             num_experts, block_m, pad_to, max_padded, max_blocks, workspace, workspace_bytes, stream);
}

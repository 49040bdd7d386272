// Fused MoE forward for gfx950: the C entry points, the mxfp8 kernels (gate/up grouped GEMM + SwiGLU +
// on-chip MX requantisation, down GEMM) and the routing-weight reduction that ends both pipelines.  The
// bf16 kernels live in fused_moe_bf16.hip.
//
// Replaces the launchers and kernels of the reference's
// prime_moe/csrc/kernels/fused_moe_bf16_kernel.cu:930-964 (launcher) and fused_moe_mxfp8_kernel.cu:56-866.
//
// Pipeline of one call (all on the caller's stream):
//   prologue (row tiles and the schedule of the two kernels; inverts the sorted order: pair id -> sorted
//             row; mxfp8: re-tiles the scales of the gathered x rows)
//   -> up kernel (gate/up GEMM + SwiGLU, activation tile -> workspace)
//   -> down kernel (y[pair id, :K] = act . W2[e]^T, bf16, -> workspace)
//      (bf16, few up jobs: the up kernel plans for itself and its join follows, no prologue; one token or two:
//      moe_few.h, where the down kernel writes `out` itself)
//   -> finalize: out[t] = bf16(sum over the token's pairs p of w[p] * y[p]), fp32 sum in pair order;
//      split == 0: added to `out` (the reference's accumulate-into-out contract of its single-kernel
//      path), split != 0: `out` overwritten.
// Both values of `split` run the same kernels: on this hardware the two-kernel pipeline is the faster
// one at every shape, so `split` only selects what finalize does with `out`.  No value is accumulated with
// atomics and every sum has a fixed order: the result is a pure function of the inputs.
#include <algorithm>

#include "moe_pipeline.h"
#include "moe_ring.h"
#include "moe_stream_mx.h"

namespace pmoe {

// What one workgroup of an mxfp8 kernel does: `n_sub` consecutive weight tiles from `wt` on for the row tile
// of `nb` blocks starting at block `first`, expert `e`.
struct Job {
    int first, nb, wt, e, n_sub;
    bool w_once;  // no other row tile of this expert: nobody else reads the weight rows of this job
};

// Crowded schedules.  Without work lists (few rows per expert on average, see use_direct) neighbouring workgroups work on
// neighbouring weight tiles of one block.  With the tokens crowded on a few experts these have several full blocks: paired
// to row tiles, and 8 weight tiles by 4 row tiles to an XCD, their token rows are read from its L2.  How the tokens are
// spread is known on the device only, so where it may matter (crowding_possible_mx) the prologue is enqueued too, and
// it and the two kernels decide by this function whether they use its lists: more than 64 rows per live block, and more
// jobs than one round of the CUs, which pairing would leave idle.  Us without lists / as decided here, K 7168, N 4096,
// tokens x top 8 on some of 256 experts: 256 on 8 (no lists) 154 / 159, on 16 250 / 188, on 64 (no lists) 491 / 495; 300 on 8
// 231 / 182, on 16 260 / 210; 512 on 8 267 / 212, on 32 411 / 354; 768 on 32 500 / 406, on 64 582 / 570, Zipf 1938 / 1938.
// The prologue that finds nothing to do costs 2 to 4 us.
__host__ __device__ __forceinline__ bool crowded_mx(int64_t pairs, int64_t n_live, int n_wt_up, int n_cus) {
    return pairs > 64 * n_live && n_live * n_wt_up > n_cus;
}
__device__ __forceinline__ bool crowded_mx(const int32_t *ntpp, int n_blocks, int64_t pairs, int n_wt_up, int n_cus) {
    return crowded_mx(pairs, min((ntpp[0] + kBlockRows - 1) / kBlockRows, n_blocks), n_wt_up, n_cus);
}
// The arguments as the kernels use them: without the work list if nobody filled it.
__device__ __forceinline__ void settle_lists(MoeArgs &a) {
    if (a.crowd && !crowded_mx(a.ntpp, a.n_blocks, (int64_t)a.M * a.top_k, a.H / 128, a.crowd)) a.work = nullptr;
}

// Workgroup id -> job.  With a work list: one load from it, which the prologue lays out by workgroup id (see
// emit_work); entries of workgroups without work are -1.  Without one (few rows per expert, see use_direct): every
// live block is a row tile of its own, its jobs are consecutive workgroups.
__device__ __forceinline__ bool resolve_job(const MoeArgs &a, Job &j) {
    if (a.work == nullptr) {
        const int n_jobs = (a.n_wtiles + a.per_job - 1) / a.per_job;
        j.first = (int)blockIdx.x / n_jobs;
        if (j.first >= min((a.ntpp[0] + kBlockRows - 1) / kBlockRows, a.n_blocks)) return false;
        j.e = a.expert_ids[j.first];
        if (j.e < 0 || j.e >= a.E) return false;
        j.nb = 1;
        j.wt = ((int)blockIdx.x - j.first * n_jobs) * a.per_job;
        j.n_sub = min(a.per_job, a.n_wtiles - j.wt);
        // (Ids past the total name the last expert, so that one's last block counts as shared.  Compared with live blocks only
        // its weights would be read with the hint too: 100 tokens that all name the last of 257 experts, K 7168, N 512, took
        // 260 us instead of 245, the tail of the up kernel being that expert's two tiles.)
        j.w_once = (j.first == 0 || a.expert_ids[j.first - 1] != j.e) &&
                   (j.first + 1 >= a.n_blocks || a.expert_ids[j.first + 1] != j.e);
        return true;
    }
    const int4 w = a.work[blockIdx.x];
    if (w.x < 0) return false;
    j.first = w.x & 0x0fffffff;
    j.nb = w.x >> 28;
    j.wt = w.y & 0xffff;
    j.e = (w.y >> 16) & 0x3ff;
    j.n_sub = ((w.y >> 26) & 0xf) + 1;
    j.w_once = (w.w & 1) != 0;
    return true;
}

// The sorted rows of a row tile: two blocks, one per group of four waves.
struct RowInfo {
    int id[2 * kBlockRows];  // up kernel: token, down kernel: pair id (the row of y it writes); -1 for padding / dropped rows
    int nvalid[2];           // per group: 1 + index of the last live row
};

// Fills RowInfo for the `nb` blocks starting at `first`; returns the largest number of 32-row
// fragments up to the last live row in any group.
template <bool TOKENS>
__device__ __forceinline__ int load_row_info(const MoeArgs &a, int first, int nb, RowInfo &ri) {
    const int tid = threadIdx.x;
    if (tid < 2) ri.nvalid[tid] = 0;
    __syncthreads();
    if (tid < 2 * kBlockRows) {
        const int g = tid >> 7, s = first * kBlockRows + tid;
        const int p = g < nb && s < a.sorted_num ? a.sorted_ids[s] : -1;
        const int tok = p / a.top_k;
        const bool ok = p >= 0 && tok < a.M;
        ri.id[tid] = ok ? (TOKENS ? tok : p) : -1;
        if (ok) atomicMax(&ri.nvalid[g], (tid & 127) + 1);
    }
    __syncthreads();
    return (max(ri.nvalid[0], ri.nvalid[1]) + 31) >> 5;
}

// Epilogue of the down GEMM.  Weight rows (output columns) sit on the MFMA M side: register i of lane
// l = output column 64 w4 + 32 f + 8(i/4) + 4(l/32) + i%4 of sorted row 32 t + l%32.  Where the outputs of a tile of 256
// columns go: the y rows of its pairs (y is indexed by pair id, row pitch
// K; the last tile of a K that is not a multiple of 256 has 128 columns).
struct YDst {
    char *base;     // first column of the tile in row 0 of y
    int64_t pitch;  // bytes per row
    int cols;       // columns to write
};
__device__ __forceinline__ YDst y_destination(const MoeArgs &a, int k0) {
    YDst d;
    d.base = a.y + (int64_t)k0 * 2;
    d.pitch = (int64_t)a.K * 2;
    d.cols = min(kWRows, a.K - k0);
    return d;
}
// Tiles with a single live fragment skip the detour through LDS: every lane stores its 8-byte runs
// straight to the destination (32 rows x 16 KB per tile at most; a barrier and an LDS round trip cost more).
// `pair_r` = pair id of this lane's row (lane % 32) of the group, < 0 if the row holds none.
__device__ __forceinline__ void store_y_direct(const YDst &d, const f32x16 (&acc)[2][4], int n_rows, int w4, int lane,
                                               int pair_r) {
    const int r = lane & 31, half = lane >> 5;
    if (r >= n_rows || pair_r < 0) return;
    char *dst = d.base + pair_r * d.pitch;
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int col = 64 * w4 + 32 * f + 8 * g + 4 * half;
            if (col < d.cols) {
                uint2 pk;
                pk.x = pack2_bf16(acc[f][0][4 * g], acc[f][0][4 * g + 1]);
                pk.y = pack2_bf16(acc[f][0][4 * g + 2], acc[f][0][4 * g + 3]);
                *reinterpret_cast<uint2 *>(dst + col * 2) = pk;
            }
        }
}
// LDS written by some lanes of a wave is read by others of the same wave: LDS operations of a wave are executed in
// order, only the compiler has to keep them so.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// Larger tiles: a wave rounds a fragment (token rows 32 t .. of its group) of its 64 columns to bf16, transposes it through a
// scratch of its own, 16 rows at a time, and stores whole 128-byte lines.  `pair` = the pair ids of the fragment's rows (rows
// without one are skipped).  Before, the groups' 128 x 256 tiles went through 132 KB of LDS: on two full blocks the first slabs of
// the next weight tile could not be requested meanwhile, now they can (down kernel, 131072
// tokens on 32 experts of K = N = 2048: 1331 -> 1298 us; 24593 tokens, K 2048 x N 8192: 812 -> 800).
constexpr int kScratchRows = 16, kScratchPitch = 144;  // 128 B, 16 B pad
constexpr int kScratchBytes = kScratchRows * kScratchPitch;
__device__ __forceinline__ void store_y_fragment(const YDst &d, const f32x16 &lo, const f32x16 &hi, char *scratch, int w4, int lane,
                                                 const int *pair) {
    const int r = lane & 31, half = lane >> 5;
    const bool in_cols = 64 * w4 < d.cols;  // (a multiple of 128: a wave's 64 columns are inside or outside)
    char *dst = d.base + 128 * w4 + (lane & 7) * 16;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        if ((r >> 4) == h) {
#pragma unroll
            for (int f = 0; f < 2; ++f)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const f32x16 &v = f ? hi : lo;
                    uint2 pk;
                    pk.x = pack2_bf16(v[4 * g], v[4 * g + 1]);
                    pk.y = pack2_bf16(v[4 * g + 2], v[4 * g + 3]);
                    *reinterpret_cast<uint2 *>(scratch + (r & 15) * kScratchPitch + 64 * f + 16 * g + 8 * half) = pk;
                }
        }
        wave_lds_order();
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int row = (lane >> 3) + 8 * i, p = pair[16 * h + row];
            const uint4 v = *reinterpret_cast<const uint4 *>(scratch + row * kScratchPitch + (lane & 7) * 16);
            if (in_cols && p >= 0) store_once(dst + (int64_t)p * d.pitch, v);
        }
        wave_lds_order();
    }
}

// SwiGLU of the up GEMM, in registers: the 2H-wide gate/up tensor never leaves the chip.  `gate` and `up` hold gate rows and
// the matching up rows of one token fragment (weight rows on the MFMA M side: register i of lane l = activation column
// 8(i/4) + 4(l/32) + i%4 of the wave's 32 and of token row l%32).  Per token row amax -> e8m0 scale + e4m3 values: the wave's 32
// columns are one MX block, of which a lane holds 16 and the lane 32 on the others.  The two swap what makes their 16 bytes
// contiguous, and a row is stored in 32 bytes without a detour through LDS (`act`: the first of the wave's columns in the lane's
// row, `scale`: the row's scale byte; `live`: the row is wanted).  Before, the group's 128 x 128 tile was collected in LDS and
// stored in whole lines: two barriers, and the next weight tile's first slabs had to
// stay clear of the 38 KB (with the down kernel's change below, both kernels at 131072 tokens on 32 experts of K = N = 2048:
// 3455 -> 3400 us).
__device__ __forceinline__ void swiglu_store(const f32x16 &gate, const f32x16 &up, char *act, uint8_t *scale, bool live, int half) {
    float v[16], amax = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = swiglu(gate[i], up[i]);
#pragma unroll
    for (int i = 0; i < 16; ++i) amax = fmaxf(amax, fabsf(v[i]));
    const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(amax), __float_as_uint(amax), false, false);
    amax = fmaxf(__uint_as_float(both[0]), __uint_as_float(both[1]));
    uint32_t e8, q[4];
    float inv;
    mx_block_scale(amax, e8, inv);
#pragma unroll
    for (int g = 0; g < 4; ++g) q[g] = pack4_e4m3(v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3], inv);
    // lanes < 32: both halves of q[0], q[1] (columns 0 .. 15), lanes >= 32: those of q[2], q[3]
    const auto a = __builtin_amdgcn_permlane32_swap(q[0], q[2], false, false), b = __builtin_amdgcn_permlane32_swap(q[1], q[3], false, false);
    if (live) {
        store_once(act + 16 * half, make_uint4(a[0], a[1], b[0], b[1]));
        if (half == 0) *scale = (uint8_t)e8;
    }
}

// ==========================================================================================
// Two-group kernels on the ring engines
// ==========================================================================================

// Common set-up of the stage-ring loader.  Token rows: `tok_row_off(row)` gives the byte offset of
// tile row `row` (0..255: block 0, then block 1) in `tok_base`; weight rows: the tile's two 128-row
// halves start at w_base[0/1] with `w_pitch` bytes per row.  Scales (mxfp8): `tok_sc_off(row)` /
// `w_sc_off(row)` are the byte offsets of the row's first 4-scale dword; the dword of the next 128-wide
// K tile lies 512 bytes on in the blocked weight scales, tok_sc_step in the token side's (512 if they are tiled,
// 4 in a row-major matrix).  Only rows up to the last live one of each block are copied; those of the two blocks are
// packed one after the other in the stage (see ring::Layout).
template <int DT, int RB, typename TokOff, typename TokScOff, typename WScOff>
__device__ __forceinline__ void setup_ring_loader(ring::Loader<RB> &ld, const ring::Layout &lay, int tid,
                                                  uint32_t w_pitch, const RowInfo &ri,
                                                  bool w_once, TokOff tok_row_off,
                                                  const uint8_t *tok_sc_base, uint32_t tok_sc_step, TokScOff tok_sc_off,
                                                  const uint8_t *w_sc_base, WScOff w_sc_off) {
    using L = ring::Loader<RB>;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
#pragma unroll
    for (int q = 0; q < L::N; ++q) {
        const int row = L::row_of(wave, lane, q);          // row inside a 128-row block / half
        const int row0 = L::row_of(wave, 0, q);            // first row of the instruction
        const uint32_t gchunk = (uint32_t)((lane % (RB / 16)) ^ ring::swz<RB>(row)) * 16u;  // global chunk of this lane's slot
        ld.w_off[q] = (uint32_t)row * w_pitch + gchunk;
        ld.w_dst[0][q] = lay.w_off + row0 * RB;
        ld.w_dst[1][q] = ld.w_dst[0][q] + 128 * RB;
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            ld.tok_dst[g][q] = -1;
            ld.tok_off[g][q] = 0;
            ld.tok_live[g][q] = ri.id[g * kBlockRows + row] >= 0;
            if (__ballot(ld.tok_live[g][q]) != 0) {
                ld.tok_dst[g][q] = g * lay.group1_off + row0 * RB;
                ld.tok_off[g][q] = tok_row_off(g * kBlockRows + row) + gchunk;
            }
        }
    }
    ld.sc_base = nullptr;
    ld.sc_off = 0;
    ld.sc_step = 0;
    ld.sc_dst = -1;
    ld.sc_live = true;
    if constexpr (DT == DT_FP8) {
        if (wave >= 4) {  // weight rows 64 (wave - 4) + lane
            const int row = 64 * (wave - 4) + lane;
            ld.sc_base = reinterpret_cast<const char *>(w_sc_base);
            ld.sc_off = w_sc_off(row);
            ld.sc_step = 512u;
            ld.sc_dst = lay.scale_off + (lay.tok_rows + 64 * (wave - 4)) * 4;
        } else if (64 * wave < lay.tok_rows) {
            // packed token rows 64 wave + lane
            const int c = 64 * wave + lane;
            ld.sc_live = c < lay.tok_rows;
            const int cc = min(c, lay.tok_rows - 1);
            const int row = cc < lay.rows0 ? cc : kBlockRows + cc - lay.rows0;
            ld.sc_base = reinterpret_cast<const char *>(tok_sc_base);
            ld.sc_off = tok_sc_off(row);
            ld.sc_step = tok_sc_step;
            ld.sc_dst = lay.scale_off + 64 * wave * 4;
        }
    }
    int lps = 2 * L::N + (ld.sc_dst >= 0);
#pragma unroll
    for (int q = 0; q < L::N; ++q) lps += (ld.tok_dst[0][q] >= 0) + (ld.tok_dst[1][q] >= 0);
    ld.lps = lps;
    ld.w_once = w_once;
    ld.make_uniform();
}

// First slab of this workgroup's walk over K: workgroups that run side by side on an XCD (consecutive
// blockIdx / 8) start 128 bytes apart, 8 distinct phases over a 1 KB period.  The spread keeps the
// workgroups that share a weight tile off the same HBM channel at the same instant, and stays short
// enough that they still meet in L2 (a 16-phase, 4 KB spread read 30 % more from HBM for the same time).
// Without a work list and with rows of whole 4 KB there are 32 phases.  Neighbouring weight tiles then run side by side all
// over the chip and the same bytes of all their rows lie on few channels.  Us with 8 phases / with 32 / in the order of
// the work lists: up kernel at 24 tokens x top 2 on 8 experts of K 4096 x N 28672 192 / 160 / 177, down kernel of K 7168 x N
// 16384 at 64 tokens 94 / 81 / 106, the whole op at 64 tokens on 32 experts of K 4096 x N 8192 298 / 272 / 305.  Rows of other
// lengths start on different channels by themselves (K 7168: 152 and 152).
template <int RB>
__device__ __forceinline__ int slab_rotation(const MoeArgs &a, int n_slabs) {
    const int phases = a.work == nullptr && (n_slabs * RB) % 4096 == 0 ? 4096 / RB : 8;
    return (int)((blockIdx.x >> 3) & (phases - 1)) % n_slabs;
}

template <int NTF>
__device__ __forceinline__ void zero_acc(f32x16 (&acc)[2][4]) {
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int t = 0; t < NTF; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[f][t][i] = 0.f;
}
// Runs the tile code of a group with `ntf` live fragments.  The two groups of a workgroup may take different cases: the
// barriers of all of them are the same.
template <typename Run>
__device__ __forceinline__ void by_fragments(int ntf, Run run) {
    switch (ntf) {
        case 0: run(std::integral_constant<int, 0>{}); break;
        case 1: run(std::integral_constant<int, 1>{}); break;
        case 2: run(std::integral_constant<int, 2>{}); break;
        case 3: run(std::integral_constant<int, 3>{}); break;
        default: run(std::integral_constant<int, 4>{}); break;
    }
}

// Up kernel tile on the stage ring: the live rows of one or two row blocks x activation
// columns [128 ht, 128 ht + 128).  LDS weight rows 0..127 are gate rows, 128..255 the matching up rows;
// wave v of a group owns gate/up rows 32v..32v+31 so gate and up of one activation element sit in the
// same lane and register.
template <int DT, int RB, int NTF>
__device__ __forceinline__ void up_tile_ring(const MoeArgs &a, const Job &job, int rows0, int rows1, const RowInfo &ri, char *lds) {
    constexpr int ES = 1;  // bytes per element
    const int first = job.first, ht = job.wt, n_sub = job.n_sub, e = job.e;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = wave >> 2, w4 = wave & 3;
    const int my_rows = grp ? rows1 : rows0;
    const int K = a.K, H = a.H, N = a.N;
    const ring::Layout lay = ring::make_layout<DT, RB>(rows0, rows1, ring::ring_bytes<DT>());

    int h0 = ht * 128;
    const int n_slabs = (K * ES) / RB;
    ring::Loader<RB> ld;
    ld.tok_base = a.x;
    ld.w_base[0] = a.w1 + ((int64_t)e * N + h0) * K * ES;
    ld.w_base[1] = ld.w_base[0] + (int64_t)H * K * ES;
    const uint32_t row_bytes = (uint32_t)(K * ES);
    const int kb = K >> 5, kt128 = K >> 7;
    auto token = [&](int row) { return (uint32_t)max(ri.id[row], 0); };
    setup_ring_loader<DT, RB>(
        ld, lay, tid, row_bytes, ri, job.w_once, [&](int row) { return token(row) * row_bytes; },
        a.work != nullptr ? reinterpret_cast<const uint8_t *>(a.xs_tiled + (int64_t)first * kt128 * kBlockRows) : a.x_scales,
        a.work != nullptr ? 512u : 4u,
        [&](int row) {
            return a.work != nullptr ? (uint32_t)(((row >> 7) * kt128 * kBlockRows + (row & 127)) * 4)
                                     : (uint32_t)(token(row) * kb);
        },
        a.w1_scales + (int64_t)e * N * kb,
        [&](int row) { return (uint32_t)blocked_scale_off((row < 128 ? h0 : H + h0 - 128) + row, 0, K >> 7); });

    const int wrow[2] = {32 * w4, 128 + 32 * w4};
    const int start = slab_rotation<RB>(a, n_slabs);
    const int tok_region = grp ? lay.group1_off : 0;
    const int64_t row0 = (int64_t)(first + grp) * kBlockRows;
    int n_pre = 0;
    for (int sub = 0; sub < n_sub; ++sub) {
        f32x16 acc[2][4];
        zero_acc<NTF>(acc);
        ring::main_loop<DT, RB, NTF>(acc, ld, lay, lds, n_slabs, wrow, lane, tok_region, start, n_pre);
        if (sub + 1 < n_sub) {
            // same token rows, the next 128 gate and 128 up rows of the expert; their first slabs under this tile's epilogue
            ld.w_base[0] += (int64_t)128 * K * ES;
            ld.w_base[1] += (int64_t)128 * K * ES;
            if (DT == DT_FP8 && wave >= 4) ld.sc_off += (uint32_t)kt128 * 512u;
            ld.make_uniform();
            n_pre = lay.stages;
            ring::pre_issue<DT, RB>(ld, lay, lds, n_slabs, start, n_pre);
        }
#pragma unroll
        for (int t = 0; t < NTF; ++t) {
            const int row = 32 * t + (lane & 31);
            uint8_t *scale = reinterpret_cast<uint8_t *>(a.act_scales + ((row0 >> 7) * (H >> 7) + (h0 >> 7)) * kBlockRows + row) + w4;
            swiglu_store(acc[0][t], acc[1][t], a.act + (row0 + row) * H + h0 + 32 * w4, scale, row < my_rows, lane >> 5);
        }
        h0 += 128;
    }
}

// LDS plan of the mxfp8 kernels: ring and row table.
template <int DT>
struct SplitLds {
    static constexpr int kRing = ring::ring_bytes<DT>();
    static constexpr int kRowInfoOff = kRing;
    static constexpr int kTotal = 160 * 1024;
    static_assert(kRowInfoOff + sizeof(RowInfo) <= kTotal, "row table does not fit its slot");
};

template <int DT>
__global__ __launch_bounds__(512) void moe_up_kernel(MoeArgs a) {
    using L = SplitLds<DT>;
    __shared__ __attribute__((aligned(1024))) char lds[L::kTotal];
    RowInfo &ri = *reinterpret_cast<RowInfo *>(lds + L::kRowInfoOff);
    settle_lists(a);
    if (a.work == nullptr) stream::invert(a, 512);  // (no prologue did)
    Job j;
    if (!resolve_job(a, j)) return;
    if (load_row_info<true>(a, j.first, j.nb, ri) == 0) return;
    const int rows0 = __builtin_amdgcn_readfirstlane(ri.nvalid[0]), rows1 = __builtin_amdgcn_readfirstlane(ri.nvalid[1]);
    const int my_rows = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) ? rows1 : rows0;
    by_fragments((my_rows + 31) >> 5, [&](auto n) { up_tile_ring<DT, ring::kRB, decltype(n)::value>(a, j, rows0, rows1, ri, lds); });
}

// Down kernel tile on the stage ring: y[rows, 256 cols of K] = act[rows, :H] . W2[e][cols, :H]^T, the
// whole reduction over H inside the workgroup; the
// routing weights are applied later, by finalize_kernel.  `ntf`: fragments of the larger group.
template <int DT, int RB, int NTF>
__device__ __forceinline__ void down_tile_ring(const MoeArgs &a, const Job &job, int ntf, int rows0, int rows1, const RowInfo &ri,
                                               char *lds) {
    constexpr int ES = 1;  // bytes per element
    const int first = job.first, kt = job.wt, n_sub = job.n_sub, e = job.e;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = wave >> 2, w4 = wave & 3;
    const int K = a.K, H = a.H;
    const int64_t row0 = (int64_t)first * kBlockRows;
    const int my_rows = grp ? rows1 : rows0;  // rows past the last live one are never read back
    const int my_pair = ri.id[grp * kBlockRows + (lane & 31)];  // (tiles of one fragment store from registers)
    const ring::Layout lay = ring::make_layout<DT, RB>(rows0, rows1, ring::ring_bytes<DT>());

    int k0 = kt * kWRows;
    const uint32_t row_bytes = (uint32_t)(H * ES);
    const int hb = H >> 5, ht128 = H >> 7;
    const int n_slabs = (H * ES) / RB;
    ring::Loader<RB> ld;
    ld.tok_base = a.act + row0 * H * ES;
    // weight rows (output columns) k0 .. k0 + 255 of the expert; the last tile of a K that is not a
    // multiple of 256 has 128 of them and reads the first half twice
    auto set_weights = [&](int k) {
        ld.w_base[0] = a.w2 + ((int64_t)e * K + k) * H * ES;
        ld.w_base[1] = (k + 128 < K) ? ld.w_base[0] + (int64_t)128 * H * ES : ld.w_base[0];
        if (DT == DT_FP8 && wave >= 4)
            ld.sc_off = (uint32_t)blocked_scale_off(min(k + 64 * (wave - 4) + lane, K - 1), 0, ht128);
    };
    set_weights(k0);
    setup_ring_loader<DT, RB>(
        ld, lay, tid, row_bytes, ri, job.w_once, [&](int row) { return (uint32_t)row * row_bytes; },
        reinterpret_cast<const uint8_t *>(a.act_scales + (int64_t)first * ht128 * kBlockRows), 512u,
        [&](int row) { return (uint32_t)(((row >> 7) * ht128 * kBlockRows + (row & 127)) * 4); },
        a.w2_scales + (int64_t)e * K * hb,
        [&](int row) { return (uint32_t)blocked_scale_off(min(k0 + row, K - 1), 0, ht128); });

    const int wrow[2] = {64 * w4, 64 * w4 + 32};
    const int start = slab_rotation<RB>(a, n_slabs);
    const int tok_region = grp ? lay.group1_off : 0;
    const int SB = lay.stage_bytes, NS = lay.stages;
    // the ring is free after main_loop (it ends with a barrier): its end holds the scratch of the waves (tiles of one fragment
    // store from registers); the next weight tile's copies start in the stages in front of it, under this tile's epilogue
    constexpr int kScratchOff = ring::ring_bytes<DT>() - 8 * kScratchBytes;
    const int ahead = __builtin_amdgcn_readfirstlane(ntf == 1 ? NS : min(NS, kScratchOff / SB));
    char *scratch = lds + kScratchOff + wave * kScratchBytes;
    int n_pre = 0;
    for (int sub = 0; sub < n_sub; ++sub) {
        f32x16 acc[2][4];
        zero_acc<NTF>(acc);
        ring::main_loop<DT, RB, NTF>(acc, ld, lay, lds, n_slabs, wrow, lane, tok_region, start, n_pre);
        const bool more = sub + 1 < n_sub;
        if (more) {
            set_weights(k0 + kWRows);
            ld.make_uniform();
            n_pre = ahead;
            ring::pre_issue<DT, RB>(ld, lay, lds, n_slabs, start, n_pre);
        }
        const YDst dst = y_destination(a, k0);
        if (ntf == 1) {
            if (NTF > 0) store_y_direct(dst, acc, my_rows, w4, lane, my_pair);
        } else {
#pragma unroll
            for (int t = 0; t < NTF; ++t)
                store_y_fragment(dst, acc[0][t], acc[1][t], scratch, w4, lane, ri.id + grp * kBlockRows + 32 * t);
            if (more && ahead < NS) __syncthreads();  // the scratch has been read: the ring may be filled there
        }
        k0 += kWRows;
    }
}

template <int DT>
__global__ __launch_bounds__(512) void moe_down_kernel(MoeArgs a) {
    using L = SplitLds<DT>;
    __shared__ __attribute__((aligned(1024))) char lds[L::kTotal];
    RowInfo &ri = *reinterpret_cast<RowInfo *>(lds + L::kRowInfoOff);
    settle_lists(a);
    Job j;
    if (!resolve_job(a, j)) return;
    const int ntf = load_row_info<false>(a, j.first, j.nb, ri);
    if (ntf == 0) return;
    const int rows0 = __builtin_amdgcn_readfirstlane(ri.nvalid[0]), rows1 = __builtin_amdgcn_readfirstlane(ri.nvalid[1]);
    const int my_rows = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) ? rows1 : rows0;
    by_fragments((my_rows + 31) >> 5, [&](auto n) { down_tile_ring<DT, ring::kRB, decltype(n)::value>(a, j, ntf, rows0, rows1, ri, lds); });
}

// Walk order of the tiles of one mxfp8 kernel: [group of 8 weight tiles][row tile][weight tile in group].
// The ~32 workgroups that run side by side on an XCD are then 4 consecutive row tiles (mostly of one
// expert) x 8 weight tiles: every token slab they fetch is shared by 8 weight tiles and every weight
// slab by the row tiles of its expert, inside that XCD's L2.
// Hardware hands consecutive workgroup ids to the 8 XCDs round-robin, so position `l` of the walk
// is given to workgroup id 8 * (l mod per_xcd) + l / per_xcd: one XCD then runs a contiguous range of
// the walk.  The entry carries everything the workgroup needs to start: x = first block | blocks << 28,
// y = first weight tile | expert << 16 | (weight tiles - 1) << 26 (experts < 1024, up to 16 weight
// tiles), w = 1 if the row tile is the only one of its expert.
//
// The work list of a kernel with n_wt weight tiles, of which a workgroup takes `per_job` consecutive ones, over `n_tiles` row
// tiles {first block | blocks << 28, expert}, has `grid` entries: -1 where the walk has ended or a block names no expert.
struct ListShape {
    int n_wt, per_job, n_jobs, total, per_xcd;
    __device__ __forceinline__ ListShape(int n_wt_, int per_job_, int n_tiles) : n_wt(n_wt_), per_job(per_job_) {
        n_jobs = (n_wt + per_job - 1) / per_job;
        total = n_tiles * n_jobs;
        per_xcd = (total + 7) >> 3;
    }
};
__device__ __forceinline__ int4 list_entry(const ListShape &l, const int2 *tiles, int n_tiles, int num_experts, int t, int j) {
    const int2 tl = tiles[t];
    if (tl.y < 0 || tl.y >= num_experts) return make_int4(-1, -1, 0, 0);
    // (the only row tile of its expert: then nobody else reads that expert's weight rows)
    const bool shared = (t > 0 && tiles[t - 1].y == tl.y) || (t + 1 < n_tiles && tiles[t + 1].y == tl.y);
    const int wt = j * l.per_job, cnt = min(l.per_job, l.n_wt - wt);
    return make_int4(tl.x, wt | (tl.y << 16) | ((cnt - 1) << 26), 0, shared ? 0 : 1);
}
constexpr int kListGroup = 8;  // weight tiles of a group of the walk
// Thread `me` of `threads` writes entries me, me + threads, ...: by position, so that neighbouring threads write neighbouring entries
// and nobody has to clear the list before.
__device__ __forceinline__ void emit_work(int4 *work, int grid, const ListShape &s, const int2 *tiles, int n_tiles, int num_experts, int me,
                                          int threads) {
    constexpr int GW = kListGroup;
    for (int w = me; w < grid; w += threads) {
        const int pos = w >> 3, l = (w & 7) * s.per_xcd + pos;
        int4 entry = make_int4(-1, -1, 0, 0);
        if (pos < s.per_xcd && l < s.total) {
            const int wg = l / (GW * n_tiles), rem = l - wg * GW * n_tiles;
            const int gw = min(GW, s.n_jobs - wg * GW), t = rem / gw;
            entry = list_entry(s, tiles, n_tiles, num_experts, t, wg * GW + rem - t * gw);
        }
        work[w] = entry;
    }
}
// The same list, a row tile of a thread after the other: where the tiles are in memory, an entry is too little to wait for them.
__device__ __forceinline__ void emit_work_by_tile(int4 *work, int grid, const ListShape &s, const int2 *tiles, int n_tiles, int num_experts,
                                                  int me, int threads) {
    constexpr int GW = kListGroup;
    for (int w = me; w < grid; w += threads) {
        const int pos = w >> 3;
        if (pos >= s.per_xcd || (w & 7) * s.per_xcd + pos >= s.total) work[w] = make_int4(-1, -1, 0, 0);
    }
    for (int t = me; t < n_tiles; t += threads) {
        const int4 first = list_entry(s, tiles, n_tiles, num_experts, t, 0);
        for (int j = 0; j < s.n_jobs; ++j) {
            const int wg = j / GW, l = wg * GW * n_tiles + t * min(GW, s.n_jobs - wg * GW) + (j - wg * GW);
            const int xcd = l / s.per_xcd, wt = j * s.per_job, cnt = min(s.per_job, s.n_wt - wt);
            work[8 * (l - xcd * s.per_xcd) + xcd] =
                first.x < 0 ? first : make_int4(first.x, (first.y & (0x3ff << 16)) | wt | ((cnt - 1) << 26), 0, first.w);
        }
    }
}

// Prologue of an mxfp8 call.  The first workgroups build the row tiles and work lists of the two-group kernels:
// consecutive blocks of one expert are paired, an expert's odd last block stays single (one pass of
// block-wide scans per 256 blocks, then the two walk orders).  Each of them works out all tiles, in LDS, and writes its
// share of the lists; only of more than kLdsTiles blocks workgroup 0 writes them alone, from tiles in the workspace, a tile at a time
// (140000 tokens on 32 experts, K = N = 2048, by position there 81.9, by tile 63.7 us).  What bounds it is
// the chain of scans; the lists of 4096 tokens on 256 experts have 22440 entries, 11264 of them jobs.
// A builder comes late to its share of the rest, so there are only as many as the lists are long (kListEntries).  Prologue with one builder /
// one per 512 entries / a quarter of the workgroups, us: 600 tokens on 8 experts (K = N = 512) 4.2 / 4.4 / 5.3, 2000 on 8 (K 2048, N 512) 4.8 /
// 4.9 / 6.0, 4000 on 16 (K 4096, N 2048) 7.2 / 6.0 / 8.8, 24593 on 32 (K = N = 2048) 17.5 / 10.8 / 10.4, 6000 on 128 (K 2048, N 1536) 13.4 /
// 7.9 / 7.7, 4096 on 257 (K 7168, N 512) 15.0 / 9.9 / 9.7.
// The re-tiling of the x scales is done with eight rows of every lane in flight, a block per workgroup and no division in the loop.  Prologue
// with a row and its token at a time and the lists by one workgroup / as it is, us: 4096 tokens on 256 experts (K 7168, N 4096) 28.7 /
// 10.9, 24593 on 32 16.6 / 10.8, 2000 on 8 9.7 / 4.9.  Beyond some 100 us the layer shows nothing of it.
// All workgroups invert the sorted order: inv[pair id] = sorted row.  Entries of pairs that are not
// in the schedule keep whatever the buffer held; the reader validates an entry against sorted_ids.
// CROWD: only for crowded schedules (`n_cus`: see crowded_mx).
constexpr int kLdsTiles = kBlockRows * 65 / 2;
constexpr int kListEntries = 512;  // of both lists, a builder each
template <bool CROWD>
__global__ __launch_bounds__(256) void moe_prologue_kernel(const int32_t *expert_ids, const int32_t *ntpp,
                                                           int n_blocks, int2 *tiles, int *n_tiles,
                                                           int4 *work_up, int n_wt_up, int per_job_up, int grid_up,
                                                           int4 *work_down, int n_wt_down, int per_job_down,
                                                           int grid_down, int num_experts,
                                                           const int32_t *sorted_ids, int sorted_num, int32_t *inv,
                                                           int n_pairs, int do_invert, const uint8_t *x_scales,
                                                           uint32_t *xs_tiled, int nkt, int top_k, int M, int n_cus) {
    if (CROWD && !crowded_mx(ntpp, n_blocks, n_pairs, n_wt_up, n_cus)) return;
    const int n_live = min((ntpp[0] + kBlockRows - 1) / kBlockRows, n_blocks);
    const int builders = n_live <= kLdsTiles ? max(min(min((grid_up + grid_down) / kListEntries, (int)gridDim.x / 4), 32), 1) : 1;
    __shared__ alignas(16) uint32_t s_sc[kBlockRows][65];  // row tiles first
    static_assert(kLdsTiles * sizeof(int2) <= sizeof(s_sc), "the row tiles fit");
    if ((int)blockIdx.x < builders) {
        __shared__ int s_max[4], s_sum[4], s_carry[2];
        const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
        int2 *table = n_live <= kLdsTiles ? reinterpret_cast<int2 *>(&s_sc[0][0]) : tiles;
        if (tid == 0) { s_carry[0] = 0; s_carry[1] = 0; }
        __syncthreads();
        for (int base = 0; base < n_live; base += 256) {
            const int b = base + tid;
            const bool live = b < n_live;
            const int e = live ? expert_ids[b] : -2;
            const int prev = (live && b > 0) ? expert_ids[b - 1] : -1;
            int v = (live && e != prev) ? b : -1;  // start of a run of equal experts
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int t = __shfl_up(v, d, 64);
                if (lane >= d) v = max(v, t);
            }
            if (lane == 63) s_max[wave] = v;
            __syncthreads();
            int run_start = s_carry[0];
            for (int w = 0; w < wave; ++w) run_start = max(run_start, s_max[w]);
            run_start = max(run_start, v);
            const bool leader = live && (((b - run_start) & 1) == 0);
            const bool paired = leader && (b + 1 < n_live) && expert_ids[b + 1] == e;
            int incl = leader ? 1 : 0;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int t = __shfl_up(incl, d, 64);
                if (lane >= d) incl += t;
            }
            if (lane == 63) s_sum[wave] = incl;
            __syncthreads();
            int off = s_carry[1];
            for (int w = 0; w < wave; ++w) off += s_sum[w];
            if (leader) table[off + incl - 1] = make_int2(b | (paired ? 2 : 1) << 28, e);
            __syncthreads();
            if (tid == 255) { s_carry[0] = run_start; s_carry[1] = off + incl; }
            __syncthreads();
        }
        const int nt = s_carry[1];
        if (blockIdx.x == 0 && tid == 0) n_tiles[0] = nt;
        __threadfence_block();
        __syncthreads();  // tiles written above are read below by other threads
        const int me = (int)blockIdx.x * 256 + tid, threads = builders * 256;
        const ListShape up(n_wt_up, per_job_up, nt), down(n_wt_down, per_job_down, nt);
        if (n_live <= kLdsTiles) {
            emit_work(work_up, grid_up, up, table, nt, num_experts, me, threads);
            emit_work(work_down, grid_down, down, table, nt, num_experts, me, threads);
        } else {
            emit_work_by_tile(work_up, grid_up, up, table, nt, num_experts, me, threads);
            emit_work_by_tile(work_down, grid_down, down, table, nt, num_experts, me, threads);
        }
        __syncthreads();  // (a workgroup that re-tiles, too, uses the LDS again)
    }
    if (do_invert) {
        const int n_rows = min(ntpp[0], sorted_num);
        const int stride = (int)(gridDim.x * blockDim.x);
        for (int s = (int)(blockIdx.x * blockDim.x + threadIdx.x); s < n_rows; s += stride) {
            const int p = sorted_ids[s];
            const int e = expert_ids[s >> 7];  // rows of a block without an expert are not computed
            if (p >= 0 && p < n_pairs && e >= 0 && e < num_experts) inv[p] = s;
        }
    }
    if (do_invert && xs_tiled != nullptr) {
        // the e8m0 scales of the gathered x rows, re-tiled for the up kernel's loader (see
        // MoeArgs::xs_tiled); rows without a token get 2^0.  One sorted block per turn, through LDS so
        // that both the reads (a row's scales) and the writes (128 rows of one K tile) are contiguous.
        // The workgroups that build the lists take no share unless there is only one.
        __shared__ int s_tok[kBlockRows];
        const int tid = threadIdx.x;
        const int workers = gridDim.x > 1 ? (int)gridDim.x - builders : 1;
        const int me = gridDim.x > 1 ? (int)blockIdx.x - builders : 0;
        const uint32_t *xs = reinterpret_cast<const uint32_t *>(x_scales);  // nkt dwords per token
        for (int b = me; b >= 0 && b < n_live; b += workers) {
            if (tid < kBlockRows) {
                const int srow = b * kBlockRows + tid;
                const int p = srow < sorted_num ? sorted_ids[srow] : -1;
                int tok = p >= 0 ? p / top_k : -1;
                if (tok >= M) tok = -1;
                s_tok[tid] = tok;
            }
            __syncthreads();
            for (int c0 = 0; c0 < nkt; c0 += 64) {
                const int cw = min(64, nkt - c0);
                // a row's dwords by 2^sh lanes, eight rows of every lane in flight
                const int sh = cw > 1 ? 32 - __builtin_clz(cw - 1) : 0, c = tid & ((1 << sh) - 1), rows = 256 >> sh;
                for (int r0 = tid >> sh; r0 < kBlockRows; r0 += 8 * rows) {
                    uint32_t v[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        const int r = r0 + u * rows, tok = r < kBlockRows && c < cw ? s_tok[r] : -1;
                        v[u] = tok >= 0 ? xs[(int64_t)tok * nkt + c0 + c] : 0x7f7f7f7fu;
                    }
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        if (r0 + u * rows < kBlockRows && c < cw) s_sc[r0 + u * rows][c] = v[u];
                }
                __syncthreads();
#pragma unroll 4
                for (int i = tid; i < kBlockRows * cw; i += 256) {
                    const int c = i >> 7, r = i & 127;
                    xs_tiled[((int64_t)b * nkt + c0 + c) * kBlockRows + r] = s_sc[r][c];
                }
                __syncthreads();
            }
        }
    }
}

// Weight-streaming kernels (moe_stream_mx.h).  n_tiles: weight tiles per block (0: the up kernel only inverts).
template <bool UP>
__global__ __launch_bounds__(512, 4) void moe_stream_kernel_mx(MoeArgs a, int n_tiles) {
    __shared__ __attribute__((aligned(1024))) stream::Shared sh;
    stream::for_each_job<UP>(a, n_tiles, [](int) { return false; },
                             [&](int blk, int e, int tile, int id) { stream::mx_run_job<UP>(a, sh, blk, e, tile, id); });
}

// Down GEMM for H = RB without a prologue (see stream::for_each_turn).
template <int RB>
__global__ __launch_bounds__(256, 2) void moe_stream_down_short_kernel_mx(MoeArgs a) {
    __shared__ __attribute__((aligned(1024))) char bufs[4][stream::ShortDownMx<RB>::kBytes];
    stream::ShortDownMx<RB> eng(a, bufs[__builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6)]);
    stream::for_each_turn(a, a.K / stream::ShortDownMx<RB>::kTurnCols, eng);
}

// out[t] = bf16(sum over the token's top_k pairs p, in pair order, of w[p] * y[p]) (ACCUMULATE: added to
// what `out` holds).  A pair counts if inv[p] is a row of the schedule that really holds p in a block with
// an expert; otherwise the schedule dropped it, nobody wrote y[p], and it contributes nothing.  A pair id
// that the schedule lists more than once contributes once (if its rows lie in blocks of different experts,
// which of them is unspecified).
//
// One wave per (token, piece of 512 columns): lanes 0 .. top_k - 1 resolve the token's pairs (inv, sorted_ids,
// expert_ids, routing weight), the result is broadcast, and then every lane reads its 8 columns of the top_k rows of y
// (contiguous: y is indexed by pair id), G loads in flight at a time.
//
// Bound by the read of y and by the chain of loads that resolves the pairs in front of it, so waves must be many, each
// with little to do: a wave per piece resolves the pairs again for every piece (from L2) and is faster all the same than
// one that keeps them for a run of pieces, and a launch as large as the work than 16384 workgroups that each come back for
// more.  Before / after, K 2048 unless said: 58.6 / 50.9 us at 8192 tokens x top 8 (5.9 TB/s), 117.5 / 98 at 16000 x 8,
// 345 / 316 at 100000 x 4, 100 / 88 at 4096 x 8 with K 7168; 15.4 / 14.7 at 2000 x 8, the same at 200 x 9.  Eight loads
// in flight instead of four cost registers: 15.6 us at 2000 x 8, 7.4 / 7.0 at 200 x 9, nothing gained above.
template <bool ACCUMULATE, int G>
__global__ __launch_bounds__(256) void finalize_kernel(const char *y, const int32_t *inv, const int32_t *sorted_ids,
                                                       const int32_t *ntpp, int sorted_num, const float *topk_w,
                                                       int top_k, int M, int K, char *out,
                                                       const int32_t *expert_ids, int num_experts, int pieces) {
    const int lane = threadIdx.x & 63;
    const int n_rows = min(ntpp[0], sorted_num);
    const int64_t n_items = (int64_t)M * pieces;
    const int64_t wave_stride = (int64_t)gridDim.x * (blockDim.x >> 6);
    for (int64_t item = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); item < n_items; item += wave_stride) {
        const int t = (int)(item / pieces);
        const int col = (int)(item - (int64_t)t * pieces) * 512 + lane * 8;
        const bool in_range = col < K;
        for (int r0 = 0; r0 < top_k; r0 += 64) {
            // lane r resolves pair r0 + r: its weight, or 0 with `ok` unset
            float w_mine = 0.f;
            bool ok = false;
            if (r0 + lane < top_k) {
                const int p = t * top_k + r0 + lane;
                const int row = inv[p];
                ok = row >= 0 && row < n_rows;
                if (ok) ok = sorted_ids[row] == p;
                if (ok) {
                    const int e = expert_ids[row >> 7];
                    ok = e >= 0 && e < num_experts;
                }
                if (ok) w_mine = topk_w[p];
            }
            const uint64_t ok_mask = __ballot(ok);
            const int n_here = min(64, top_k - r0);
            float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            if (r0 > 0 || ACCUMULATE) {
                if (in_range) {
                    const uint4 prev = *reinterpret_cast<const uint4 *>(out + ((int64_t)t * K + col) * 2);
                    const uint32_t u[4] = {prev.x, prev.y, prev.z, prev.w};
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        v[2 * j] = bf16_bits_to_f32(u[j] & 0xffffu);
                        v[2 * j + 1] = bf16_bits_to_f32(u[j] >> 16);
                    }
                }
            }
            for (int g0 = 0; g0 < n_here; g0 += G) {
                uint4 q[G];
                float w[G];
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const int r = g0 + g;  // wave-uniform
                    const bool live = r < n_here && ((ok_mask >> r) & 1);
                    w[g] = __shfl(w_mine, r < 64 ? r : 0, 64);
                    q[g] = make_uint4(0, 0, 0, 0);
                    if (live && in_range) q[g] = load_once(y + ((int64_t)(t * top_k + r0 + r) * K + col) * 2);
                    if (!live) w[g] = 0.f;
                }
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const uint32_t u[4] = {q[g].x, q[g].y, q[g].z, q[g].w};
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        v[2 * j] += w[g] * bf16_bits_to_f32(u[j] & 0xffffu);
                        v[2 * j + 1] += w[g] * bf16_bits_to_f32(u[j] >> 16);
                    }
                }
            }
            if (in_range) {
                uint32_t o[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) o[j] = pack2_bf16(v[2 * j], v[2 * j + 1]);
                store_once(out + ((int64_t)t * K + col) * 2, make_uint4(o[0], o[1], o[2], o[3]));
            }
        }
    }
}

// ------------------------------------------------------------------------------------------ host

struct WorkspaceLayout {
    size_t n_tiles_off, tiles_off, work_up_off, work_down_off, inv_off, y_off, act_off, act_scales_off, xs_tiled_off, total;
};

// Workspace of an mxfp8 call.
static WorkspaceLayout workspace_layout(int M, int K, int N, int sorted_num, int top_k) {
    WorkspaceLayout l{};
    const size_t H = (size_t)N / 2;
    const size_t rows = align_up((size_t)sorted_num, kBlockRows);
    const size_t blocks = rows / kBlockRows;
    size_t off = 0;
    l.n_tiles_off = off;
    off += 256;
    l.tiles_off = off;
    off = align_up(off + blocks * sizeof(int2), 256);
    l.work_up_off = off;
    off = align_up(off + align_up(blocks * (H / 128), 8) * sizeof(int4), 256);
    l.work_down_off = off;
    const size_t n_wt_down = ((size_t)K + kWRows - 1) / kWRows;
    off = align_up(off + align_up(blocks * n_wt_down, 8) * sizeof(int4), 256);
    l.inv_off = off;
    const size_t pairs = (size_t)M * (size_t)std::max(top_k, 1);
    off = align_up(off + pairs * sizeof(int32_t), 256);
    l.y_off = off;  // one row per pair id
    off = align_up(off + pairs * K * 2, 256);
    l.act_off = off;
    off = align_up(off + rows * H, 256);
    l.act_scales_off = off;
    off = align_up(off + rows * (H / 32), 256);
    l.xs_tiled_off = off;
    off = align_up(off + rows * ((size_t)K / 32), 256);
    l.total = off;
    return l;
}

static int grid_for(int n_tiles) { return (n_tiles + 7) / 8 * 8; }

// CUs that launches are sized for (0: those of the device); see pmoe_set_compute_units in the header.
static thread_local int g_compute_units = 0;
int resident_grid() {
    static thread_local int cached_dev = -1, cached = 0;
    if (g_compute_units > 0) return g_compute_units;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 256;
    if (dev != cached_dev) {
        int cus = 0;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 8) cus = 256;
        cached = cus / 8 * 8;
        cached_dev = dev;
    }
    return cached;
}

// Which phases of the pipeline the fused entry points enqueue (all by default); see
// pmoe_set_phase_mask in the header.
static thread_local int g_phase_mask = PMOE_PHASE_ALL;
int phase_mask() { return g_phase_mask; }
// Weight tiles a workgroup of the mxfp8 kernels takes in a row (0: chosen per launch); see
// pmoe_set_tiles_per_workgroup in the header.
static thread_local int g_tiles_per_wg = 0;

// A workgroup of the mxfp8 kernels can keep its token rows and take several weight tiles in a row: it
// saves the set-up of all but the first and starts each tile's copies under the epilogue of the one before, as far as
// the ring has stages in front of the epilogue's scratch, but the coarser work balances worse over the
// CUs.  Two tiles when that leaves enough rounds of workgroups
// per CU: 8 for the down kernel, whose tiles are short, 20 for the up kernel (blocks are paired to row tiles, hence
// 16 and 40 in terms of blocks).  Two against one tile, K = N = 2048 on 32 experts, each kernel behind the one in
// front of it: down 123 / 125 us at 12000 tokens (14 blocks x weight tiles per CU), 461 / 518 at 60000, 1027 / 1190 at 131072; up
// 959 / 973 at 60000 tokens (59), 2090 / 2108 at 131072, but 207 / 199 at 12000; DeepSeek-V3-like prefill (down 30, up 17 per CU):
// down 725 / 756, up 1550 / 1533.  Three and four tiles (which need not divide the weight tiles): down 130 and 136 at 12000,
// 464 and 474 at 60000, 1157 and 1112 at 131072, up 995 and 966 at 60000.
static int tiles_per_workgroup(bool down, int n_blocks, int n_wt) {
    if (g_tiles_per_wg > 0) return std::min(g_tiles_per_wg, n_wt);
    return (int64_t)n_blocks * n_wt >= (int64_t)resident_grid() * (down ? 16 : 40) ? std::min(2, n_wt) : 1;
}

void launch_finalize(const MoeArgs &a, void *out, int split, int n_wt_down, hipStream_t s) {
    (void)n_wt_down;
    const int pieces = (a.K + 511) / 512;
    const int64_t waves = (int64_t)a.M * pieces;
    const int blocks = (int)std::min<int64_t>((waves + 3) / 4, 1 << 20);
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(blocks), dim3(256), 0, s, a.y, a.inv, a.sorted_ids, a.ntpp, a.sorted_num,
                           a.topk_w, a.top_k, a.M, a.K, static_cast<char *>(out), a.expert_ids, a.E, pieces);
    };
    if (split) {
        if (a.top_k <= 2) launch(finalize_kernel<false, 2>);
        else launch(finalize_kernel<false, 4>);
    } else {
        if (a.top_k <= 2) launch(finalize_kernel<true, 2>);
        else launch(finalize_kernel<true, 4>);
    }
}

struct SchedBuffers {
    int2 *tiles;
    int *n_tiles;
    int4 *work_up;
    int4 *work_down;
};

// Blocks with work that the host can expect: an expert each, and no more than there are pairs.
static int64_t expected_blocks(const MoeArgs &a) {
    return std::min<int64_t>(a.n_blocks, std::min<int64_t>(a.E, (int64_t)a.M * a.top_k));
}
// Few rows per expert: blocks hardly ever share an expert, so there is nothing to pair and no schedule to build, and
// consecutive workgroups on consecutive weight tiles read one narrow window of the weights.  Whole op with / without
// the prologue and its work lists (256 experts of K 7168 x N 4096, top 8): 290 / 304 us at 5 tokens, 1824 / 1835 at 512
// (16 rows per expert), 1938 / 1922 at 1024; skewed (Zipf) 931 / 951 at 64, 1751 / 1880 at 512.  With few up jobs for
// the chip the streaming up kernel pays longer: 37 experts of K 4096 x N 256, top 9: 53 / 71 us at 128 tokens, 58 / 94
// at 256 (62 rows per expert).
static bool use_direct(const MoeArgs &a) {
    const int64_t rows = expected_blocks(a) * (a.H / 128) < resident_grid() / 2 ? 64 : 24;
    return (int64_t)a.M * a.top_k <= rows * a.E;
}

// The prologue, with work lists for grids of grid_up and grid_down workgroups that take per_up and per_down weight tiles.
static void launch_prologue(const MoeArgs &a, const SchedBuffers &sb, int per_up, int grid_up, int per_down, int grid_down,
                            hipStream_t s) {
    // the work lists are needed by the two kernels even when the rest of the prologue is masked off
    const int do_invert = (g_phase_mask & PMOE_PHASE_PROLOGUE) ? 1 : 0;
    const int blocks = do_invert ? std::max(1, std::min((a.sorted_num + kBlockRows - 1) / kBlockRows, a.crowd ? 48 : 1024)) : 1;
    hipLaunchKernelGGL(a.crowd ? moe_prologue_kernel<true> : moe_prologue_kernel<false>, dim3(blocks), dim3(256), 0, s, a.expert_ids, a.ntpp, a.n_blocks, sb.tiles, sb.n_tiles,
                       sb.work_up, a.H / 128, per_up, grid_up, sb.work_down, (a.K + kWRows - 1) / kWRows, per_down, grid_down, a.E,
                       a.sorted_ids, a.sorted_num, a.inv, a.M * a.top_k, do_invert, a.x_scales, a.xs_tiled, a.K >> 7, a.top_k, a.M,
                       a.crowd);
}

// An expert has at most M rows (more only if a token names it twice, which is not looked for): up to 128 it has one block.
// Crowded blocks hold 96 rows or more on average.
static bool crowding_possible_mx(const MoeArgs &a, int n_cus) {
    const int64_t pairs = (int64_t)a.M * a.top_k;
    return a.M > kBlockRows && crowded_mx(pairs, pairs / 96, a.H / 128, n_cus);
}

static int launch_direct_pipeline(MoeArgs a, const SchedBuffers &sb, void *out, int split, hipStream_t s) {
    const int mask = g_phase_mask, n_cus = resident_grid();
    const int64_t blocks = expected_blocks(a);
    const int n_wt_up = a.H / 128, n_wt_down = (a.K + kWRows - 1) / kWRows;
    // narrow jobs while wide tiles do not give every CU one (us at 128 / 256 / 640 / 1024 wide jobs, stream against
    // ring, whole op: 75.5 / 81.7, 130 / 129, 291 / 290, 419 / 406)
    const bool stream_up = blocks * n_wt_up < n_cus;
    // Narrow jobs while the wide tiles are few and hold a row each, or do not give every CU one and hold a few (stream
    // against ring, whole op, us; 256 experts, K 7168, H 2048: 71.6 / 75.5 at 1 token, 126 / 130 at 2, 288 / 291 at 5, 408 / 406
    // at 8; 8 experts, K 4096, H 14336: 206 / 232 at 4 tokens x top 2, 266 / 295 at 16; 64 experts, K 2048, tokens x top 4: H 384
    // 33.8 / 34.1 at 12, 47.8 / 41.9 at 32, H 1536 75.1 / 82.2, 105 / 105; 128 experts, K 2048, H 768, top 8: 125.9 / 120.1 at 64)
    const int64_t down_jobs = blocks * n_wt_down;
    const bool stream_down = a.H <= 256 || (down_jobs < 5 * n_cus && (int64_t)a.M * a.top_k <= (down_jobs <= n_cus ? 4 : 1) * blocks);
    auto launch_stream = [&](auto kernel, int n_tiles) {
        const int grid = (int)std::min<int64_t>((int64_t)a.n_blocks * std::max(n_tiles, 1), 2 * n_cus);
        if (grid > 0) hipLaunchKernelGGL(kernel, dim3(grid), dim3(512), 0, s, a, n_tiles);
    };
    const int per_up = tiles_per_workgroup(false, (int)blocks, n_wt_up), per_down = tiles_per_workgroup(true, (int)blocks, n_wt_down);
    const int grid_up = grid_for(a.n_blocks * ((n_wt_up + per_up - 1) / per_up));
    const int grid_down = grid_for(a.n_blocks * ((n_wt_down + per_down - 1) / per_down));
    auto launch_ring = [&](auto kernel, const int4 *list, int n_wt, int per_job, int grid) {
        MoeArgs d = a;
        d.work = a.crowd ? list : nullptr;
        d.n_wtiles = n_wt;
        d.per_job = per_job;
        if (grid > 0) hipLaunchKernelGGL(kernel, dim3(grid), dim3(512), 0, s, d);
    };
    if (!stream_up && !stream_down && crowding_possible_mx(a, n_cus)) {
        a.crowd = n_cus;
        launch_prologue(a, sb, per_up, grid_up, per_down, grid_down, s);
    }
    if (mask & PMOE_PHASE_UP) {
        if (stream_up) launch_stream(moe_stream_kernel_mx<true>, a.H / 32);
        else launch_ring(moe_up_kernel<DT_FP8>, sb.work_up, n_wt_up, per_up, grid_up);
    } else if (mask & PMOE_PHASE_PROLOGUE) {
        launch_stream(moe_stream_kernel_mx<true>, 0);
    }
    if (mask & PMOE_PHASE_DOWN) {
        if (a.H <= 256) {
            // (257 experts of K 7168, H 256: 250 against 282 us at 128 tokens; 37 of K 4096, H 128: 23 / 29 at 8)
            const int grid = (int)std::min<int64_t>((int64_t)a.n_blocks * (a.K / 128), 2 * n_cus);
            if (grid > 0) {
                if (a.H == 128) hipLaunchKernelGGL(moe_stream_down_short_kernel_mx<128>, dim3(grid), dim3(256), 0, s, a);
                else hipLaunchKernelGGL(moe_stream_down_short_kernel_mx<256>, dim3(grid), dim3(256), 0, s, a);
            }
        } else if (stream_down) {
            launch_stream(moe_stream_kernel_mx<false>, a.K / 64);
        } else {
            launch_ring(moe_down_kernel<DT_FP8>, sb.work_down, n_wt_down, per_down, grid_down);
        }
    }
    if (mask & PMOE_PHASE_FINALIZE) launch_finalize(a, out, split, n_wt_down, s);
    return check_launch("fused_moe_mxfp8 launch");
}

static int launch_mxfp8_pipeline(MoeArgs a, const SchedBuffers &sb, void *out, int split, hipStream_t s) {
    constexpr int DT = DT_FP8;
    const int mask = g_phase_mask;
    a.n_blocks = (a.sorted_num + kBlockRows - 1) / kBlockRows;
    if (use_direct(a)) return launch_direct_pipeline(a, sb, out, split, s);
    a.n_wtiles = a.H / 128;
    const int n_wt_down = (a.K + kWRows - 1) / kWRows;
    const int per_up = tiles_per_workgroup(false, a.n_blocks, a.n_wtiles);
    const int per_down = tiles_per_workgroup(true, a.n_blocks, n_wt_down);
    const int grid_up = grid_for(a.n_blocks * ((a.n_wtiles + per_up - 1) / per_up));
    const int grid_down = grid_for(a.n_blocks * ((n_wt_down + per_down - 1) / per_down));
    launch_prologue(a, sb, per_up, grid_up, per_down, grid_down, s);
    if (a.n_blocks > 0) {
        a.work = sb.work_up;
        if (mask & PMOE_PHASE_UP) hipLaunchKernelGGL((moe_up_kernel<DT>), dim3(grid_up), dim3(512), 0, s, a);
        MoeArgs d = a;
        d.n_wtiles = n_wt_down;
        d.work = sb.work_down;
        if (mask & PMOE_PHASE_DOWN) hipLaunchKernelGGL((moe_down_kernel<DT>), dim3(grid_down), dim3(512), 0, s, d);
    }
    if (mask & PMOE_PHASE_FINALIZE) launch_finalize(a, out, split, n_wt_down, s);
    return check_launch("fused_moe_mxfp8 launch");
}

}  // namespace pmoe

using namespace pmoe;

extern "C" void pmoe_set_phase_mask(int mask) { g_phase_mask = mask; }
extern "C" void pmoe_set_compute_units(int n) { g_compute_units = n <= 0 ? 0 : std::max(n / 8 * 8, 8); }
extern "C" void pmoe_set_tiles_per_workgroup(int n) { g_tiles_per_wg = n < 0 ? 0 : (n > 16 ? 16 : n); }

extern "C" size_t pmoe_fused_moe_bf16_workspace_bytes(int M, int K, int N, int num_experts,
                                                      int sorted_num, int top_k, int split) {
    (void)split;
    if (M <= 0 || K <= 0 || N <= 0 || sorted_num < 0) return 0;
    MoeArgs a{};
    a.M = M; a.K = K; a.N = N; a.H = N / 2; a.E = num_experts; a.sorted_num = sorted_num; a.top_k = top_k;
    return bf16_workspace(a, nullptr);
}

extern "C" size_t pmoe_fused_moe_mxfp8_workspace_bytes(int M, int K, int N, int num_experts,
                                                       int sorted_num, int top_k, int split) {
    (void)num_experts;
    (void)split;
    if (M <= 0 || K <= 0 || N <= 0 || sorted_num < 0) return 0;
    return workspace_layout(M, K, N, sorted_num, top_k).total;
}

static int check_tuning(const char *op, int block_m, int block_n, int warp_n, int stages,
                        int max_stages) {
    PMOE_REQUIRE((block_n == 64 && warp_n == 4) || (block_n == 32 && warp_n == 8),
                 "%s: (block_n, warp_n) must be (64, 4) or (32, 8), got (%d, %d)", op, block_n, warp_n);
    PMOE_REQUIRE(stages > 0 && stages <= max_stages, "%s supports stages in 1..%d, got %d", op, max_stages, stages);
    PMOE_REQUIRE(block_m == 128, "%s requires block_m=128, got %d", op, block_m);
    return PMOE_OK;
}

extern "C" int pmoe_fused_moe_bf16(const void *x, const void *w, const void *w2, void *out,
                                   const int32_t *sorted_token_ids, const int32_t *expert_idxs,
                                   const int32_t *num_tokens_post_padded, const float *topk_weights,
                                   int top_k, int M, int K, int N, int num_experts, int sorted_num,
                                   int block_m, int block_n, int warp_n, int stages, int bpc, int cpc,
                                   int split, void *workspace, size_t workspace_bytes, void *stream) {
    PMOE_REQUIRE(M > 0, "fused_moe_bf16: x has no rows");
    PMOE_REQUIRE(K > 0 && (K & 127) == 0, "K dimension must be a multiple of 128");
    PMOE_REQUIRE(N > 0 && (N & 255) == 0, "fused_moe_bf16: N must be a multiple of 256, got %d", N);
    if (int rc = check_tuning("fused_moe_bf16", block_m, block_n, warp_n, stages, 5)) return rc;
    PMOE_REQUIRE(bpc == 1 && cpc == 1, "bpc=cpc=1 is the only supported configuration");
    PMOE_REQUIRE(!split || stages <= 4, "split=True requires stages<=4, got stages=%d", stages);
    PMOE_REQUIRE(top_k > 0 && num_experts > 0 && sorted_num >= 0, "fused_moe_bf16: bad top_k / num_experts / sorted_num");
    PMOE_REQUIRE(num_experts <= 1024, "fused_moe_bf16: at most 1024 experts, got %d", num_experts);
    // the gather addresses a token row by a 32-bit byte offset from x
    PMOE_REQUIRE((uint64_t)M * (uint64_t)K * 2u < (1ull << 32), "fused_moe_bf16: x must be smaller than 4 GiB, got %d x %d", M, K);
    PMOE_REQUIRE(x && w && w2 && out && sorted_token_ids && expert_idxs && num_tokens_post_padded && topk_weights,
                 "fused_moe_bf16: null pointer");
    MoeArgs a{};
    a.x = static_cast<const char *>(x);
    a.w1 = static_cast<const char *>(w);
    a.w2 = static_cast<const char *>(w2);
    a.sorted_ids = sorted_token_ids;
    a.expert_ids = expert_idxs;
    a.ntpp = num_tokens_post_padded;
    a.topk_w = topk_weights;
    a.top_k = top_k; a.M = M; a.K = K; a.N = N; a.H = N / 2; a.E = num_experts; a.sorted_num = sorted_num;
    const size_t need = bf16_workspace(a, nullptr);
    PMOE_REQUIRE(workspace && workspace_bytes >= need, "fused_moe_bf16: workspace of %zu bytes needed, got %zu", need, workspace_bytes);
    PMOE_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 255) == 0, "fused_moe_bf16: workspace must be 256-byte aligned");
    bf16_workspace(a, static_cast<char *>(workspace));
    return launch_bf16_pipeline(a, out, split, static_cast<hipStream_t>(stream));
}

extern "C" int pmoe_fused_moe_mxfp8(const void *x, const void *x_scales, const void *w,
                                    const void *w_scales, const void *w2, const void *w2_scales,
                                    void *out, const int32_t *sorted_token_ids,
                                    const int32_t *expert_idxs, const int32_t *num_tokens_post_padded,
                                    const float *topk_weights, int top_k, int M, int K, int N,
                                    int num_experts, int sorted_num, int block_m, int block_n,
                                    int warp_n, int stages, int bpc, int split, void *workspace,
                                    size_t workspace_bytes, void *stream) {
    PMOE_REQUIRE(M > 0, "fused_moe_mxfp8: x has no rows");
    PMOE_REQUIRE(K > 0 && (K & 255) == 0, "K dimension must be a multiple of 256 on the mxfp8 path");
    PMOE_REQUIRE(N > 0 && (N & 255) == 0, "N dimension must be a multiple of 256 on the mxfp8 path");
    if (int rc = check_tuning("fused_moe_mxfp8", block_m, block_n, warp_n, stages, 4)) return rc;
    PMOE_REQUIRE(bpc == 1, "mxfp8 supports bpc=1 only");
    PMOE_REQUIRE(top_k > 0 && num_experts > 0 && sorted_num >= 0, "fused_moe_mxfp8: bad top_k / num_experts / sorted_num");
    PMOE_REQUIRE(num_experts <= 1024, "fused_moe_mxfp8: at most 1024 experts, got %d", num_experts);
    // the gather addresses a token row by a 32-bit byte offset from x
    PMOE_REQUIRE((uint64_t)M * (uint64_t)K < (1ull << 32), "fused_moe_mxfp8: x must be smaller than 4 GiB, got %d x %d", M, K);
    PMOE_REQUIRE(x && x_scales && w && w_scales && w2 && w2_scales && out && sorted_token_ids && expert_idxs &&
                     num_tokens_post_padded && topk_weights,
                 "fused_moe_mxfp8: null pointer");
    const WorkspaceLayout l = workspace_layout(M, K, N, sorted_num, top_k);
    PMOE_REQUIRE(workspace && workspace_bytes >= l.total, "fused_moe_mxfp8: workspace of %zu bytes needed, got %zu", l.total, workspace_bytes);
    PMOE_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 255) == 0, "fused_moe_mxfp8: workspace must be 256-byte aligned");
    MoeArgs a{};
    a.x = static_cast<const char *>(x);
    a.x_scales = static_cast<const uint8_t *>(x_scales);
    a.w1 = static_cast<const char *>(w);
    a.w1_scales = static_cast<const uint8_t *>(w_scales);
    a.w2 = static_cast<const char *>(w2);
    a.w2_scales = static_cast<const uint8_t *>(w2_scales);
    a.sorted_ids = sorted_token_ids;
    a.expert_ids = expert_idxs;
    a.ntpp = num_tokens_post_padded;
    a.topk_w = topk_weights;
    char *ws = static_cast<char *>(workspace);
    a.y = ws + l.y_off;
    a.inv = reinterpret_cast<int32_t *>(ws + l.inv_off);
    a.act = ws + l.act_off;
    a.act_scales = reinterpret_cast<uint32_t *>(ws + l.act_scales_off);
    a.xs_tiled = reinterpret_cast<uint32_t *>(ws + l.xs_tiled_off);
    a.top_k = top_k; a.M = M; a.K = K; a.N = N; a.H = N / 2; a.E = num_experts; a.sorted_num = sorted_num;
    SchedBuffers sb;
    sb.n_tiles = reinterpret_cast<int *>(ws + l.n_tiles_off);
    sb.tiles = reinterpret_cast<int2 *>(ws + l.tiles_off);
    sb.work_up = reinterpret_cast<int4 *>(ws + l.work_up_off);
    sb.work_down = reinterpret_cast<int4 *>(ws + l.work_down_off);
    return launch_mxfp8_pipeline(a, sb, out, split, static_cast<hipStream_t>(stream));
}

// Weight-streaming mxfp8 kernels for few rows per expert (decode batches), gfx950: the counterpart of moe_stream.h.
//
// Same jobs, ring and bound; what differs is the arithmetic.  A slab is 256 B = 256 elements per row = four 64-wide
// steps of v_mfma_scale_f32_32x32x64_f8f6f4.  A job always has two units of 32 weight rows: in the up kernel they
// give 32 activation columns, one MX block, whose scale then is a matter of one workgroup.  Wave v works on unit
// v / 4 and step v % 4 of every slab.  The 4-scale dwords (128 elements of a row) ride along in the stage: the weight
// scales from their blocked layout, the token scales row major from x_scales (up) or from the tiled ones the up
// kernel leaves (down); no prologue re-tiles anything.
//
// H may be an odd multiple of 128: the last slab of the down kernel then has only its first half.
#pragma once
#include "moe_stream.h"

namespace pmoe {
namespace stream {

constexpr int kMxScaleBytes = (kPassRows + 64) * 2 * 4;  // of a stage: token rows, weight rows; two dwords each
static_assert(kMxScaleBytes % 1024 == 0, "stages stay 1 KB aligned");

struct MxLoader {
    const char *w_base[2];  // wave-uniform: first of the wave's rows of unit u
    const char *tok_base;   // wave-uniform
    const char *sc_base;    // wave-uniform
    uint32_t w_off, tok_off[2], chunk;
    uint32_t sc_off;        // this lane's scale dword
    uint32_t sc_step;       // bytes from one slab's to the next's
    bool sc_second;         // this lane's dword is the slab's second K tile's
    int sc_dst;             // where this wave's scale dwords go in a stage's scale region, -1: it copies none
    bool sc_live;
    bool tok_live[2];
    bool tok_any[2];
    int lps;
    bool w_once;

    // `left`: bytes of a row from this slab on (256, or 128 at the end of an odd row)
    __device__ __forceinline__ void issue(char *stage, int tok_bytes, int wave, int slab, uint32_t left) const {
        const uint32_t koff = (uint32_t)slab * kRB;
        const bool in = chunk < left;  // this lane's chunk lies inside the row
        char *w = stage + tok_bytes + 4 * wave * kRB;
        if (in) {
#pragma unroll
            for (int q = 0; q < 2; ++q)
                if (tok_any[q]) {
                    if (tok_live[q]) ring::copy16(tok_base, tok_off[q] + koff, stage + (32 * q + 4 * wave) * kRB);
                }
            if (w_once) {
#pragma unroll
                for (int u = 0; u < 2; ++u) ring::copy16_once(w_base[u], w_off + koff, w + u * kUnitBytes);
            } else {
#pragma unroll
                for (int u = 0; u < 2; ++u) ring::copy16(w_base[u], w_off + koff, w + u * kUnitBytes);
            }
        }
        if (sc_dst >= 0) {
            // (half a slab has no second K tile: its lanes fetch the first one's dword, 512 bytes before)
            const uint32_t back = sc_second && left <= 128 ? 512u : 0u;
            if (sc_live) ring::copy4(sc_base, sc_off + (uint32_t)slab * sc_step - back, stage + tok_bytes + 2 * kUnitBytes + sc_dst);
        }
    }
};

// One pass over the contraction: acc[t] += the wave's unit x token fragment t, for the wave's steps.
template <int NF>
__device__ __forceinline__ void mx_k_loop(f32x16 (&acc)[NF], const MxLoader &ld, char *ring_lds, int tok_bytes,
                                          int row_bytes, int wave, int lane, int start) {
    const int stage_bytes = tok_bytes + 2 * kUnitBytes + kMxScaleBytes;
    const int ns = min(kMaxStages, kRing / stage_bytes);
    const int n_slabs = (row_bytes + kRB - 1) / kRB;
    const int r = lane & 31, half = lane >> 5, step = wave & 3;
    const int off = r * kRB + (((4 * step + half) ^ (r & 15)) << 4);  // first 16 bytes of the lane's K block 0; block 1: ^ 32
    const int sel = 8 * (2 * (step & 1) + half);                      // its scale's byte in the row's dword
    const int w_at = tok_bytes + (wave >> 2) * kUnitBytes, sc_at = tok_bytes + 2 * kUnitBytes;
    const int w_sc_at = sc_at + kPassRows * 8 + ((wave >> 2) * 64 + (step >> 1) * 32 + r) * 4;
    const int t_sc_at = sc_at + ((step >> 1) * kPassRows + r) * 4;
    int slab = start;  // next slab to issue (rotated order)
    auto issue_next = [&](int stage) {
        ld.issue(ring_lds + stage * stage_bytes, tok_bytes, wave, slab, (uint32_t)(row_bytes - slab * kRB));
        if (++slab == n_slabs) slab = 0;
    };
    for (int s = 0; s < ns - 1 && s < n_slabs; ++s) issue_next(s);
    int cur = 0, kt_slab = start;
    for (int kt = 0; kt < n_slabs; ++kt) {
        ring::wait_and_barrier_dyn(ld.lps * min(ns - 2, n_slabs - 1 - kt));
        if (kt + ns - 1 < n_slabs) issue_next(cur == 0 ? ns - 1 : cur - 1);
        if (64 * step < row_bytes - kt_slab * kRB) {
            const char *st = ring_lds + cur * stage_bytes;
            auto frag = [&](const char *p) {
                const i32x4 lo = *reinterpret_cast<const i32x4 *>(p + off);
                const i32x4 hi = *reinterpret_cast<const i32x4 *>(p + (off ^ 32));
                return i32x8{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
            };
            const i32x8 w = frag(st + w_at);
            const int ws = (int)((*reinterpret_cast<const uint32_t *>(st + w_sc_at) >> sel) & 0xffu);
#pragma unroll
            for (int t = 0; t < NF; ++t) {
                const i32x8 b = frag(st + t * kUnitBytes);
                const int bs = (int)((*reinterpret_cast<const uint32_t *>(st + t_sc_at + t * 128) >> sel) & 0xffu);
                acc[t] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w, b, acc[t], 0, 0, 0, ws, 0, bs);
            }
        }
        if (++cur == ns) cur = 0;
        if (++kt_slab == n_slabs) kt_slab = 0;
    }
    __syncthreads();  // every stage has been read: the ring is scratch now
}

// Sum of the four partial sums of unit u (waves 4 u .. 4 u + 3), registers 4 i4 .. of lane `lane`.
__device__ __forceinline__ float4 mx_sum(const char *scratch, int u, int i4, int lane) {
    const float4 *src = reinterpret_cast<const float4 *>(scratch) + u * 1024 + 64 * i4 + lane;
    float4 s = src[0];
#pragma unroll
    for (int w = 1; w < 4; ++w) {
        const float4 v = src[w * 256];
        s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
    return s;
}

template <int NF, typename Finish>
__device__ __forceinline__ void mx_run_pass(const MxLoader &ld, char *ring_lds, int n, int row_bytes, int wave, int lane,
                                            int start, Finish finish) {
    f32x16 acc[NF];
#pragma unroll
    for (int t = 0; t < NF; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[t][i] = 0.f;
    mx_k_loop<NF>(acc, ld, ring_lds, ((n + 3) & ~3) * kRB, row_bytes, wave, lane, start);
    float4 *mine = reinterpret_cast<float4 *>(ring_lds) + wave * 256 + lane;
#pragma unroll
    for (int t = 0; t < NF; ++t) {
        if (t > 0) __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; ++i) mine[64 * i] = make_float4(acc[t][4 * i], acc[t][4 * i + 1], acc[t][4 * i + 2], acc[t][4 * i + 3]);
        __syncthreads();
        finish(t);
    }
    __syncthreads();  // the ring may be filled again
}

// One job, as in moe_stream.h with two units: act[rows, 32 columns] and its MX scale, or y[pair, 64 columns].
template <bool UP>
__device__ __forceinline__ void mx_run_job(const MoeArgs &a, Shared &sh, int blk, int e, int tile, int id) {
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

    MxLoader ld;
    const uint32_t row_bytes = (uint32_t)(UP ? K : H);
    const int sub = lane >> 4;  // row of the lane inside an instruction
    ld.chunk = (uint32_t)((lane & 15) ^ ((4 * wave + sub) & 15)) * 16u;
    ld.w_off = (uint32_t)sub * row_bytes + ld.chunk;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        int64_t row;
        if (UP) row = (int64_t)e * a.N + (wave >= 4 ? H : 0) + (tile * 2 + u) * 16 + 4 * (wave & 3);
        else row = (int64_t)e * K + (tile * 2 + u) * 32 + 4 * wave;
        ld.w_base[u] = ring::uniform_ptr((UP ? a.w1 : a.w2) + row * row_bytes);
    }
    ld.tok_base = ring::uniform_ptr(UP ? a.x : a.act + (int64_t)blk * kBlockRows * row_bytes);
    ld.w_once = n_rows <= kPassRows;
    const int n_slabs = (int)((row_bytes + kRB - 1) / kRB), n_kt = (int)(row_bytes >> 7);
    const int start = (blk + tile) % n_slabs;

    for (int row0 = 0; row0 < n_rows; row0 += kPassRows) {
        const int n = min(kPassRows, n_rows - row0);
        ld.lps = 2;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int row = 32 * q + 4 * wave + sub;
            const int p = row < n ? sh.pair[row0 + row] : -1;
            ld.tok_live[q] = p >= 0;
            ld.tok_off[q] = (UP ? (uint32_t)max(p, 0) / (uint32_t)a.top_k : (uint32_t)(row0 + row)) * row_bytes + ld.chunk;
            ld.tok_any[q] = __ballot(p >= 0) != 0;
            ld.lps += ld.tok_any[q] ? 1 : 0;
        }
        // scales: waves 0, 1 the token rows' (K tile 0 / 1 of the slab), waves 2, 3 the rows' of weight unit 0 / 1
        ld.sc_dst = -1;
        ld.sc_live = false;
        ld.sc_second = wave < 2 ? wave == 1 : lane >= 32;
        ld.sc_base = nullptr;
        ld.sc_off = ld.sc_step = 0;
        if (wave < 2) {
            const int p = lane < n ? sh.pair[row0 + lane] : -1;
            ld.sc_live = p >= 0;
            if (UP) {
                ld.sc_base = reinterpret_cast<const char *>(a.x_scales);
                ld.sc_off = ((uint32_t)max(p, 0) / (uint32_t)a.top_k) * (row_bytes / 32) + wave * 4;
                ld.sc_step = 8;
            } else {
                ld.sc_base = reinterpret_cast<const char *>(a.act_scales + (int64_t)blk * n_kt * kBlockRows);
                ld.sc_off = (uint32_t)((wave * kBlockRows + row0 + lane) * 4);
                ld.sc_step = 2 * kBlockRows * 4;
            }
            ld.sc_dst = wave * kPassRows * 4;
        } else if (wave < 4) {
            const int u = wave - 2, i = lane & 31;
            const int row = UP ? (i < 16 ? 0 : H) + (tile * 2 + u) * 16 + (i & 15) : (tile * 2 + u) * 32 + i;
            ld.sc_base = reinterpret_cast<const char *>(UP ? a.w1_scales + (int64_t)e * a.N * (K >> 5) : a.w2_scales + (int64_t)e * K * (H >> 5));
            ld.sc_off = (uint32_t)blocked_scale_off(row, lane >> 5, n_kt);
            ld.sc_step = 1024;
            ld.sc_live = true;
            ld.sc_dst = kPassRows * 8 + u * 256;
        }
        ld.sc_base = ring::uniform_ptr(ld.sc_base);
        if (ld.sc_dst >= 0 && __ballot(ld.sc_live) == 0) ld.sc_dst = -1;
        ld.lps += ld.sc_dst >= 0 ? 1 : 0;
        auto finish = [&](int t) {
            if (UP) {
                // one wave: lane (row, half) takes 16 of the row's 32 columns, its partner (lane ^ 32) the others
                if (wave == 0) {
                    const int row = row0 + 32 * t + (lane & 31);
                    const int p = row < row0 + n ? sh.pair[row] : -1;
                    float v[2][2][4], amax = 0.f;
#pragma unroll
                    for (int u = 0; u < 2; ++u)
#pragma unroll
                        for (int q = 0; q < 2; ++q) {
                            const float4 g = mx_sum(sh.ring, u, q, lane), up = mx_sum(sh.ring, u, q + 2, lane);
                            v[u][q][0] = swiglu(g.x, up.x);
                            v[u][q][1] = swiglu(g.y, up.y);
                            v[u][q][2] = swiglu(g.z, up.z);
                            v[u][q][3] = swiglu(g.w, up.w);
#pragma unroll
                            for (int i = 0; i < 4; ++i) amax = fmaxf(amax, fabsf(v[u][q][i]));
                        }
                    amax = fmaxf(amax, __shfl_xor(amax, 32, 64));
                    uint32_t e8;
                    float inv;
                    mx_block_scale(amax, e8, inv);
                    if (p >= 0) {
                        char *dst = a.act + ((int64_t)blk * kBlockRows + row) * H + tile * 32 + 4 * (lane >> 5);
#pragma unroll
                        for (int u = 0; u < 2; ++u)
#pragma unroll
                            for (int q = 0; q < 2; ++q)
                                *reinterpret_cast<uint32_t *>(dst + 16 * u + 8 * q) =
                                    pack4_e4m3(v[u][q][0], v[u][q][1], v[u][q][2], v[u][q][3], inv);
                        if (lane < 32)
                            reinterpret_cast<uint8_t *>(a.act_scales)[(((int64_t)blk * (H >> 7) + (tile >> 2)) * kBlockRows + row) * 4 + (tile & 3)] = (uint8_t)e8;
                    }
                }
            } else {
                const int u = tid >> 8, q = (tid >> 6) & 3;
                const int row = row0 + 32 * t + (lane & 31);
                const int p = row < row0 + n ? sh.pair[row] : -1;
                const float4 v = mx_sum(sh.ring, u, q, lane);
                uint2 pk;
                pk.x = pack2_bf16(v.x, v.y);
                pk.y = pack2_bf16(v.z, v.w);
                const int col = (tile * 2 + u) * 32 + 8 * q + 4 * (lane >> 5);
                if (p >= 0) *reinterpret_cast<uint2 *>(a.y + ((int64_t)p * K + col) * 2) = pk;
            }
        };
        if (n <= 32) mx_run_pass<1>(ld, sh.ring, n, (int)row_bytes, wave, lane, start, finish);
        else mx_run_pass<2>(ld, sh.ring, n, (int)row_bytes, wave, lane, start, finish);
    }
    __syncthreads();  // the table may be written again
}

// mxfp8, RB = H = 128 or 256 bytes per row; a turn is 4 or 2 units of 32 weight rows (16 contiguous KB), their 4-scale
// dwords go straight into registers.
template <int RB>
struct ShortDownMx {
    static constexpr int kUnits = 16384 / (32 * RB);
    static constexpr int kSteps = RB / 64;   // 64-wide steps of the contraction
    static constexpr int kTiles = RB / 128;  // 128-wide scale tiles
    static constexpr int kChunks = RB / 16;
    static constexpr int kBytes = 16384;
    static constexpr int kTurnCols = 32 * kUnits;
    static __device__ __forceinline__ int swz(int row) { return RB == 128 ? (row >> 1) & 7 : row & 15; }

    const MoeArgs &a;
    char *buf;
    i32x8 w[kUnits][kSteps], b[kSteps] = {};
    uint32_t w_sc[kTiles][kUnits], w_sc_next[kTiles][kUnits], b_sc[kTiles] = {};

    __device__ __forceinline__ ShortDownMx(const MoeArgs &args, char *lds) : a(args), buf(lds) {}
    __device__ __forceinline__ void load_tokens(i32x8 (&dst)[kSteps], uint32_t (&sc)[kTiles], int blk, int row0, int pair) const {
        const int lane = threadIdx.x & 63, row = row0 + (lane & 31);
        if ((unsigned)pair >= (unsigned)(a.M * a.top_k)) return;  // (as in ShortDown)
        const char *tok = a.act + ((int64_t)blk * kBlockRows + row) * RB + (lane >> 5) * 16;
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
            const i32x4 lo = *reinterpret_cast<const i32x4 *>(tok + 64 * s), hi = *reinterpret_cast<const i32x4 *>(tok + 64 * s + 32);
            dst[s] = i32x8{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        }
#pragma unroll
        for (int kt = 0; kt < kTiles; ++kt) sc[kt] = a.act_scales[((int64_t)blk * kTiles + kt) * kBlockRows + row];
    }
    __device__ __forceinline__ void request(int e, int turn) {
        const int lane = threadIdx.x & 63, sub = lane / kChunks;
        const uint32_t lane_off = (uint32_t)sub * RB + (uint32_t)((lane % kChunks) ^ swz(sub)) * 16u;
        const int row = turn * kTurnCols;
        const char *src = ring::uniform_ptr(a.w2 + ((int64_t)e * a.K + row) * RB);
#pragma unroll
        for (int i = 0; i < 16; ++i)
            ring::copy16_once(src, (lane_off ^ (uint32_t)(swz(i * (1024 / RB)) << 4)) + i * 1024u, buf + i * 1024);
#pragma unroll
        for (int kt = 0; kt < kTiles; ++kt) {
            const uint32_t *sc = reinterpret_cast<const uint32_t *>(
                a.w2_scales + (int64_t)e * a.K * (RB / 32) + blocked_scale_off(row + (lane & 31), kt, kTiles));
#pragma unroll
            for (int g = 0; g < kUnits; ++g) w_sc_next[kt][g] = sc[g];
        }
    }
    __device__ __forceinline__ void request_tokens(int blk, int pair) { load_tokens(b, b_sc, blk, 0, pair); }
    __device__ __forceinline__ void wait() {
        const int lane = threadIdx.x & 63, r = lane & 31, half = lane >> 5;
        asm volatile("s_waitcnt vmcnt(0)" : : : "memory");  // the turn has landed
        // (taken over here: the compiler's wait for these, placed behind the next copies, would wait for those too)
#pragma unroll
        for (int kt = 0; kt < kTiles; ++kt) {
#pragma unroll
            for (int g = 0; g < kUnits; ++g) {
                w_sc[kt][g] = w_sc_next[kt][g];
                asm volatile("" : "+v"(w_sc[kt][g]));
            }
            asm volatile("" : "+v"(b_sc[kt]));
        }
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
            asm volatile("" : "+v"(b[s]));
#pragma unroll
            for (int g = 0; g < kUnits; ++g) {
                const char *row = buf + (32 * g + r) * RB;
                const i32x4 lo = *reinterpret_cast<const i32x4 *>(row + (((4 * s + half) ^ swz(r)) << 4));
                const i32x4 hi = *reinterpret_cast<const i32x4 *>(row + (((4 * s + 2 + half) ^ swz(r)) << 4));
                w[g][s] = i32x8{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");  // it is in registers: the buffer may be filled again
    }
    __device__ __forceinline__ void compute(int blk, int turn, int id0, int id1, int n_rows) {
        const int lane = threadIdx.x & 63, r = lane & 31, half = lane >> 5;
        int p = __shfl(id0, r, 64);
        for (int row0 = 0;;) {
            const bool live = (unsigned)p < (unsigned)(a.M * a.top_k);
            char *dst = a.y + ((int64_t)(live ? p : 0) * a.K + kTurnCols * turn + 4 * half) * 2;
#pragma unroll
            for (int g = 0; g < kUnits; ++g) {
                f32x16 acc;
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
                for (int s = 0; s < kSteps; ++s) {
                    const int sel = 8 * (2 * (s & 1) + half);
                    acc = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w[g][s], b[s], acc, 0, 0, 0,
                                                                          (int)((w_sc[s >> 1][g] >> sel) & 0xffu), 0,
                                                                          (int)((b_sc[s >> 1] >> sel) & 0xffu));
                }
                asm volatile("" : "+v"(acc));  // (kept out of the branch: every lane's scale takes part)
                if (live) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        uint2 pk;
                        pk.x = pack2_bf16(acc[4 * q], acc[4 * q + 1]);
                        pk.y = pack2_bf16(acc[4 * q + 2], acc[4 * q + 3]);
                        *reinterpret_cast<uint2 *>(dst + (32 * g + 8 * q) * 2) = pk;
                    }
                }
            }
            row0 += 32;
            if (row0 >= n_rows) break;
            p = __shfl(row0 < 64 ? id0 : id1, (row0 & 32) + r, 64);
            load_tokens(b, b_sc, blk, row0, p);
        }
    }
};

}  // namespace stream
}  // namespace pmoe

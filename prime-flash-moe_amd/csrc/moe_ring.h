// Stage-ring engine of the mxfp8 grouped-GEMM kernels (512 threads), gfx950, and the copy primitives that the
// bf16 engine (moe_tall.h) shares with it.
//
// Tile: token rows x 256 weight rows.  The contraction is consumed in slabs of RB = 128 bytes per row: whole cache
// lines (with 64-byte slabs and twice the stages the decode shape ran 32 %, the DeepSeek-like prefill 40 % slower).
// Slabs are copied global -> LDS by the direct-to-LDS path (global_load_lds_*: no staging registers, no ds_write)
// into a ring of stages.  Two barriers per slab: one opens a slab that has landed, one gives its stage back as soon as
// every wave holds the slab's remaining operands in registers, so that up to all stages are in flight while the last
// third of the matrix instructions of a slab runs (see main_loop).
//
// The ring is sized per tile.  A stage holds only the token rows up to a group's last live one (group 0's first,
// then group 1's, each rounded up to the 8 rows of a copy instruction), the 256 weight rows and the scale dwords of
// both; as many stages as fit the LDS budget are used, at most 8.  The fewer token rows a tile has, the
// closer it is to a pure stream of weights from HBM, and what keeps HBM busy then is weight bytes in
// flight per CU.  (Rounded up to whole 32-row fragments, tiles of 129 to 160 rows had two stages instead of three: with
// 128 rows per expert on average that is every second expert.)
//
// Stage layout: [token rows][RB] [256 weight rows][RB] [scale dwords: token rows, weight rows].  Operand reads of a group's
// last fragment run past its rows into what lies behind them, which only reaches output rows nobody reads.
// A row is RB/16 chunks of 16 B; chunk c of row r sits in slot c ^ swizzle(r), swizzle(r) = (r >> 1) & 7: the 16-byte MFMA operand reads of 16 consecutive rows then cover all 64 LDS
// banks exactly once.  The copy engine writes lane l of a wave instruction to bytes [16 l, 16 l + 16)
// behind a wave-uniform base (one instruction = 1 KB = 1024 / RB rows), so the swizzle is applied on
// the global side (the lane landing in slot s of row r fetches chunk s ^ swizzle(r)).
//
// mxfp8 scales ride along: the 4-scale dword (128 K) of every row of the tile is copied with each
// slab into the stage's scale region, 4 bytes per lane.
//
// All copies are issued as inline assembly: the compiler cannot tell the stage being read from
// the stages being filled and would otherwise make every LDS read wait for all copies in
// flight.  The hardware load counter (vmcnt) still counts them, per wave and in issue order; a
// wave that issues `lps` copy instructions per stage has slab k when at most lps * (stages still
// behind it) of its copies are pending.
#pragma once
#include "moe_tile.h"

namespace pmoe {
namespace ring {

constexpr int kMaxStages = 8;

constexpr int kRB = 128;  // row bytes of a slab
template <int RB>
__device__ __forceinline__ int swz(int row) {
    static_assert(RB == 128, "the swizzle of 128-byte rows");
    return (row >> 1) & 7;
}

// Geometry of a tile's ring; every member is wave-uniform.
struct Layout {
    int rows0;        // token rows of group 0 in a stage, a multiple of 8
    int tok_rows;     // of both groups
    int group1_off;   // byte offset of group 1's token rows inside a stage
    int w_off;        // byte offset of the weight rows
    int scale_off;    // byte offset of the scale dwords (mxfp8)
    int stage_bytes;
    int stages;
};
// rows0, rows1: 1 + index of each group's last live row.
template <int DT, int RB>
__device__ __forceinline__ Layout make_layout(int rows0, int rows1, int budget) {
    Layout l;
    l.rows0 = (rows0 + 7) & ~7;
    l.tok_rows = l.rows0 + ((rows1 + 7) & ~7);
    l.group1_off = l.rows0 * RB;
    l.w_off = l.tok_rows * RB;
    l.scale_off = l.w_off + kWRows * RB;
    const int bytes = l.scale_off + (DT == DT_FP8 ? (l.tok_rows + kWRows) * 4 : 0);
    l.stage_bytes = (bytes + 255) & ~255;
    l.stages = min(kMaxStages, budget / l.stage_bytes);
    return l;
}
// LDS the ring may use, a multiple of 256 bytes (the kernels put their row table behind it).  Three stages hold up to 152
// token rows.
template <int DT>
constexpr int ring_bytes() {
    static_assert(DT == DT_FP8, "the stage ring serves the mxfp8 kernels");
    return 160 * 1024 - 1280;
}

__device__ __forceinline__ uint32_t lds_addr(const char *p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char *)p;
}
// M0 holds the LDS address of a direct-to-LDS copy.  The statements below write it without declaring it: the
// compiler reserves the register and rejects it in a clobber list.  That is sound only while the compiler itself
// keeps no value in M0 across a statement, so the kernels that use these primitives stay clear of everything that
// makes it use M0 on gfx950: the LDS-DMA builtins (__builtin_amdgcn_global_load_lds, raw_buffer_load_lds), GWS
// and s_sendmsg builtins, register-indexed moves (accumulators and fragment arrays are indexed by constants after
// unrolling only), readlane / writelane with a lane number that is not a compile-time constant.  A host test
// compiles the two translation units that include this file to assembly and fails if a kernel that contains a
// copy touches M0 anywhere outside these statements (tests/test_host.py); a GPU test runs the tile paths with the
// most copies between two barriers on poisoned LDS (tests/test_gpu_lds_copies.py).
__device__ __forceinline__ void copy16(const char *base, uint32_t voff, const char *lds_dst) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(base), "s"(lds_addr(lds_dst)) : "memory");
}
// The same copy with the non-temporal hint, for weight rows that no other workgroup reads (an expert with a
// single row tile): the lines leave the caches first.  The decode shape streams its weights 12 % faster
// with it; weight rows that several row tiles share lose up to 20 % with it.
__device__ __forceinline__ void copy16_once(const char *base, uint32_t voff, const char *lds_dst) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1 nt" : : "v"(voff), "s"(base), "s"(lds_addr(lds_dst)) : "memory");
}
__device__ __forceinline__ void copy4(const char *base, uint32_t voff, const char *lds_dst) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dword %0, %1" : : "v"(voff), "s"(base), "s"(lds_addr(lds_dst)) : "memory");
}
// A wave-uniform pointer, read through lane 0 so that the compiler keeps it in scalar registers.
__device__ __forceinline__ const char *uniform_ptr(const char *p) {
    const uint64_t v = (uint64_t)(uintptr_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (const char *)(uintptr_t)(((uint64_t)hi << 32) | lo);
}
template <int N>
__device__ __forceinline__ void wait_and_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(N) : "memory");
}
// This wave's LDS reads have returned; joins the workgroup barrier.
__device__ __forceinline__ void all_read() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory"); }
// Waits until at most `n` (wave-uniform, <= 30) of this wave's copies are in flight and its LDS
// reads have returned, then joins the workgroup barrier.  The wait count is an immediate of the
// instruction, hence the switch (at most 9 copies per stage x 3 stages behind the current one).
__device__ __forceinline__ void wait_and_barrier_dyn(int n) {
    switch (n) {
#define PMOE_WB(k) case k: wait_and_barrier<k>(); break;
        PMOE_WB(1) PMOE_WB(2) PMOE_WB(3) PMOE_WB(4) PMOE_WB(5) PMOE_WB(6) PMOE_WB(7) PMOE_WB(8) PMOE_WB(9)
        PMOE_WB(10) PMOE_WB(11) PMOE_WB(12) PMOE_WB(13) PMOE_WB(14) PMOE_WB(15) PMOE_WB(16) PMOE_WB(17)
        PMOE_WB(18) PMOE_WB(19) PMOE_WB(20) PMOE_WB(21) PMOE_WB(22) PMOE_WB(23) PMOE_WB(24) PMOE_WB(25)
        PMOE_WB(26) PMOE_WB(27) PMOE_WB(28) PMOE_WB(29) PMOE_WB(30)
#undef PMOE_WB
        default: wait_and_barrier<0>(); break;
    }
}

// Per-thread description of the copies of one stage.  A 128-row block of token rows or half of the
// weight tile takes N = RB / 64 instructions of every wave: instruction q of wave w moves rows
// q * 8 * rpc + rpc * w .. + rpc - 1 of it (rpc = 1024 / RB rows per instruction).  Token rows behind the last
// live one are not copied, nor are rows without a token in front of it
// (an instruction whose rows all lack one is dropped: the wait counts rely on every issued
// instruction having an active lane).  Scales: at most one 4-byte-per-lane instruction per
// wave.
template <int RB>
struct Loader {
    static constexpr int N = RB / 64;
    static constexpr int kRowsPerCopy = 1024 / RB;
    const char *tok_base;
    const char *w_base[2];
    uint32_t tok_off[2][N];
    uint32_t w_off[N];
    const char *sc_base;  // wave-uniform: activation scales or weight scales
    uint32_t sc_off;      // this lane's row in them
    uint32_t sc_step;     // bytes between consecutive 128-wide K tiles: 4 (row major) or 512 (blocked)
    bool sc_live;         // this lane has a row
    int tok_dst[2][N];    // LDS offset inside a stage of this wave's token rows; -1: nothing to copy
    bool tok_live[2][N];  // this lane's row holds a token (rows without one are not fetched: what the
                          // stage holds for them only reaches their own, unused, output rows)
    int w_dst[2][N];      // LDS offsets of this wave's weight rows
    int sc_dst;           // LDS offset of this wave's scale dwords; -1: none
    int lps;              // copy instructions this wave issues per stage
    bool w_once;          // wave-uniform: the weight rows are read by this workgroup only (see copy16_once)

    // Row inside a 128-row block that lane `lane` of wave `wave` moves with instruction q.
    static __device__ __forceinline__ int row_of(int wave, int lane, int q) {
        return q * 8 * kRowsPerCopy + kRowsPerCopy * wave + lane / (RB / 16);
    }
    // The base pointers feed scalar operands of the copy instructions: pin them to scalar registers.
    __device__ __forceinline__ void make_uniform() {
        tok_base = uniform_ptr(tok_base);
        w_base[0] = uniform_ptr(w_base[0]);
        w_base[1] = uniform_ptr(w_base[1]);
        sc_base = uniform_ptr(sc_base);
    }
    // Copy c (a constant once the caller's loop is unrolled) of this wave's share of a stage: kWPieces of weight rows,
    // which every wave issues, then the token rows, then the scales.
    static constexpr int kWPieces = 2 * N, kPieces = 4 * N + 1;
    __device__ __forceinline__ void issue_piece(int c, char *stage, int slab) const {
        const uint32_t koff = (uint32_t)slab * RB;
        const int b = (c / N) & 1, q = c % N;
        if (c < kWPieces) {
            if (w_once) copy16_once(w_base[b] + koff, w_off[q], stage + w_dst[b][q]);
            else copy16(w_base[b] + koff, w_off[q], stage + w_dst[b][q]);
        } else if (c < 2 * kWPieces) {
            if (tok_dst[b][q] >= 0) {
                if (tok_live[b][q]) copy16(tok_base + koff, tok_off[b][q], stage + tok_dst[b][q]);
            }
        } else if (sc_dst >= 0) {
            if (sc_live) copy4(sc_base + (uint32_t)slab * sc_step, sc_off, stage + sc_dst);
        }
    }
    __device__ __forceinline__ void issue(char *stage, int slab) const {
#pragma unroll
        for (int c = 0; c < kPieces; ++c) issue_piece(c, stage, slab);
    }
};

// Operands of one 64-wide K step of a wave: weight fragments a[f], token fragments b[t], and for the slab the step
// belongs to the scale dwords of their rows (4 scales = 128 contraction elements).
//
// One v_mfma_scale_f32_32x32x64_f8f6f4 per (weight fragment, token fragment) and step.  Registers 0-3 of both lane
// halves form K block 0 of the step (lanes < 32 its first 16 bytes, lanes >= 32 the last 16), registers 4-7 K block
// 1; the scale of block 0 is taken from lanes < 32 and that of block 1 from lanes >= 32 (measured on gfx950).  So a
// lane's scale byte in step j is byte 2 j + lane / 32 of its dword: shifted right by 8 (lane / 32) once per slab, the
// instruction picks byte 2 j itself.
template <int NTF>
struct Operands {
    i32x8 a[2], b[NTF];
    int sa[2], sb[NTF];
};
__device__ __forceinline__ i32x8 lds_frag(const char *p, int off) {
    const i32x4 lo = *reinterpret_cast<const i32x4 *>(p + off);
    const i32x4 hi = *reinterpret_cast<const i32x4 *>(p + (off ^ 32));
    return i32x8{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
}
// Nothing crosses this point in the instruction schedule: the order written is the order issued.
#define PMOE_RING_FENCE() __builtin_amdgcn_sched_barrier(0)

// Matrix instructions of weight fragment F with token fragment t in step J.
template <int NTF, int J, int F>
__device__ __forceinline__ void mma(f32x16 (&acc)[2][4], const Operands<NTF> &o, int t) {
    acc[F][t] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(o.a[F], o.b[t], acc[F][t], 0, 0, 2 * J, o.sa[F], 2 * J, o.sb[t]);
    asm volatile("" : "+v"(acc[F][t]));  // stays here: the compiler would sink it past the copies and keep its operands
}

// Issues slabs 0 .. n - 1 of a tile (at most as many as there are stages, in rotated order from `start`) into
// stages 0, 1, ...
template <int DT, int RB>
__device__ __forceinline__ void pre_issue(const Loader<RB> &ld, const Layout &lay, char *lds, int n_slabs, int start,
                                          int n) {
    const int SB = lay.stage_bytes;
    for (int s = 0; s < n; ++s) {
        if (s >= n_slabs) break;
        int slab = s + start;
        if (slab >= n_slabs) slab -= n_slabs;
        ld.issue(lds + s * SB, slab);
    }
}
// K loop of a group with NTF live fragments.  NTF = 0 is the loop of the waves without matrix work (a group without live
// rows): they only issue their share of the copies and join the barriers, which are the same ones for every
// NTF: the two groups of a tile need not have the same number.  `tok_region` = byte
// offset of this wave's group inside a stage's token rows.
//
// The slabs are visited in rotated order, starting at slab `start`: workgroups
// that run side by side and share rows then ask for different cache lines at any one time instead
// of queueing on the same ones.  The sum over K does not depend on the order.
//
// Geometry and wait counts are wave-uniform run-time values (the wait count goes through a switch).
//
// A slab's stage is given back (second barrier) before its matrix instructions are done.  NTF <= 2: all operands of a
// slab are read first.  NTF = 3 and 4 have registers for one 64-wide step: the operands of step 1 replace those of step 0 as
// these are used up, the stage goes back behind step 0, the copies into it are spread over the matrix instructions of
// step 1 (a wave waits where the CU's copy path does not take its next copy: issued in one run, 9 copies held up the
// wave's matrix instructions), and the barrier that opens the next slab sits in the middle of step 1, whose second
// half covers the first reads of that slab.  Before, one barrier per slab opened it and its copies followed in one
// run: a tile of two full blocks has LDS for two stages, so the copy path went idle once per slab.
// 24593 tokens on 32 experts (K = N = 2048): 899 -> 855 us for the layer (882 with the copies in one run);
// 4096 tokens on 256 experts (K 7168, N 4096): 2712 -> 2649 us.  Reading both steps first at NTF = 4 spills registers:
// 1019 and 2981 us.
//
// Slab 0 goes to stage 0, the following ones to the stages behind it (wrapping).  `n_pre`: the
// caller has already issued slabs 0 .. n_pre - 1 (see pre_issue; a workgroup that runs one tile
// after another issues them under the previous tile's epilogue).
template <int DT, int RB, int NTF>
__device__ __forceinline__ void main_loop(f32x16 (&acc)[2][4], const Loader<RB> &ld, const Layout &lay, char *lds,
                                          int n_slabs, const int (&wrow)[2], int lane, int tok_region, int start,
                                          int n_pre) {
    static_assert(DT == DT_FP8 && RB == 128, "two scaled matrix instructions of 64 e4m3 per slab and accumulator");
    const int SB = lay.stage_bytes, NS = lay.stages;
    auto rot = [&](int s) {
        s += start;
        return s >= n_slabs ? s - n_slabs : s;
    };
    for (int s = n_pre; s < NS; ++s)
        if (s < n_slabs) ld.issue(lds + s * SB, rot(s));
    const int lps = ld.lps;
    // opens slab k: it has landed once at most the copies of the later slabs (up to NS - 1) are pending
    // (copies and stores of an epilogue that are in flight too only make the counted waits longer)
    auto open = [&](int k) { wait_and_barrier_dyn(lps * min(NS - 1, n_slabs - 1 - k)); };
    // gives the stage of slab k, which every wave has read, to slab k + NS
    auto refill = [&](int k, int off) {
        if (k + NS < n_slabs) {
            all_read();
            ld.issue(lds + off, rot(k + NS));
        }
    };
    int cur_off = 0;  // stage of slab kt
    auto next = [&](int off) { return off + SB >= NS * SB ? 0 : off + SB; };
    open(0);
    if constexpr (NTF > 0) {
        const int r = lane & 31, half = lane >> 5, sh = 8 * half;
        const int off0 = r * RB + ((half ^ swz<RB>(r)) << 4);
        const int w_at[2] = {lay.w_off + wrow[0] * RB, lay.w_off + wrow[1] * RB};
        const int tok_sc_at = lay.scale_off + (tok_region / RB + r) * 4;
        const int w_sc_at[2] = {lay.scale_off + (lay.tok_rows + wrow[0] + r) * 4,
                                lay.scale_off + (lay.tok_rows + wrow[1] + r) * 4};
        auto read_a = [&](Operands<NTF> &o, int f, const char *st, int j) { o.a[f] = lds_frag(st + w_at[f], off0 ^ (64 * j)); };
        auto read_b = [&](Operands<NTF> &o, int t, const char *st, int j) { o.b[t] = lds_frag(st + tok_region + t * 32 * RB, off0 ^ (64 * j)); };
        auto read_sa = [&](Operands<NTF> &o, int f, const char *st) { o.sa[f] = *reinterpret_cast<const int *>(st + w_sc_at[f]); };
        auto read_sb = [&](Operands<NTF> &o, int t, const char *st) { o.sb[t] = *reinterpret_cast<const int *>(st + tok_sc_at + 128 * t); };
        if constexpr (NTF <= 2) {
            for (int kt = 0; kt < n_slabs; ++kt) {
                const char *st = lds + cur_off;
                Operands<NTF> o[2];
#pragma unroll
                for (int f = 0; f < 2; ++f) {
                    read_sa(o[0], f, st);
                    read_a(o[0], f, st, 0);
                }
#pragma unroll
                for (int t = 0; t < NTF; ++t) {
                    read_sb(o[0], t, st);
                    read_b(o[0], t, st, 0);
                }
#pragma unroll
                for (int f = 0; f < 2; ++f) read_a(o[1], f, st, 1);
#pragma unroll
                for (int t = 0; t < NTF; ++t) read_b(o[1], t, st, 1);
                refill(kt, cur_off);
#pragma unroll
                for (int f = 0; f < 2; ++f) o[0].sa[f] = o[1].sa[f] = (int)((uint32_t)o[0].sa[f] >> sh);
#pragma unroll
                for (int t = 0; t < NTF; ++t) {
                    o[0].sb[t] = o[1].sb[t] = (int)((uint32_t)o[0].sb[t] >> sh);
                    mma<NTF, 0, 0>(acc, o[0], t);
                    mma<NTF, 0, 1>(acc, o[0], t);
                }
#pragma unroll
                for (int t = 0; t < NTF; ++t) {
                    mma<NTF, 1, 0>(acc, o[1], t);
                    mma<NTF, 1, 1>(acc, o[1], t);
                }
                cur_off = next(cur_off);
                if (kt + 1 < n_slabs) open(kt + 1);
            }
        } else {
            Operands<NTF> o;
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                read_a(o, f, lds + cur_off, 0);
                read_sa(o, f, lds + cur_off);
            }
#pragma unroll
            for (int t = 0; t < NTF; ++t) {
                read_b(o, t, lds + cur_off, 0);
                read_sb(o, t, lds + cur_off);
            }
            // step 0 of the slab in stage `st`: the operands are replaced as they are used up by those of step 1
            auto step0 = [&](const char *st) {
                o.sa[0] = (int)((uint32_t)o.sa[0] >> sh);
#pragma unroll
                for (int t = 0; t < NTF; ++t) {
                    o.sb[t] = (int)((uint32_t)o.sb[t] >> sh);
                    mma<NTF, 0, 0>(acc, o, t);
                    PMOE_RING_FENCE();
                }
                read_a(o, 0, st, 1);
                o.sa[1] = (int)((uint32_t)o.sa[1] >> sh);
                PMOE_RING_FENCE();
#pragma unroll
                for (int t = 0; t < NTF; ++t) {
                    mma<NTF, 0, 1>(acc, o, t);
                    read_b(o, t, st, 1);
                    PMOE_RING_FENCE();
                }
                read_a(o, 1, st, 1);
                PMOE_RING_FENCE();
            };
            for (int kt = 0; kt < n_slabs - 1; ++kt) {
                step0(lds + cur_off);
                const bool fill = kt + NS < n_slabs;
                char *fill_st = lds + cur_off;
                const int fslab = rot(fill ? kt + NS : 0);
                if (fill) all_read();
                auto copies = [&](int c0, int c1) {
                    if (fill) {
#pragma unroll
                        for (int c = 0; c < Loader<RB>::kPieces; ++c)
                            if (c >= c0 && c < c1) ld.issue_piece(c, fill_st, fslab);
                    }
                    PMOE_RING_FENCE();
                };
                constexpr int W = Loader<RB>::kWPieces, P = Loader<RB>::kPieces - W;
                cur_off = next(cur_off);
                const char *st = lds + cur_off;
#pragma unroll
                for (int t = 0; t < NTF; ++t) {
                    mma<NTF, 1, 0>(acc, o, t);
                    copies(t * W / NTF, (t + 1) * W / NTF);
                }
                wait_and_barrier_dyn(lps * min(NS - 2, n_slabs - 2 - kt) + (fill ? W : 0));
                read_a(o, 0, st, 0);
                read_sa(o, 0, st);
                PMOE_RING_FENCE();
#pragma unroll
                for (int t = 0; t < NTF; ++t) {
                    mma<NTF, 1, 1>(acc, o, t);
                    read_b(o, t, st, 0);
                    read_sb(o, t, st);
                    copies(W + t * P / NTF, W + (t + 1) * P / NTF);
                }
                read_a(o, 1, st, 0);
                read_sa(o, 1, st);
                PMOE_RING_FENCE();
            }
            step0(lds + cur_off);
#pragma unroll
            for (int t = 0; t < NTF; ++t) {
                mma<NTF, 1, 0>(acc, o, t);
                mma<NTF, 1, 1>(acc, o, t);
            }
        }
        // the sums are complete here: the compiler would move matrix instructions into the branches of the epilogue
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int t = 0; t < NTF; ++t) asm volatile("" : "+v"(acc[f][t]));
    } else {
        for (int kt = 0; kt < n_slabs - 1; ++kt) {
            refill(kt, cur_off);
            cur_off = next(cur_off);
            open(kt + 1);
        }
    }
    __syncthreads();  // all reads of the last stages are done: the ring may be reused as scratch
}

}  // namespace ring
}  // namespace pmoe

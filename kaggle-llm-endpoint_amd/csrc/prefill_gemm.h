// Grouped GEMMs of the prefill for CB3, IQ2_S, IQ3_S, IQ4_XS, Q2_K and Q3_K experts on the gfx950 matrix cores (the
// reference's moe_ragged_gateup / moe_ragged_down, pallas_moe.py:622-755, and the rounding forms of its other bf16
// prefill branches, resident.py:122-135,169-210):
//   prefill_kernel<MODE, WP, FORM>  one workgroup per (block, row range) streams the block's expert once for all
//                       its rows: each wavefront owns 64 (CB3) or 32 weight rows x up to 80 rows of activations (5
//                       MFMA token tiles; 128 and 8 in the wide launches), decodes every weight once (CB3: the decoder
//                       of cb3_tiles.h; the block formats: the planes straight into the A operand) and reuses it
//                       across the token tiles; the block's activation rows are
//                       staged one column tile (160 / 128 columns) at a time in LDS;
//                         gate/up: h = bf16(silu(min(g, L)) * clip(u, -L, L)), g and u f32    (pallas_moe.py:682)
//                         down:    y = bf16(h Wd^T), f32 accumulation                        (pallas_moe.py:747)
//                       FORM adds the other branches' rounding points at compile time (kPfRoundGU, kPfScaleH, kPfY32).
// Each (MODE, FORM) is instantiated for every format in a translation unit of its own (k_prefill.hip), which
// exports launch_prefill_<MODE>_<FORM>.
#pragma once
#include <type_traits>

#include "cb3_tiles.h"
#include "formats.h"

namespace mi {

// IQ3_S grid levels (internal linkage: every translation unit that launches a kernel carries its own copy)
static __constant__ uint32_t kPfGrid[512] = {
#include "iq3s_grid.inc"
};
static __constant__ uint32_t kPfGrid2[2048] = {
#include "iq2s_grid.inc"
};
static __constant__ int8_t kPfKv[16] = {
#include "iq4nl_kvalues.inc"
};

constexpr int kPfTT = 5;                   // token tiles of 16 rows per block
constexpr int kPfWideTT = 8;               // ... of the wide launches (block formats, many rows per expert)
constexpr int kPfWaves = 4;                // CB3: wavefronts per workgroup ...
constexpr int kPfRtw = 4;                  // ... and row tiles per wavefront (64 weight rows)
// The block formats: 128 rows per workgroup, 4 wavefronts of 32 rows in at most 168 registers and 49 KB of LDS, so that
// three wavefronts per SIMD cover each other's table gathers, barriers and loads.  IQ2_S + IQ4_XS layer, D 6144, I 2048,
// against two wavefronts of 64 rows (256 registers, 77 KB) with the same decoders: 27 tokens 319 -> 292 us, 512 tokens
// the same; in launch order by token tiles with the last blocks' tasks dealt singly 285 and 531 (from 541)
//
// The wide launches decode a weight once for up to 128 rows instead of 80, with two wavefronts per SIMD (acc and staging
// of 8 token tiles): fewer decodes where an expert's rows fill such blocks, fewer wavefronts where they do not.
constexpr int kPfBWaves = 4, kPfBRtw = 2;
constexpr int pf_per_simd(int tt, bool block) { return !block || tt > kPfTT ? 2 : 3; }
constexpr int kPfXPitch = 88;              // dwords per staged activation row of one column tile (80 + 8: the
                                           // fastest pitch for this read pattern on gfx950, measured)
constexpr int pf_gpitch(int tt) { return 16 * tt + 4; }   // floats per row of the gate/up epilogue's exchange (skewed banks)
constexpr int kXcds = 8;                   // accelerator complex dies of MI355X (one L2 each)
constexpr uint32_t kXOut = 0x80000000u;    // activation offset past every buffer's byte range (reads zero)

// ------------------------------------------------------------------------------------------------ grouped GEMM
struct PfArgs {
    Cb3Table t0, t1;                       // CB3 tables -- gate/up: gate, up; down: down (twice)
    Iq3Table i0, i1;                       // IQ3_S tables, the same roles
    Iq4Table k0, k1;                       // IQ4_XS tables, the same roles
    Iq2Table j0, j1;                       // IQ2_S tables, the same roles
    KqTable q0, q1;                        // Q2_K / Q3_K tables, the same roles
    int R, K;                              // output columns (rows of the table), input columns
    const int32_t *blk_expert, *blk_n, *blk_order, *n_blocks, *tok_row;
    const uint16_t *x;                     // gate/up: x [T, K] gathered through tok_row; down: h [Rp, K]
    uint32_t x_bytes;                      // bytes of x (< 2^31)
    int gather;
    uint16_t *out;                         // gate/up: h [Rp, R]; down: y [Rp, R]
    float limit;
    int RBG;                               // workgroups per block
    const float *w_row;                    // gate/up with kPfScaleH: the plan's routing weight of every row
    float *out32;                          // down with kPfY32: y [Rp, R] in f32
    int wide;                              // blocks of kPfWideTT token tiles
    int P;                                 // workgroups resident at once over the chip
    float *part;                           // split tasks' piece sums: P x pf_part_bytes
    uint32_t *cnt;                         // split tasks' piece counters: P, zero between launches
};

// A task of the launch's last, partial round is split along K into pieces (at most kPfMaxPieces, whole super tiles
// each); a piece stores its accumulators here (pf_part_bytes per piece).
constexpr int kPfMaxPieces = 4;
constexpr int pf_part_bytes(int tt, bool block) { return (block ? kPfBWaves * kPfBRtw : kPfWaves * kPfRtw) * tt * 64 * 16; }

// Rounding forms of the epilogues (FORM, a compile-time set; the ragged kernels use none):
constexpr int kPfRoundGU = 1;   // gate/up: g and u rounded to bf16 before the SwiGLU (the XLA einsums' bf16 outputs)
constexpr int kPfScaleH = 2;    // gate/up: h = bf16(f32(bf16(swiglu)) * w_row[row]) (the sweeps' weighted activations)
constexpr int kPfY32 = 4;       // down: y stored in f32 into out32, not rounded (the sweeps)

// k-steps M..4 of column tile C.  cbr[r] holds the codebook of row tile r's current group: it switches to LDS slot
// C + 1 at step 4 - C and is carried into the next column tile, which starts in that group, so a super tile reads
// each of its five groups from LDS once.  NTT (the block's token tiles) is a compile-time count, so a step's B
// reads and matrix-core instructions form one straight-line block.
template <int NTT, int C, int M>
__device__ __forceinline__ void pf_steps(const uint4 (&wv)[kPfRtw], const uint4 *cbrow, uint4 (&cbr)[kPfRtw],
                                         const uint32_t *xrow, f32x4 (&acc)[kPfRtw][NTT]) {
    if constexpr (M < 5) {
        // one k-step at a time: left free, the scheduler hoists every step's LDS reads and decodes and spills
        if constexpr (M > 0) __builtin_amdgcn_sched_barrier(0);
        if constexpr (M == 4 - C) {
#pragma unroll
            for (int r = 0; r < kPfRtw; ++r) cbr[r] = cbrow[(C + 1) * 64 + 16 * r];
        }
        // the step's B operands first; then row tile by row tile, so the decode of row tile r + 1 (vector ALU)
        // issues while the matrix-core instructions of row tile r run
        uint4 b[NTT];
#pragma unroll
        for (int tt = 0; tt < NTT; ++tt) b[tt] = *(const uint4 *)(xrow + tt * 16 * kPfXPitch + 16 * M);
        uint32_t s0, s1;
        cb3_sel<M>(wv[0], s0, s1);
        bf16x8 A = cb3_weights8(s0, s1, cbr[0]);
#pragma unroll
        for (int r = 0; r < kPfRtw; ++r) {
            bf16x8 An = A;
            if (r + 1 < kPfRtw) {
                cb3_sel<M>(wv[r + 1], s0, s1);
                An = cb3_weights8(s0, s1, cbr[r + 1]);
            }
#pragma unroll
            for (int tt = 0; tt < NTT; ++tt) acc[r][tt] = mfma16(A, b[tt], acc[r][tt]);
            A = An;
        }
        pf_steps<NTT, C, M + 1>(wv, cbrow, cbr, xrow, acc);
    }
}

// Code words of the wavefront's row tiles, two column tiles ahead (the matrix-core work per column tile is long
// enough that a deeper ring only costs registers).
struct PfRegs {
    uint4 ring[2][kPfRtw];    // slot c & 1 = column tile c
    uint4 cbv[5];             // codebook groups of the next super tile, as in Cb3Regs
    uint4 cbr[kPfRtw];        // codebook of the current group, per row tile (lane (q, i): row 16 r + i)
};

// Column tile C of super tile st (codebook slots as in cb3_ctile), B operands from the staged tile.
template <int NTT, int C>
__device__ __forceinline__ void pf_ctile(const Cb3Wave &w, PfRegs &s, int st, const uint32_t *xrow,
                                         f32x4 (&acc)[kPfRtw][NTT]) {
    const int lane = threadIdx.x & 63;
    const int gn = 5 * (st + 1);
    const uint4 *cbrow = w.cbl + (lane & 15);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (C == 0) {
        w.cbl[0 * 64 + lane] = s.cbv[0];
        w.cbl[1 * 64 + lane] = s.cbv[1];
        s.cbv[0] = cb3_group(w, gn);
        s.cbv[1] = cb3_group(w, gn + 1);
#pragma unroll
        for (int r = 0; r < kPfRtw; ++r) s.cbr[r] = cbrow[16 * r];
    } else {
        w.cbl[(C + 1) * 64 + lane] = s.cbv[C + 1];
        s.cbv[C + 1] = cb3_group(w, gn + C + 1);
    }
    const int ct = 4 * st + C;
    uint4 wv[kPfRtw];
#pragma unroll
    for (int r = 0; r < kPfRtw; ++r) {
        wv[r] = s.ring[C & 1][r];
        s.ring[C & 1][r] = cb3_tile(w, ct + 2, r);
    }
    pf_steps<NTT, C, 0>(wv, cbrow, s.cbr, xrow, acc);
}

// Bytes per staged activation row of a 128-column tile (the block formats).  16-byte chunk c of row i sits at chunk
// c ^ (i & 15): the 16 rows of an operand read, and the 16 chunks of a row written, fall on different banks.  A lane's
// chunk of step j is act_chunk(q) plus a constant of j on other bits, so an exclusive or with that constant finds it.
constexpr int kPfXRow = 256;

template <class WP, int TT>
struct PfShared {
    alignas(16) typename WP::Table tab;                      // the format's table, or CB3's codebook slots
    // column tiles ct (even/odd) of the block's rows, double-buffered; gate/up epilogue: gate accumulators
    static constexpr int kXBuf = 16 * TT * (WP::kCols == 128 ? kPfXRow / 4 : kPfXPitch);
    alignas(16) uint32_t xs[2][kXBuf];           // read and written 16 bytes at a time
    uint32_t xrowoff[16 * TT];                     // byte offset of every row's activations, or kXOut
    int last;                                    // split task: this workgroup's piece arrived last
};

// ------------------------------------------------------------------------------------------------ weight providers
// The block formats' decode and its LDS table gathers share a step with the matrix-core work, and with up to 5 token
// tiles per decoded weight they, not the MFMAs, set the pace.  Per 8 weights (a lane's A operand) the loops issue
// (vector instructions / table gathers, before -> now): IQ2_S 44 / 2 x 16 bytes -> 25 / 8 bytes (levels through a
// byte-permute table of the three scaled levels and their negatives), IQ3_S 41 / 3 x 16 -> 31 / 2 x 8, IQ4_XS 35 /
// 4 x 8 -> 23 / 4 x 4 (f16 levels widened inside the multiply), Q2_K 48 -> 28 (byte-permute table).  Measured at
// D 6144, I 2048, 64 experts, top-8, same bits: IQ2_S + IQ4_XS 27 tokens 453 -> 330 us, 512 tokens 705 -> 577, IQ3_S
// 1999 tokens 2288 -> 1919.
//
// A provider streams the weights of one wavefront's kRtw row tiles of expert e, one column tile at a time, and
// runs the tile's k-steps on the matrix cores against the staged activations.  Its state is two values the workgroup
// body keeps as locals: Wave (addressing, fixed per wavefront) and Regs (the loads in flight).
//   init(w, s, a, sh, mat, e, rg, wave, lane, st0, st1)   set up w for super tiles [st0, st1) (column tiles
//                                               [4 st0, 4 st1)), issue the first column tiles' loads into s
//   n_tiles(a, mat)                             column tiles of a row
//   tile<NTT, C>(w, s, st, xt, acc)             column tile 4 st + C; xt = the staged tile at row jt, lane group q (CB3)
//   tile<NTT, C>(w, s, st, xb, xoff, acc)       the same of the block formats; xb = the staged tile, xoff = the lane's byte
//                                               offset of chunk act_chunk(q) of row jt
//   kCols                                       columns per tile
//   kRtw, kWaves                                row tiles per wavefront, wavefronts per workgroup
//   kQOff (CB3)                                 dwords between lane groups' activations in a step
//   kSplit                                      whether the launch's last round of tasks is split into K pieces

// CB3: 160-column tiles of the code-tile layout; codebook slots per 640-column super tile (cb3_tiles.h).
//
// Split: the last round's tasks in K pieces.  The code for it costs registers that the CB3 loop does not have, and every
// piece stores and reads 80 KB of sums, so it is a kernel of its own, taken for rows of kPfCb3SplitTiles super tiles
// and more.  Whole / split, one launch, us (the plan's blocks from 16 to 1000 tokens): gate/up of K = 6144 (10 super tiles)
// 40 tokens 167 / 150, 100 173 / 161, 512 329 / 320, 1000 577 / 583; K = 4096 (7) 64 tokens 61.7 / 62.9, 333 105 / 102, 512
// 148 / 150; K = 3072 (5) 64 tokens 53.5 / 55.4; down of K = 2048 (4) 100 tokens 91 / 95, 512 178 / 173; K = 1536 (3) 512
// tokens 75 / 81; K = 768 (2) 40 tokens 19.8 / 25.0.
constexpr int kPfCb3SplitTiles = 8;

template <bool Split>
struct PfCb3 {
    struct Table {
        uint4 cbl[kPfWaves * 5 * 64];            // per-wavefront codebook slots (20 KB)
    };
    static constexpr bool kLdsOnlyBarrier = false;
    static constexpr int kCols = kCb3TileCols;
    static constexpr bool kSplit = Split;
    static constexpr int kRtw = kPfRtw, kWaves = kPfWaves;
    static constexpr int kQOff = 4;
    using Wave = Cb3Wave;
    using Regs = PfRegs;
    static __device__ __forceinline__ int n_tiles(const PfArgs &a, int mat) { return (mat ? a.t1 : a.t0).CT; }
    static __device__ __forceinline__ void init(Wave &w, Regs &s, const PfArgs &a, Table &sh, int mat, int e,
                                                int rg, int wave, int lane, int st0, int st1) {
        const Cb3Table &tb = mat ? a.t1 : a.t0;
        const uint32_t *qt = tb.qs + (size_t)e * tb.CT * tb.RT * 256;
        const uint32_t *cbe = tb.cb + (size_t)e * tb.G * tb.R * 4;
        w.qb = __builtin_amdgcn_make_buffer_rsrc((void *)qt, (short)0, 0x7fffffff, kBufferWord3);
        w.qnull = __builtin_amdgcn_make_buffer_rsrc((void *)qt, (short)0, 0, kBufferWord3);
        w.cbb = __builtin_amdgcn_make_buffer_rsrc((void *)cbe, (short)0, 0x7fffffff, kBufferWord3);
        w.cbnull = __builtin_amdgcn_make_buffer_rsrc((void *)cbe, (short)0, 0, kBufferWord3);
        w.ct_bytes = (uint32_t)tb.RT * 1024u;
        w.rt_bytes = (uint32_t)(rg * kPfRtw) * 1024u;
        w.g_bytes = (uint32_t)tb.R * 16u;
        w.row_bytes = (uint32_t)(rg * 64) * 16u;
        w.cta = 4 * st0;
        w.ctb = min(tb.CT, 4 * st1);
        w.g_first = 5 * st0;
        w.g_last = min(tb.G, 5 * st1) - 1;
        w.lane16 = (uint32_t)lane * 16u;
        w.cblane16 = (uint32_t)lane * 16u;
        w.xh = w.xl = nullptr;
        w.cbl = sh.cbl + wave * 5 * 64;
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int r = 0; r < kPfRtw; ++r) s.ring[c][r] = cb3_tile(w, 4 * st0 + c, r);
#pragma unroll
        for (int c = 0; c < 5; ++c) s.cbv[c] = cb3_group(w, 5 * st0 + c);
    }
    template <int NTT, int C>
    static __device__ __forceinline__ void tile(const Wave &w, Regs &s, int st, const uint32_t *xt,
                                                f32x4 (&acc)[kPfRtw][NTT]) {
        pf_ctile<NTT, C>(w, s, st, xt, acc);
    }
};

// One column tile of a block format, software-pipelined over its 8 A operands f = 2 j + r (k-step j, row tile r): while
// operand f meets the token tiles on the matrix cores, operand f + 1 is decoded and the table gathers of f + 2 are in
// flight, one matrix-core instruction between every few vector ones.  The pipeline runs on across tiles (s.A: the next
// tile's operand 0, s.g: the gathers of its operand 1), and each k-step's activations are read under the last row
// tile's matrix-core work of the step before.
//
// Free of this order the compiler clumped a step's decode and its MFMAs and waited for each gather where it was
// issued.
template <class WP, int NTT, int C>
__device__ __forceinline__ void pf_tile(const typename WP::Wave &w, typename WP::Regs &s, int st, const char *xb, uint32_t xoff,
                                        f32x4 (&acc)[kPfBRtw][NTT]) {
    constexpr int F = 4 * kPfBRtw;
    const int ct = 4 * st + C;
    uint4 b[NTT];
#pragma unroll
    for (int t = 0; t < NTT; ++t) b[t] = WP::acts(xb, xoff, t, 0);
#pragma unroll
    for (int f = 0; f < F; ++f) {
        const int r = f % kPfBRtw, j = f / kPfBRtw;
        const int f1 = (f + 1) % F, f2 = (f + 2) % F;
        const int c1 = f + 1 < F ? C : (C + 1) & 3, c2 = f + 2 < F ? C : (C + 1) & 3;
        __builtin_amdgcn_sched_barrier(0);
        const typename WP::Gather g2 = WP::gather(w, s.v[c2 & 1][f2 % kPfBRtw], c2, f2 / kPfBRtw);
        const bf16x8 An = WP::weights8(w, s, c1, f1 % kPfBRtw, f1 / kPfBRtw);
        if (f == F - 1) {
            // this tile's plane words have all been decoded: their slot's next column tile (zeros past the range)
#pragma unroll
            for (int rr = 0; rr < kPfBRtw; ++rr) WP::load(w, ct + 2, s.v[C & 1][rr], rr, ct + 2 < w.CT);
        }
#pragma unroll
        for (int t = 0; t < NTT; ++t) {
            acc[r][t] = mfma16(s.A, b[t], acc[r][t]);
            if (r == kPfBRtw - 1 && j < 3) b[t] = WP::acts(xb, xoff, t, j + 1);
        }
        __builtin_amdgcn_sched_group_barrier(0x2, 6, 0);                       // the gathers' addresses
        __builtin_amdgcn_sched_group_barrier(0x100, WP::kGathers, 0);
#pragma unroll
        for (int t = 0; t < NTT; ++t) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            if (r == kPfBRtw - 1 && j < 3) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x2, (WP::kValu - 6 + NTT - 1) / NTT, 0);
        }
        s.A = An;
        s.g = g2;
    }
}

// The first operand of a row's first column tile (plane words in slot 0).
template <class WP>
__device__ __forceinline__ void pf_tile_begin(const typename WP::Wave &w, typename WP::Regs &s) {
    s.g = WP::gather(w, s.v[0][0], 0, 0);
    s.A = WP::weights8(w, s, 0, 0, 0);
    s.g = WP::gather(w, s.v[0][1], 0, 0);
}

// IQ3_S: the reference's planes (planes.py:136-170, row on the minor axis) decoded straight into the matrix cores'
// A operand.  A column tile is 128 columns = 8 words = half a 256-weight block.  In k-steps 2m and 2m + 1 (m = 0, 1)
// lane (row i, group q) holds weights 0..7 and 8..15 of word 4m + q of the tile: the k order inside a step is free
// as long as the activations are read in the same order.  A weight is bf16(level * scale), scale = f16(d) * (1 + 2 sc)
// in f32 (the product is exact), rounded once to nearest even as the reference's tiles are (pallas_moe.py:341-350,
// with _decode_iq3_s :127-144); the sign is set on the rounded value (the rounding is symmetric).
constexpr int kIq3TileCols = 128;

__device__ __forceinline__ uint32_t pf_bf16_pair(float a, float b) {   // round to nearest even
    // one v_cvt_pk_bf16_f32 (an array of two __bf16 compiles to two conversions, a shift and an or)
    const bf16x2 v = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(uint32_t, v);
}

// f16 half H (0 low, 1 high) of v times s in f32 (v_fma_mix_f32: the f16 is widened in the instruction).
template <int H>
__device__ __forceinline__ float pf_mix(uint32_t v, float s) {
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    return fmaf((float)__builtin_bit_cast(f16x2, v)[H], s, 0.0f);
}

// The 16-bit values at bytes sel[b] of a table of up to 8 entries held as low and high bytes (entries 0..3 in *0, 4..7
// in *1), for the 4 selector bytes of sel: two dwords of bf16 pairs.
__device__ __forceinline__ uint2 pf_lookup4(uint32_t lo0, uint32_t lo1, uint32_t hi0, uint32_t hi1, uint32_t sel) {
    const uint32_t l = perm(lo1, lo0, sel), h = perm(hi1, hi0, sel);
    return make_uint2(perm(h, l, 0x05010400u), perm(h, l, 0x07030602u));
}

// One plane word (4 bytes) per lane at base + off if `use`, else zero: a buffer load through a descriptor whose
// range is empty when unused (no memory touched), so no branch surrounds the load and the compiler's wait counts
// stay exact (a load under a branch made it wait for every load in flight where the branch rejoins).  base must be
// wave-uniform: the lane's word and row go into off.
__device__ __forceinline__ uint32_t pf_word(const char *base, uint32_t off, bool use) {
    const __amdgpu_buffer_rsrc_t r =
        __builtin_amdgcn_make_buffer_rsrc((void *)base, (short)0, use ? 0x7fffffff : 0, kBufferWord3);
    return __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0);
}

struct PfIq3Wave {
    const char *qs, *sg, *qh, *sc, *dd;     // expert e's planes
    uint32_t rpitch;                        // bytes per plane row (4 R)
    uint32_t lrow;                          // the lane's byte offset in a plane row (row jt of the wavefront)
    int q;                                  // the lane's group
    int CT;                                 // column tiles of a row
    const uint2 *grid;                      // LDS: the grid's levels as f16
};
struct PfIq3Regs {
    // plane words of column tile ct in slot ct & 1, per row tile: qs of words q and 4 + q, their sg words, qh, sc, d
    uint32_t v[2][kPfBRtw][7];
    struct { uint2 lo, hi; } g;     // pf_tile's state: the next operand's gathers (levels of weights 0..3, 4..7) ...
    bf16x8 A;                       // ... and the operand to multiply
};

struct PfIq3 {
    struct Table {
        uint2 iq3grid[512];                      // grid entry -> its 4 levels as f16 (4 KB)
    };
    static constexpr bool kLdsOnlyBarrier = true;
    static constexpr bool kSplit = true;    // the last round's tasks split into K pieces
    static constexpr int kCols = kIq3TileCols;
    static constexpr int kRtw = kPfBRtw, kWaves = kPfBWaves;
    using Wave = PfIq3Wave;
    using Regs = PfIq3Regs;
    static __device__ __forceinline__ int n_tiles(const PfArgs &a, int mat) {
        return (mat ? a.i1 : a.i0).K / kIq3TileCols;
    }
    static __device__ __forceinline__ void load(const Wave &w, int ct, uint32_t (&u)[7], int r, bool use) {
        const uint32_t o = w.lrow + 64u * (uint32_t)r, P = w.rpitch;
        const uint32_t oq = (uint32_t)w.q * P + o, oq2 = (uint32_t)(w.q >> 1) * P + o;
        u[0] = pf_word(w.qs + (size_t)(8 * ct) * P, oq, use);
        u[1] = pf_word(w.qs + (size_t)(8 * ct + 4) * P, oq, use);
        u[2] = pf_word(w.sg + (size_t)(4 * ct) * P, oq2, use);
        u[3] = pf_word(w.sg + (size_t)(4 * ct + 2) * P, oq2, use);
        u[4] = pf_word(w.qh + (size_t)ct * P, o, use);
        u[5] = pf_word(w.sc + (size_t)(ct >> 1) * P, o, use);
        u[6] = pf_word(w.dd + (size_t)(ct >> 2) * P, o, use);
    }
    static __device__ __forceinline__ void init(Wave &w, Regs &s, const PfArgs &a, Table &sh, int mat, int e,
                                                int rg, int wave, int lane, int st0, int st1) {
        const Iq3Table &tb = mat ? a.i1 : a.i0;
        const size_t R = (size_t)tb.R;
        w.qs = (const char *)(tb.qs + (size_t)e * tb.W * R);
        w.sg = (const char *)(tb.sg + (size_t)e * (tb.W / 2) * R);
        w.qh = (const char *)(tb.qh + (size_t)e * (tb.W / 8) * R);
        w.sc = (const char *)(tb.sc + (size_t)e * (tb.W / 16) * R);
        w.dd = (const char *)(tb.d + (size_t)e * ((tb.nblk + 1) / 2) * R);
        w.rpitch = 4u * (uint32_t)tb.R;
        w.q = lane >> 4;
        w.lrow = 4u * (uint32_t)(rg * 16 * kPfBRtw + (lane & 15));
        w.CT = min(tb.K / kIq3TileCols, 4 * st1);          // prefetch no column tile past the range
        w.grid = sh.iq3grid;
        (void)wave;
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int r = 0; r < kPfBRtw; ++r) load(w, 4 * st0 + c, s.v[c][r], r, true);
    }
    static constexpr bool kHalfChunk = false;
    static constexpr int kValu = 32, kGathers = 2;
    using Gather = decltype(Regs::g);
    static __device__ __forceinline__ uint32_t act_chunk(int q) { return 2 * q; }
    static __device__ __forceinline__ uint4 acts(const char *xb, uint32_t xoff, int t, int j) {
        return *(const uint4 *)(xb + t * 16 * kPfXRow + (xoff ^ 16 * (8 * (j >> 1) + (j & 1))));
    }
    // the grid entries of step j's 8 weights, column tile c (mod 4), for the row tile whose plane words are u
    static __device__ __forceinline__ Gather gather(const Wave &w, const uint32_t (&u)[7], int, int j) {
        const int m = j >> 1, half = j & 1;
        const uint32_t word = m ? u[1] : u[0], qh4 = u[4] >> (4 * w.q) >> (16 * m);
        const uint32_t i0 = ((word >> (16 * half)) & 255u) | (((qh4 >> (2 * half)) & 1u) << 8);
        const uint32_t i1 = ((word >> (16 * half + 8)) & 255u) | (((qh4 >> (2 * half + 1)) & 1u) << 8);
        return {w.grid[i0], w.grid[i1]};
    }
    // the 8 weights of step j of column tile c (mod 4), row tile r, from the gathers in s.g
    static __device__ __forceinline__ bf16x8 weights8(const Wave &w, const Regs &s, int c, int r, int j) {
        const uint32_t (&u)[7] = s.v[c & 1][r];
        const int m = j >> 1, half = j & 1, q = w.q;
        // the word's 16 signs; sg2 has sign 2p at bit 2p and sign 2p + 1 at bit 2p + 16, a pair's two bf16 sign
        // bits once shifted left by 15 - 2p
        const uint32_t sg = ((m ? u[3] : u[2]) >> (16 * (q & 1))) & 0xffffu, sg2 = (sg << 15) | sg;
        const uint32_t nib = (u[5] >> (4 * (q >> 1)) >> (16 * (c & 1) + 8 * m)) & 15u;
        const float scale = f16_bits_to_f32(u[6] >> (16 * (c >> 1))) * (float)(1u + 2u * nib);
        const uint2 g0 = s.g.lo, g1 = s.g.hi;
        const int sh = 15 - 8 * half;
        uint4 A;
        A.x = pf_bf16_pair(pf_mix<0>(g0.x, scale), pf_mix<1>(g0.x, scale)) ^ ((sg2 << sh) & 0x80008000u);
        A.y = pf_bf16_pair(pf_mix<0>(g0.y, scale), pf_mix<1>(g0.y, scale)) ^ ((sg2 << (sh - 2)) & 0x80008000u);
        A.z = pf_bf16_pair(pf_mix<0>(g1.x, scale), pf_mix<1>(g1.x, scale)) ^ ((sg2 << (sh - 4)) & 0x80008000u);
        A.w = pf_bf16_pair(pf_mix<0>(g1.y, scale), pf_mix<1>(g1.y, scale)) ^ ((sg2 << (sh - 6)) & 0x80008000u);
        return __builtin_bit_cast(bf16x8, A);
    }
    template <int NTT, int C>
    static __device__ __forceinline__ void tile(const Wave &w, Regs &s, int st, const char *xb, uint32_t xoff,
                                                f32x4 (&acc)[kPfBRtw][NTT]) {
        pf_tile<PfIq3, NTT, C>(w, s, st, xb, xoff, acc);
    }
};

// IQ2_S: the reference's planes (planes.py:17-21, 136-170) decoded straight into the A operand.  A column tile is
// 128 columns = 4 words (half a 256-weight block).  In k-step j lane (row i, group q) holds group j of word q of the
// tile, i.e. columns 32q + 8j .. 32q + 8j + 7: the k order inside a step is free as long as the activations are read
// in the same order, and this one lets a lane read only its own word of each plane.  A weight is bf16(level * scale),
// scale = f16(d) * (0.5 + sc) * 0.25 in f32 (the product is exact), rounded once to nearest even as the reference's
// tiles are (pallas_moe.py:105-124, 341-350); the sign is set on the rounded value (the rounding is symmetric).
struct PfIq2Wave {
    const char *qs, *sg, *qh, *sc, *dd;     // expert e's planes
    uint32_t rpitch;                        // bytes per plane row (4 R)
    uint32_t lrow;                          // the lane's byte offset in a plane row (row jt of the wavefront)
    int q, CT;
    const uint2 *code;                      // LDS: grid entry -> 8 level codes
};
struct PfIq2Regs {
    uint32_t v[2][kPfBRtw][5];   // column tile ct in slot ct & 1, per row tile: the lane's qs and sg words, qh, sc, d
    // The scaled levels of one 16-weight scale group as a byte table: entry c (0..2) is bf16(level c * scale), entry
    // c + 4 its negative; low bytes, high bytes, high bytes of the negatives.
    struct Levels {
        uint32_t lo, hi, neg;
    } lv[kPfBRtw];               // per row tile, steps 2 jj and 2 jj + 1
    uint2 g;                    // pf_tile's state: the next operand's gather (8 level codes) ...
    bf16x8 A;                   // ... and the operand to multiply
};

struct PfIq2 {
    struct Table {
        uint2 iq2code[1024];                     // grid entry -> its 8 levels as codes 0..2, one byte each (8 KB)
    };
    static constexpr bool kLdsOnlyBarrier = true;
    static constexpr bool kSplit = true;    // the last round's tasks split into K pieces
    static constexpr int kCols = 128;
    static constexpr int kRtw = kPfBRtw, kWaves = kPfBWaves;
    using Wave = PfIq2Wave;
    using Regs = PfIq2Regs;
    static __device__ __forceinline__ int n_tiles(const PfArgs &a, int mat) { return (mat ? a.j1 : a.j0).K / 128; }
    static __device__ __forceinline__ void load(const Wave &w, int ct, uint32_t (&u)[5], int r, bool use) {
        const uint32_t o = w.lrow + 64u * (uint32_t)r, P = w.rpitch, oq = (uint32_t)w.q * P + o;
        u[0] = pf_word(w.qs + (size_t)(4 * ct) * P, oq, use);
        u[1] = pf_word(w.sg + (size_t)(4 * ct) * P, oq, use);
        u[2] = pf_word(w.qh + (size_t)ct * P, o, use);                  // byte q: word 4 ct + q
        u[3] = pf_word(w.sc + (size_t)ct * P, o, use);
        u[4] = pf_word(w.dd + (size_t)(ct >> 2) * P, o, use);
    }
    static __device__ __forceinline__ void init(Wave &w, Regs &s, const PfArgs &a, Table &sh, int mat, int e,
                                                int rg, int wave, int lane, int st0, int st1) {
        const Iq2Table &tb = mat ? a.j1 : a.j0;
        const size_t R = (size_t)tb.R;
        w.qs = (const char *)(tb.qs + (size_t)e * tb.W * R);
        w.sg = (const char *)(tb.sg + (size_t)e * tb.W * R);
        w.qh = (const char *)(tb.qh + (size_t)e * (tb.W / 4) * R);
        w.sc = (const char *)(tb.sc + (size_t)e * (tb.W / 4) * R);
        w.dd = (const char *)(tb.d + (size_t)e * ((tb.nblk + 1) / 2) * R);
        w.rpitch = 4u * (uint32_t)tb.R;
        w.q = lane >> 4;
        w.lrow = 4u * (uint32_t)(rg * 16 * kPfBRtw + (lane & 15));
        w.CT = min(tb.K / 128, 4 * st1);                   // prefetch no column tile past the range
        w.code = sh.iq2code;
        (void)wave;
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int r = 0; r < kPfBRtw; ++r) load(w, 4 * st0 + c, s.v[c][r], r, true);
    }
    static constexpr bool kHalfChunk = false;
    static constexpr int kValu = 26, kGathers = 1;
    using Gather = uint2;
    static __device__ __forceinline__ uint32_t act_chunk(int q) { return 4 * q; }
    static __device__ __forceinline__ uint4 acts(const char *xb, uint32_t xoff, int t, int j) {
        return *(const uint4 *)(xb + t * 16 * kPfXRow + (xoff ^ 16 * j));
    }
    static __device__ __forceinline__ PfIq2Regs::Levels levels(const Wave &w, const uint32_t (&u)[5], int c, int jj) {
        const uint32_t nib = (u[3] >> (8 * w.q) >> (4 * jj)) & 15u;
        const float scale = f16_bits_to_f32(u[4] >> (16 * (c >> 1))) * 0.25f * (0.5f + (float)nib);
        const uint32_t c01 = pf_bf16_pair(8.0f * scale, 25.0f * scale), c2 = pf_bf16_pair(43.0f * scale, 0.0f);
        PfIq2Regs::Levels t;
        t.lo = perm(c2, c01, 0x0c040200u);
        t.hi = perm(c2, c01, 0x0c050301u);
        t.neg = t.hi ^ 0x80808080u;
        return t;
    }
    // the level codes of step j (group j of the lane's word) for the row tile whose plane words are u
    static __device__ __forceinline__ Gather gather(const Wave &w, const uint32_t (&u)[5], int, int j) {
        return w.code[((u[0] >> (8 * j)) & 255u) | (((u[2] >> (8 * w.q) >> (2 * j)) & 3u) << 8)];
    }
    // the 8 weights of step j of column tile c (mod 4), row tile r, from the gather in s.g
    static __device__ __forceinline__ bf16x8 weights8(const Wave &w, Regs &s, int c, int r, int j) {
        const uint32_t (&u)[5] = s.v[c & 1][r];
        if ((j & 1) == 0) s.lv[r] = levels(w, u, c, j >> 1);
        const PfIq2Regs::Levels &t = s.lv[r];
        // 4 sign bits to bit 2 of 4 bytes: one 24-bit multiply (shifts by 2, 9, 16, 23: no two bits meet)
        const uint32_t s0 = __umul24((u[1] >> (8 * j)) & 15u, 0x810204u) & 0x04040404u;
        const uint32_t s1 = __umul24((u[1] >> (8 * j + 4)) & 15u, 0x810204u) & 0x04040404u;
        const uint2 a0 = pf_lookup4(t.lo, t.lo, t.hi, t.neg, s.g.x | s0), a1 = pf_lookup4(t.lo, t.lo, t.hi, t.neg, s.g.y | s1);
        return __builtin_bit_cast(bf16x8, make_uint4(a0.x, a0.y, a1.x, a1.y));
    }
    template <int NTT, int C>
    static __device__ __forceinline__ void tile(const Wave &w, Regs &s, int st, const char *xb, uint32_t xoff,
                                                f32x4 (&acc)[kPfBRtw][NTT]) {
        pf_tile<PfIq2, NTT, C>(w, s, st, xb, xoff, acc);
    }
};

// Q2_K / Q3_K: the reference's planes (planes.py:34-41, 136-170) decoded straight into the A operand.  A column tile
// is 128 columns = half a block (half n = ct % 2); k-step j is the shift-j stripe of the half: lane (row i, group q)
// holds columns 32 j + 8 q .. 32 j + 8 q + 7 = bytes 0..3 of plane words q' = 2q, 2q + 1 at shift 2j (natural
// order), scale byte 8 n + 2 j + (q >= 2).  A weight is the reference's f32 value rounded once to bf16: Q2_K
// fma(v, d * sc, -dmin * m) (d * sc * v is exact: one rounding, as iqquant.py:213), Q3_K (v + 4 hbit - 4) * d * (sc - 32)
// (exact) (pallas_moe.py:165-209, 341-350).
struct PfKqWave {
    const char *qs, *sc, *dd, *hm;          // expert e's planes (hm: Q3_K)
    uint32_t rpitch;                        // bytes per plane row (4 R)
    uint32_t lrow;                          // the lane's byte offset in a plane row (row jt of the wavefront)
    int q, CT;
};
struct PfKqRegs {
    uint32_t v[2][kPfBRtw][7];   // column tile ct in slot ct & 1, per row tile: qs words 2q, 2q + 1, sc x 2, d, hm x 2
    struct {} g;                // pf_tile's state: no gathers, the operand to multiply
    bf16x8 A;
};

template <bool Q3>
struct PfKq {
    struct Table {};
    static constexpr bool kLdsOnlyBarrier = true;
    static constexpr bool kSplit = true;    // the last round's tasks split into K pieces
    static constexpr int kCols = 128;
    static constexpr int kRtw = kPfBRtw, kWaves = kPfBWaves;
    using Wave = PfKqWave;
    using Regs = PfKqRegs;
    static __device__ __forceinline__ int n_tiles(const PfArgs &a, int mat) { return (mat ? a.q1 : a.q0).K / 128; }
    static __device__ __forceinline__ void load(const Wave &w, int ct, uint32_t (&u)[7], int r, bool use) {
        const uint32_t o = w.lrow + 64u * (uint32_t)r, P = w.rpitch;
        const uint32_t oa = (uint32_t)(2 * w.q) * P + o, ob = oa + P;
        const int b = ct >> 1;
        u[0] = pf_word(w.qs + (size_t)(8 * ct) * P, oa, use);
        u[1] = pf_word(w.qs + (size_t)(8 * ct) * P, ob, use);
        u[2] = pf_word(w.sc + (size_t)(2 * ct) * P, o, use);
        u[3] = pf_word(w.sc + (size_t)(2 * ct + 1) * P, o, use);
        u[4] = pf_word(w.dd + (size_t)b * P, o, use);
        if constexpr (Q3) {
            u[5] = pf_word(w.hm + (size_t)(8 * b) * P, oa, use);
            u[6] = pf_word(w.hm + (size_t)(8 * b) * P, ob, use);
        }
    }
    static __device__ __forceinline__ void init(Wave &w, Regs &s, const PfArgs &a, Table &sh, int mat, int e,
                                                int rg, int wave, int lane, int st0, int st1) {
        const KqTable &tb = mat ? a.q1 : a.q0;
        const size_t R = (size_t)tb.R;
        w.qs = (const char *)(tb.qs + (size_t)e * 16 * tb.nblk * R);
        w.sc = (const char *)(tb.sc + (size_t)e * 4 * tb.nblk * R);
        w.dd = (const char *)(tb.d + (size_t)e * tb.nblk * R);
        w.hm = Q3 ? (const char *)(tb.hm + (size_t)e * 8 * tb.nblk * R) : nullptr;
        w.rpitch = 4u * (uint32_t)tb.R;
        w.q = lane >> 4;
        w.lrow = 4u * (uint32_t)(rg * 16 * kPfBRtw + (lane & 15));
        w.CT = min(tb.K / 128, 4 * st1);                   // prefetch no column tile past the range
        (void)sh;
        (void)wave;
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int r = 0; r < kPfBRtw; ++r) load(w, 4 * st0 + c, s.v[c][r], r, true);
    }
    // 4 weights from the 4 byte-sized values of t (each 0..3, Q3_K 0..7): f32 -> bf16 pairs
    static __device__ __forceinline__ uint2 four(uint32_t t, float m, float a) {
        const float v0 = (float)(t & 255u), v1 = (float)((t >> 8) & 255u);       // v_cvt_f32_ubyte0..3
        const float v2 = (float)((t >> 16) & 255u), v3 = (float)(t >> 24);
        return make_uint2(pf_bf16_pair(fmaf(v0, m, a), fmaf(v1, m, a)), pf_bf16_pair(fmaf(v2, m, a), fmaf(v3, m, a)));
    }
    static constexpr bool kHalfChunk = false;
    static constexpr int kValu = Q3 ? 34 : 27, kGathers = 0;
    using Gather = decltype(Regs::g);
    static __device__ __forceinline__ uint32_t act_chunk(int q) { return q; }
    static __device__ __forceinline__ uint4 acts(const char *xb, uint32_t xoff, int t, int j) {
        return *(const uint4 *)(xb + t * 16 * kPfXRow + (xoff ^ 16 * (4 * j)));
    }
    static __device__ __forceinline__ Gather gather(const Wave &, const uint32_t (&)[7], int, int) { return {}; }
    // the 8 weights of step j (shift stripe j) of column tile c (mod 4), row tile r
    static __device__ __forceinline__ bf16x8 weights8(const Wave &w, const Regs &s, int c, int r, int j) {
        const uint32_t (&u)[7] = s.v[c & 1][r];
        const int n = c & 1;
        const uint32_t sb = ((j >> 1 ? u[3] : u[2]) >> (16 * (j & 1) + 8 * (w.q >> 1))) & 255u;
        const float d = f16_bits_to_f32(u[4] & 0xffffu);
        uint32_t t0 = (u[0] >> (2 * j)) & 0x03030303u, t1 = (u[1] >> (2 * j)) & 0x03030303u;
        float m, a;
        if (Q3) {
            t0 |= ((u[5] >> (4 * n + j)) & 0x01010101u) << 2;
            t1 |= ((u[6] >> (4 * n + j)) & 0x01010101u) << 2;
            m = d * ((float)sb - 32.0f);                              // exact
            a = -4.0f * m;
        } else {
            // the scale group's four values as a byte table: v = 0..3 -> bf16(v * m + a), 0 * m too (d may be infinite)
            m = d * (float)(sb & 15u);
            a = -(f16_bits_to_f32(u[4] >> 16) * (float)(sb >> 4));
            const uint32_t c01 = pf_bf16_pair(fmaf(0.0f, m, a), m + a), c23 = pf_bf16_pair(fmaf(2.0f, m, a), fmaf(3.0f, m, a));
            const uint32_t lo = perm(c23, c01, 0x06040200u), hi = perm(c23, c01, 0x07050301u);
            const uint2 l0 = pf_lookup4(lo, lo, hi, hi, t0), l1 = pf_lookup4(lo, lo, hi, hi, t1);
            return __builtin_bit_cast(bf16x8, make_uint4(l0.x, l0.y, l1.x, l1.y));
        }
        const uint2 l0 = four(t0, m, a), l1 = four(t1, m, a);
        return __builtin_bit_cast(bf16x8, make_uint4(l0.x, l0.y, l1.x, l1.y));
    }
    template <int NTT, int C>
    static __device__ __forceinline__ void tile(const Wave &w, Regs &s, int st, const char *xb, uint32_t xoff,
                                                f32x4 (&acc)[kPfBRtw][NTT]) {
        pf_tile<PfKq<Q3>, NTT, C>(w, s, st, xb, xoff, acc);
    }
};

// IQ4_XS: the reference's planes (planes.py:26-28, 136-170) decoded straight into the A operand.  A column tile is
// 128 columns (4 sub-blocks of 32, half a block); the k-step of sub-block i takes, for lane group q, plane word 4i + q:
// byte j of it holds sub-block columns 4q + j (low nibble) and 16 + 4q + j (high nibble).  The lane's A elements are
// columns 4q .. 4q+3 then 16 + 4q .. 16 + 4q + 3, so the activations are read as two 8-byte pieces of the staged
// tile.  A weight is bf16(level * f16(d) * (s - 32)): the f32 product is exact and rounded once to nearest even, as
// the reference's tiles are (pallas_moe.py:147-162, 341-350).
struct PfIq4Wave {
    const char *qs, *sl, *sh, *dd;          // expert e's planes
    uint32_t rpitch;                        // bytes per plane row (4 R)
    uint32_t lrow;                          // the lane's byte offset in a plane row (row jt of the wavefront)
    int q, CT;
    const uint32_t *pair;                   // LDS: byte -> its two levels as f16
};
struct PfIq4Regs {
    uint32_t v[2][kPfBRtw][7];   // column tile ct in slot ct & 1, per row tile: the 4 words, sl, sh, d
    uint4 g;                    // pf_tile's state: the next operand's gathers (level pairs of the word's 4 bytes) ...
    bf16x8 A;                   // ... and the operand to multiply
};

struct PfIq4 {
    struct Table {
        uint32_t iq4pair[256];                   // byte -> f16 levels of its low and its high nibble (1 KB)
    };
    static constexpr bool kLdsOnlyBarrier = true;
    static constexpr bool kSplit = true;    // the last round's tasks split into K pieces
    static constexpr int kCols = 128;
    static constexpr int kRtw = kPfBRtw, kWaves = kPfBWaves;
    using Wave = PfIq4Wave;
    using Regs = PfIq4Regs;
    static __device__ __forceinline__ int n_tiles(const PfArgs &a, int mat) { return (mat ? a.k1 : a.k0).K / 128; }
    static __device__ __forceinline__ void load(const Wave &w, int ct, uint32_t (&u)[7], int r, bool use) {
        const uint32_t o = w.lrow + 64u * (uint32_t)r, P = w.rpitch, oq = (uint32_t)w.q * P + o;
#pragma unroll
        for (int j = 0; j < 4; ++j) u[j] = pf_word(w.qs + (size_t)(16 * ct + 4 * j) * P, oq, use);
        u[4] = pf_word(w.sl + (size_t)(ct >> 1) * P, o, use);
        u[5] = pf_word(w.sh + (size_t)(ct >> 1) * P, o, use);
        u[6] = pf_word(w.dd + (size_t)(ct >> 2) * P, o, use);
    }
    static __device__ __forceinline__ void init(Wave &w, Regs &s, const PfArgs &a, Table &sh, int mat, int e,
                                                int rg, int wave, int lane, int st0, int st1) {
        const Iq4Table &tb = mat ? a.k1 : a.k0;
        const size_t R = (size_t)tb.R;
        w.qs = (const char *)(tb.qs + (size_t)e * tb.W * R);
        w.sl = (const char *)(tb.sl + (size_t)e * tb.nblk * R);
        w.sh = (const char *)(tb.sh + (size_t)e * tb.nblk * R);
        w.dd = (const char *)(tb.d + (size_t)e * ((tb.nblk + 1) / 2) * R);
        w.rpitch = 4u * (uint32_t)tb.R;
        w.q = lane >> 4;
        w.lrow = 4u * (uint32_t)(rg * 16 * kPfBRtw + (lane & 15));
        w.CT = min(tb.K / 128, 4 * st1);                   // prefetch no column tile past the range
        w.pair = sh.iq4pair;
        (void)wave;
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int r = 0; r < kPfBRtw; ++r) load(w, 4 * st0 + c, s.v[c][r], r, true);
    }
    static constexpr bool kHalfChunk = true;
    static constexpr int kValu = 24, kGathers = 4;
    using Gather = uint4;
    static __device__ __forceinline__ uint32_t act_chunk(int q) { return q >> 1; }      // odd lane groups: its second half
    static __device__ __forceinline__ uint4 acts(const char *xb, uint32_t xoff, int t, int j) {
        const char *row = xb + t * 16 * kPfXRow;
        const uint2 lo = *(const uint2 *)(row + (xoff ^ 16 * (4 * j)));
        const uint2 hi = *(const uint2 *)(row + (xoff ^ 16 * (4 * j + 2)));
        return make_uint4(lo.x, lo.y, hi.x, hi.y);
    }
    // the level pairs of step j's word for the row tile whose plane words are u (one read per nibble from 16 entries,
    // free of bank conflicts, costs more in extra instructions than the conflicts do: down 128 -> 151 us at 27 tokens)
    static __device__ __forceinline__ Gather gather(const Wave &w, const uint32_t (&u)[7], int, int j) {
        const uint32_t x = u[j];
        return make_uint4(w.pair[x & 255u], w.pair[(x >> 8) & 255u], w.pair[(x >> 16) & 255u], w.pair[x >> 24]);
    }
    // the 8 weights of step j (sub-block 4 (c % 2) + j) of column tile c (mod 4), row tile r, from the gathers in s.g
    static __device__ __forceinline__ bf16x8 weights8(const Wave &, const Regs &s, int c, int r, int j) {
        const uint32_t (&u)[7] = s.v[c & 1][r];
        const int i = 4 * (c & 1) + j;
        const int sv = (int)(((u[4] >> (4 * i)) & 15u) | (((u[5] >> (2 * i)) & 3u) << 4)) - 32;
        const float scale = f16_bits_to_f32(u[6] >> (16 * (c >> 1))) * (float)sv;
        const uint4 p = s.g;
        uint4 A;
        A.x = pf_bf16_pair(pf_mix<0>(p.x, scale), pf_mix<0>(p.y, scale));
        A.y = pf_bf16_pair(pf_mix<0>(p.z, scale), pf_mix<0>(p.w, scale));
        A.z = pf_bf16_pair(pf_mix<1>(p.x, scale), pf_mix<1>(p.y, scale));
        A.w = pf_bf16_pair(pf_mix<1>(p.z, scale), pf_mix<1>(p.w, scale));
        return __builtin_bit_cast(bf16x8, A);
    }
    template <int NTT, int C>
    static __device__ __forceinline__ void tile(const Wave &w, Regs &s, int st, const char *xb, uint32_t xoff,
                                                f32x4 (&acc)[kPfBRtw][NTT]) {
        pf_tile<PfIq4, NTT, C>(w, s, st, xb, xoff, acc);
    }
};

// One workgroup: block g (expert e, rows row0 .. row0 + n - 1, NTT = ceil(n / 16) token tiles), row range rbg.
// piece / np: the workgroup runs super tiles [piece n_st / np, (piece + 1) n_st / np) of the task (np == 1: all of
// them); sti: the split task's index among the launch's split tasks (counter and piece sums).
template <int MODE, int NTT, class WP, int FORM, int TT>
__device__ __forceinline__ void prefill_body(const PfArgs &a, PfShared<WP, TT> &sh, int g, int rbg, int e, int n, int piece,
                                             int np, int sti) {
    uint32_t *xs = &sh.xs[0][0], *xrowoff = sh.xrowoff;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int kTm = 16 * TT;                         // rows per block of the plan
    const int row0 = g * kTm;
    const int mat = MODE == 0 ? (wave & 1) : 0;
    constexpr int kRtw = WP::kRtw, kWaves = WP::kWaves;
    constexpr bool kBlock = WP::kCols == 128;             // a block format
    // this wavefront's group of 16 kRtw rows
    const int rg = rbg * (kWaves >> (MODE == 0)) + (MODE == 0 ? (wave >> 1) : wave);

    const int CT = WP::n_tiles(a, mat);
    const int n_st = (CT + 3) >> 2;                     // super tiles of a row (the last one maybe partial)
    const int s0 = WP::kSplit ? piece * n_st / np : 0, s1 = WP::kSplit ? (piece + 1) * n_st / np : n_st;
    const int ct_end = min(CT, 4 * s1);
    typename WP::Wave w;
    typename WP::Regs s;
    WP::init(w, s, a, sh.tab, mat, e, rg, wave, lane, s0, s1);

    // activation tile: the block's 16 NTT rows x kXU uint4 (WP::kCols columns), staged as buffer loads by
    // kXRows x kXU threads, kXRows rows per pass (thread t: row t / kXU + kXRows j, uint4 column t % kXU), so every
    // pass is a constant offset from the first; rows >= n and columns >= K take an offset past the buffer's range,
    // which reads zero
    constexpr int kXU = WP::kCols / 8;                        // 20 (CB3) or 16 (IQ3_S)
    constexpr int kXRows = (64 * kWaves) / kXU;               // 12 or 32
    constexpr int kXBuf = PfShared<WP, TT>::kXBuf;                // dwords per tile buffer
    constexpr int kXJ = (16 * NTT + kXRows - 1) / kXRows;
    const __amdgpu_buffer_rsrc_t xbuf =
        __builtin_amdgcn_make_buffer_rsrc((void *)a.x, (short)0, (int)a.x_bytes, kBufferWord3);
    if (tid < kTm) {
        uint32_t o = kXOut;
        if (tid < n) o = (uint32_t)(a.gather ? a.tok_row[row0 + tid] : row0 + tid) * (uint32_t)a.K * 2u;
        xrowoff[tid] = o;
    }
    __syncthreads();
    const int xr0 = tid / kXU, xc8 = tid - xr0 * kXU;
    const bool stager = tid < kXRows * kXU;
    uint4 xr[kXJ];
    // byte offset of the thread's piece j in column tile 0; the block formats hold theirs in registers for the whole
    // row (read from LDS at every tile they were a chain of LDS latencies at its start; CB3 has no registers left)
    auto piece_off = [&](int j) {
        const int row = xr0 + kXRows * j;
        return stager && row < 16 * NTT ? xrowoff[row] + 16u * (uint32_t)xc8 : kXOut;
    };
    uint32_t xo[kXJ];
    if constexpr (kBlock) {
#pragma unroll
        for (int j = 0; j < kXJ; ++j) xo[j] = piece_off(j);
    }
    const __amdgpu_buffer_rsrc_t xnull = __builtin_amdgcn_make_buffer_rsrc((void *)a.x, (short)0, 0, kBufferWord3);
    // use: whether the tile is staged at all (no branch around the loads: from an empty range they read zeros)
    auto load_x = [&](int ct, bool use) {
        const int lim = (a.K - WP::kCols * ct) >> 3;          // uint4 columns of this tile inside the row
        const __amdgpu_buffer_rsrc_t r = use ? xbuf : xnull;
#pragma unroll
        for (int j = 0; j < kXJ; ++j) {
            // K is whole 128-column tiles; a CB3 row may end inside its last 160-column tile
            const uint32_t o = kBlock ? xo[j] : xc8 < lim ? piece_off(j) : kXOut;
            xr[j] = bload(r, o, (uint32_t)(2 * WP::kCols * ct));
        }
    };
    auto store_x = [&](int buf) {
#pragma unroll
        for (int j = 0; j < kXJ; ++j) {
            const int row = xr0 + kXRows * j;
            const int at = kBlock ? row * (kPfXRow / 4) + 4 * (xc8 ^ (row & 15)) : row * kPfXPitch + 4 * xc8;
            if (stager && row < 16 * NTT) *(uint4 *)(xs + buf * kXBuf + at) = xr[j];
        }
    };
    load_x(4 * s0, true);
    if constexpr (kBlock) pf_tile_begin<WP>(w, s);      // the format's LDS table: published above
    store_x(0);

    f32x4 acc[kRtw][NTT];
#pragma unroll
    for (int r = 0; r < kRtw; ++r)
#pragma unroll
        for (int t = 0; t < NTT; ++t) acc[r][t] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int jt = lane & 15, q = lane >> 4;

    // one barrier per column tile: tile ct sits in buffer ct & 1 (= C & 1); the next tile's loads are issued first
    // (ahead of this tile's code and codebook loads, so waiting for them never waits for those) and stored into the
    // other buffer after this tile's matrix-core work, which every wavefront finished reading one barrier earlier.
    // The block formats' barrier orders LDS only (lds_barrier): a full __syncthreads also waits for every weight
    // load in flight, the prefetched next tiles included (IQ3_S 831 -> 761 us at 512 tokens with it).  CB3 keeps the
    // full barrier and the branch around its staging loads: without them its GEMMs measured slower.
    auto step = [&](auto Cc, int st) {
        constexpr int C = decltype(Cc)::value;
        const int ct = 4 * st + C;
        if constexpr (WP::kLdsOnlyBarrier) {
            lds_barrier();
            load_x(ct + 1, ct + 1 < ct_end);                // no branch around the loads
        } else {
            __syncthreads();
            if (ct + 1 < ct_end) load_x(ct + 1, true);
        }
        if constexpr (kBlock)
            WP::template tile<NTT, C>(w, s, st, (const char *)(xs + (C & 1) * kXBuf),
                                      jt * kPfXRow + 16 * (WP::act_chunk(q) ^ jt) + (WP::kHalfChunk ? 8 * (q & 1) : 0), acc);
        else WP::template tile<NTT, C>(w, s, st, xs + jt * kPfXPitch + WP::kQOff * q + (C & 1) * kXBuf, acc);
        if (ct + 1 < ct_end) store_x((C + 1) & 1);
    };
    const int st_full = min(CT >> 2, s1);
    int st = s0;
    for (; st < st_full; ++st) {
        step(std::integral_constant<int, 0>{}, st);
        step(std::integral_constant<int, 1>{}, st);
        step(std::integral_constant<int, 2>{}, st);
        step(std::integral_constant<int, 3>{}, st);
    }
    const int nct = ct_end - 4 * st;                    // 0..3 column tiles of a last, partial super tile
    if (nct > 0) step(std::integral_constant<int, 0>{}, st);
    if (nct > 1) step(std::integral_constant<int, 1>{}, st);
    if (nct > 2) step(std::integral_constant<int, 2>{}, st);

    if (WP::kSplit && np > 1) {
        // a piece of a split task: its sums go to memory (stored through this XCD's L2), then the piece is counted;
        // the piece that arrives last adds all of them in piece order (the same order whichever arrives last) and
        // runs the epilogue.  Nothing waits for another workgroup.  The other pieces' sums are read with device-coherent
        // (sc1) loads after the count, so no older copy of a line in this XCD's L2 can be returned.
        const __amdgpu_buffer_rsrc_t pr =
            __builtin_amdgcn_make_buffer_rsrc((void *)a.part, (short)0, 0x7fffffff, kBufferWord3);
        const uint32_t lane_off = 16u * (uint32_t)lane;
        auto part_off = [&](int pc, int r, int t) {
            return (uint32_t)(sti * np + pc) * (uint32_t)pf_part_bytes(TT, kBlock) +
                   (uint32_t)((wave * kRtw + r) * TT + t) * 1024u + lane_off;
        };
#pragma unroll
        for (int r = 0; r < kRtw; ++r)
#pragma unroll
            for (int t = 0; t < NTT; ++t) wt_store4(pr, part_off(piece, r, t), acc[r][t]);
        __builtin_amdgcn_s_waitcnt(0);                  // this wavefront's stores have completed
        __syncthreads();                                // ... and every wavefront's
        if (tid == 0) sh.last = counter_add(a.cnt + sti, 1u) == (uint32_t)(np - 1);
        __syncthreads();
        if (!sh.last) return;
        if (tid == 0) counter_reset(a.cnt + sti);       // zero again for the next launch
        // every piece's sums from memory, this one's too (its stores have completed), added in piece order
#pragma unroll
        for (int r = 0; r < kRtw; ++r)
#pragma unroll
            for (int t = 0; t < NTT; ++t) acc[r][t] = (f32x4){0.f, 0.f, 0.f, 0.f};
        for (int pc = 0; pc < np; ++pc) {
#pragma unroll
            for (int r = 0; r < kRtw; ++r)
#pragma unroll
                for (int t = 0; t < NTT; ++t)
                    acc[r][t] += coherent_load4(pr, part_off(pc, r, t));
        }
    }

    // epilogue: lane (jt, q) holds rows 16 r + 4 q + i (i = 0..3) of the wavefront's 16 kRtw rows for tokens 16 t + jt
    const int rbase = rg * 16 * kRtw;
    if constexpr (MODE == 0) {
        // gate accumulators of as many (gate, up) pairs as the activation buffers hold at once: [rows][kGPitch]
        constexpr int kPairs = kBlock ? kWaves / 2 : 1, kGPitch = pf_gpitch(TT);
        static_assert(kPairs * 16 * kRtw * kGPitch <= 2 * kXBuf, "the exchange fits the tile buffers");
        float *gbuf = (float *)xs + (kPairs > 1 ? (wave >> 1) * 16 * kRtw * kGPitch : 0);
        for (int pair = 0; pair < kWaves / 2; pair += kPairs) {
            const bool mine = kPairs > 1 || (wave >> 1) == pair;
            __syncthreads();
            if (mine && !(wave & 1)) {
#pragma unroll
                for (int r = 0; r < kRtw; ++r)
#pragma unroll
                    for (int t = 0; t < NTT; ++t)
#pragma unroll
                        for (int i = 0; i < 4; ++i) gbuf[(16 * r + 4 * q + i) * kGPitch + 16 * t + jt] = acc[r][t][i];
            }
            __syncthreads();
            if (mine && (wave & 1)) {
                constexpr bool round_gu = FORM & kPfRoundGU, scale_h = FORM & kPfScaleH;
#pragma unroll
                for (int t = 0; t < NTT; ++t) {
                    const int tok = 16 * t + jt;
                    if (tok < n) {
                        float wr = 1.0f;
                        if constexpr (scale_h) wr = a.w_row[row0 + tok];
#pragma unroll
                        for (int r = 0; r < kRtw; ++r) {
                            float hv[4];
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                float gv = gbuf[(16 * r + 4 * q + i) * kGPitch + tok], uv = acc[r][t][i];
                                if constexpr (round_gu) {
                                    gv = round_bf16(gv);
                                    uv = round_bf16(uv);
                                }
                                hv[i] = swiglu_clamped(gv, uv, a.limit);
                                if constexpr (scale_h) hv[i] = round_bf16(hv[i]) * wr;
                            }
                            uint2 v;
                            v.x = f32_to_bf16_rne(hv[0]) | (f32_to_bf16_rne(hv[1]) << 16);
                            v.y = f32_to_bf16_rne(hv[2]) | (f32_to_bf16_rne(hv[3]) << 16);
                            *(uint2 *)(a.out + (size_t)(row0 + tok) * a.R + rbase + 16 * r + 4 * q) = v;
                        }
                    }
                }
            }
        }
    } else if constexpr ((FORM & kPfY32) != 0) {
#pragma unroll
        for (int t = 0; t < NTT; ++t) {
            const int tok = 16 * t + jt;
            if (tok < n) {
#pragma unroll
                for (int r = 0; r < kRtw; ++r)
                    *(float4 *)(a.out32 + (size_t)(row0 + tok) * a.R + rbase + 16 * r + 4 * q) =
                        make_float4(acc[r][t][0], acc[r][t][1], acc[r][t][2], acc[r][t][3]);
            }
        }
    } else {
#pragma unroll
        for (int t = 0; t < NTT; ++t) {
            const int tok = 16 * t + jt;
            if (tok < n) {
#pragma unroll
                for (int r = 0; r < kRtw; ++r) {
                    uint2 v;
                    v.x = f32_to_bf16_rne(acc[r][t][0]) | (f32_to_bf16_rne(acc[r][t][1]) << 16);
                    v.y = f32_to_bf16_rne(acc[r][t][2]) | (f32_to_bf16_rne(acc[r][t][3]) << 16);
                    *(uint2 *)(a.out + (size_t)(row0 + tok) * a.R + rbase + 16 * r + 4 * q) = v;
                }
            }
        }
    }
}

template <int MODE, class WP, int FORM, int TT>   // MODE 0: gate/up -> h, 1: down -> y; FORM: kPf* rounding forms
__global__ void __launch_bounds__(64 * WP::kWaves, pf_per_simd(TT, WP::kCols == 128)) prefill_kernel(PfArgs a) {
    __shared__ PfShared<WP, TT> sh;
    // Workgroups are dispatched to the XCDs round-robin.  The blocks, in launch order (most token tiles first), are
    // dealt to the XCDs eight at a time, all workgroups of a block on one XCD, so the block's activation rows are
    // fetched into one L2 and read there by every workgroup.  The tasks of the blocks left over are dealt one by one:
    // whole, they would give some XCDs a block more than the others, an eighth of a launch of 64 blocks.
    // A launch runs n_blocks x RBG tasks on P resident workgroups.  The tasks of the last, partial round (its
    // blocks' tasks: the last sb blocks) are split along K into np pieces each, so that they spread over the slots
    // that free up: np = P / (their tasks), at most kPfMaxPieces and at most the row's super tiles.
    const int nb = *a.n_blocks;
    int sb = 0, np = 1;
    if constexpr (WP::kSplit) {
        const int r = (nb * a.RBG) % a.P;
        if (r > 0) {
            sb = (r + a.RBG - 1) / a.RBG;
            const int n_st = (WP::n_tiles(a, 0) + 3) >> 2;
            np = min(min(a.P / (sb * a.RBG), kPfMaxPieces), n_st);
            if (np < 2) np = 1, sb = 0;
        }
    }
    const int xcd = blockIdx.x % kXcds, li = blockIdx.x / kXcds;
    const int rounds = (nb - sb) / kXcds;               // blocks per XCD dealt whole
    int o, rbg, piece = 0, sti = 0, pieces = 1;
    if (li < rounds * a.RBG) {
        o = (li / a.RBG) * kXcds + xcd;
        rbg = li % a.RBG;
    } else {
        const int t = (li - rounds * a.RBG) * kXcds + xcd;
        const int whole = (nb - sb - rounds * kXcds) * a.RBG;
        if (t < whole) {
            o = rounds * kXcds + t / a.RBG;
            rbg = t % a.RBG;
        } else {
            const int i = t - whole;
            if (i >= np * sb * a.RBG) return;           // past the last task
            sti = i / np;
            piece = i - sti * np;
            pieces = np;
            o = nb - sb + sti / a.RBG;
            rbg = sti % a.RBG;
        }
    }
    const int g = __builtin_amdgcn_readfirstlane(a.blk_order[o]);
    const int e = __builtin_amdgcn_readfirstlane(a.blk_expert[g]);
    const int n = __builtin_amdgcn_readfirstlane(a.blk_n[g]);
    // the format's LDS table (published by the barrier after the row offsets)
    const auto f16_pair = [](float lo, float hi) {
        return (uint32_t)__builtin_bit_cast(unsigned short, (_Float16)lo) |
               (uint32_t)__builtin_bit_cast(unsigned short, (_Float16)hi) << 16;
    };
    if constexpr (std::is_same<WP, PfIq3>::value) {
        for (int i = threadIdx.x; i < 512; i += 64 * WP::kWaves) {
            const uint32_t v = kPfGrid[i];
            sh.tab.iq3grid[i] = make_uint2(f16_pair((float)(v & 255u), (float)((v >> 8) & 255u)),
                                       f16_pair((float)((v >> 16) & 255u), (float)(v >> 24)));
        }
    }
    if constexpr (std::is_same<WP, PfIq2>::value) {
        // levels 8, 25, 43 -> codes 0, 1, 2
        for (int i = threadIdx.x; i < 1024; i += 64 * WP::kWaves)
            sh.tab.iq2code[i] = make_uint2((kPfGrid2[2 * i] >> 4) & 0x03030303u, (kPfGrid2[2 * i + 1] >> 4) & 0x03030303u);
    }
    if constexpr (std::is_same<WP, PfIq4>::value) {
        for (int i = threadIdx.x; i < 256; i += 64 * WP::kWaves)
            sh.tab.iq4pair[i] = f16_pair((float)kPfKv[i & 15], (float)kPfKv[i >> 4]);
    }
    if constexpr (TT == kPfTT) {
        switch ((n + 15) >> 4) {
            case 1: prefill_body<MODE, 1, WP, FORM, TT>(a, sh, g, rbg, e, n, piece, pieces, sti); break;
            case 2: prefill_body<MODE, 2, WP, FORM, TT>(a, sh, g, rbg, e, n, piece, pieces, sti); break;
            case 3: prefill_body<MODE, 3, WP, FORM, TT>(a, sh, g, rbg, e, n, piece, pieces, sti); break;
            case 4: prefill_body<MODE, 4, WP, FORM, TT>(a, sh, g, rbg, e, n, piece, pieces, sti); break;
            default: prefill_body<MODE, 5, WP, FORM, TT>(a, sh, g, rbg, e, n, piece, pieces, sti); break;
        }
    } else {
        switch ((n + 31) >> 5) {                        // even counts: rows past n are zeros
            case 1: prefill_body<MODE, 2, WP, FORM, TT>(a, sh, g, rbg, e, n, piece, pieces, sti); break;
            case 2: prefill_body<MODE, 4, WP, FORM, TT>(a, sh, g, rbg, e, n, piece, pieces, sti); break;
            case 3: prefill_body<MODE, 6, WP, FORM, TT>(a, sh, g, rbg, e, n, piece, pieces, sti); break;
            default: prefill_body<MODE, 8, WP, FORM, TT>(a, sh, g, rbg, e, n, piece, pieces, sti); break;
        }
    }
}

// Launches prefill_kernel<MODE, *, FORM> for the table format qtype (MI_QT_*) on grid workgroups.
template <int MODE, int FORM, class WP>
void launch_prefill_block(dim3 grid, hipStream_t s, const PfArgs &a) {
    if (a.wide)
        hipLaunchKernelGGL((prefill_kernel<MODE, WP, FORM, kPfWideTT>), grid, dim3(64 * kPfBWaves), 0, s, a);
    else
        hipLaunchKernelGGL((prefill_kernel<MODE, WP, FORM, kPfTT>), grid, dim3(64 * kPfBWaves), 0, s, a);
}

template <int MODE, int FORM>
int launch_prefill(int qtype, dim3 grid, hipStream_t s, const PfArgs &a) {
    switch (qtype) {
        case MI_QT_IQ3_S: launch_prefill_block<MODE, FORM, PfIq3>(grid, s, a); break;
        case MI_QT_IQ4_XS: launch_prefill_block<MODE, FORM, PfIq4>(grid, s, a); break;
        case MI_QT_IQ2_S: launch_prefill_block<MODE, FORM, PfIq2>(grid, s, a); break;
        case MI_QT_Q2_K: launch_prefill_block<MODE, FORM, PfKq<false>>(grid, s, a); break;
        case MI_QT_Q3_K: launch_prefill_block<MODE, FORM, PfKq<true>>(grid, s, a); break;
        case MI_QT_CB3:
            if (a.K >= 4 * kCb3TileCols * (kPfCb3SplitTiles - 1) + 1)
                hipLaunchKernelGGL((prefill_kernel<MODE, PfCb3<true>, FORM, kPfTT>), grid, dim3(64 * kPfWaves), 0, s, a);
            else
                hipLaunchKernelGGL((prefill_kernel<MODE, PfCb3<false>, FORM, kPfTT>), grid, dim3(64 * kPfWaves), 0, s, a);
            break;
        default: return MI_ERR_QTYPE;
    }
    return hipGetLastError() == hipSuccess ? MI_OK : MI_ERR_LAUNCH;
}

// the instantiations, one translation unit each (k_prefill.hip)
int launch_prefill_0_0(int qtype, dim3 grid, hipStream_t s, const PfArgs &a);   // ragged gate/up
int launch_prefill_0_1(int qtype, dim3 grid, hipStream_t s, const PfArgs &a);   // kPfRoundGU
int launch_prefill_0_2(int qtype, dim3 grid, hipStream_t s, const PfArgs &a);   // kPfScaleH
int launch_prefill_0_3(int qtype, dim3 grid, hipStream_t s, const PfArgs &a);   // kPfRoundGU | kPfScaleH
int launch_prefill_1_0(int qtype, dim3 grid, hipStream_t s, const PfArgs &a);   // down, bf16 y
int launch_prefill_1_4(int qtype, dim3 grid, hipStream_t s, const PfArgs &a);   // down, f32 y

}  // namespace mi

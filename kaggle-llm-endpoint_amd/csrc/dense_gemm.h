// Dense GEMM of many tokens against int8 or bf16 weights on the gfx950 matrix cores: the gate/up and down products of
// mlp_partial (model.py:125-127) for more tokens than the streaming kernels of int8_project.hip take at once (32; the
// single projections take them 32 at a time).  Those read every weight once per 32 tokens; here a workgroup's weight tile is converted once and meets 64 or
// 128 tokens.
//
// Tile: 128 weight rows (PAIR: 64 of gate and the same 64 of up) x 32 NT tokens x 64 columns, 4 wavefronts as 2 x 2,
// each 64 rows x 16 NT tokens in 16x16x32 tiles.  The weights go through registers, where int8 becomes exactly the
// reference's bf16(f32(q) * s), into LDS beside the bf16 activations; two LDS buffers, so a step's matrix-core work
// overlaps the next step's conversion and the loads of the one after, with one LDS-only barrier per step.  16-byte
// LDS chunk c of row r sits at c ^ (r & 7): the rows of a fragment read fall on different banks without padding.
// Gate and up rows of one output meet in one lane, so the SwiGLU runs on the accumulators.
//
// mlp_partial at D 6144, I 2048, int8 leaves (the 32-token calls before -> these kernels): 512 tokens 481 -> 73 us
// (528 TFLOP/s over the call's two GEMMs and the SwiGLU sums), 1500 tokens about 1440 -> 180 us.  What bounds it now:
// the fragment reads from LDS, 16 KB per wavefront and k-step pair against 32 matrix-core instructions.
//
// With few tiles the columns are split over S workgroups per tile (f32 partials [S, B, n_out], added in split order
// by swiglu_pair_i8 / split_reduce_i8).
#pragma once

namespace mi {

struct DgArgs {
    const uint16_t *x;          // bf16 [B, K]
    int B, K, n_out;            // n_out: rows of each table (PAIR: of gate and of up)
    const int8_t *w[2];         // int8 rows or tiles, or bf16 rows (kW16); PAIR: gate, up; else both the one table
    const float *s[2];          // the tables' scales (MI_I8_*; kW16: unused)
    int tiled;                  // int8 in the layout of mi_int8_tile
    int mt, nt, S;              // weight tiles, token tiles, column splits
    float limit;                // PAIR: the SwiGLU clamp
    uint16_t *h;                // PAIR, S == 1: h [B, n_out]
    uint16_t *y_bf16;           // !PAIR, S == 1: y [B, n_out], either may be null
    float *y_f32;
    float *part[2];             // S > 1: [S, B, n_out] of gate and up (PAIR), of the table (else part[0])
};

constexpr int kDgRows = 128;    // weight rows per tile
constexpr int kDgCols = 64;     // columns per step

template <int SA, bool PAIR, int NT>
__global__ void __launch_bounds__(256, 2) dense_gemm_kernel(DgArgs a) {
    constexpr bool W16 = SA == kW16;
    constexpr int kPieces = W16 ? 4 : 2;        // 16-byte weight pieces per thread and step
    constexpr int kTok = 32 * NT;               // tokens per tile
    __shared__ uint4 wl[2][kDgRows * 8], xl[2][kTok * 8];
    // workgroups go to the XCDs round-robin: the token tiles of one (weight tile, split) sit 8 apart, on one XCD, and
    // share its weights through that L2
    const int xcd = blockIdx.x % 8, li = blockIdx.x / 8;
    const int nti = li % a.nt, g = (li / a.nt) * 8 + xcd;
    if (g >= a.mt * a.S) return;
    const int mti = g % a.mt, split = g / a.mt;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave & 1, wn = wave >> 1;
    const int nsteps = a.K / kDgCols;
    const int t0 = split * nsteps / a.S, t1 = (split + 1) * nsteps / a.S;
    const int tok0 = nti * kTok;
    const int row0 = mti * (PAIR ? kDgRows / 2 : kDgRows);   // first row of the tile in its table(s)

    // ---- weight pieces: piece j of a thread is 16 bytes of LDS row wr[j]; table j / (kPieces / 2) of a pair
    const int K = a.K, rt = a.n_out / 16;
    int wr[kPieces], wc[kPieces], voff[kPieces];
#pragma unroll
    for (int j = 0; j < kPieces; ++j) {
        if (W16) {                               // 8 lanes per row: 128 contiguous bytes
            wr[j] = (tid >> 3) + 32 * j;
            wc[j] = tid & 7;
            voff[j] = (PAIR ? wr[j] & 63 : wr[j]) * 2 * K + 16 * wc[j];
        } else if (a.tiled) {                    // lane i + 16 q of half h of row tile t: columns 32 q + 16 h
            const int t = (tid >> 6) + 4 * j, hh = (tid >> 5) & 1, qs = (tid >> 4) & 1, i = tid & 15;
            wr[j] = 16 * t + i;
            wc[j] = 2 * (2 * qs + hh);
            voff[j] = ((PAIR ? t & 3 : t) * 2 + hh) * 1024 + (i + 16 * qs) * 16;
        } else {                                 // 4 lanes per row: 64 contiguous bytes
            wr[j] = (tid >> 2) + 64 * j;
            wc[j] = 2 * (tid & 3);
            voff[j] = (PAIR ? wr[j] & 63 : wr[j]) * K + 8 * wc[j];
        }
    }
    __amdgpu_buffer_rsrc_t wb[2];
    const float *sp[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        const int8_t *base = a.w[m] + (a.tiled ? (size_t)(row0 / 16) * 2048 : (size_t)row0 * K * (W16 ? 2 : 1));
        wb[m] = __builtin_amdgcn_make_buffer_rsrc((void *)base, (short)0, 0x7fffffff, kBufWord3);
        sp[m] = a.s[m];
    }
    float sc[kPieces], ns128[kPieces];           // the per-row scale of every piece
#pragma unroll
    for (int j = 0; j < kPieces; ++j) {
        sc[j] = SA == MI_I8_COL_SCALES ? sp[j >= kPieces / 2][row0 + (PAIR ? wr[j] & 63 : wr[j])] : 1.0f;
        ns128[j] = -128.0f * sc[j];
    }
    // ---- activations: 8 lanes per token row; rows past B read row B - 1 (their outputs are not stored)
    const __amdgpu_buffer_rsrc_t xb =
        __builtin_amdgcn_make_buffer_rsrc((void *)(a.x + (size_t)tok0 * K), (short)0, 0x7fffffff, kBufWord3);
    int xoff[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) xoff[j] = min((tid >> 3) + 32 * j, a.B - 1 - tok0) * 2 * K + 16 * (tid & 7);

    uint4 wreg[kPieces], xreg[NT];
    auto load = [&](int t) {
        const int soff = W16 ? 128 * t : a.tiled ? (t >> 1) * rt * 2048 + (t & 1) * 512 : 64 * t;
#pragma unroll
        for (int j = 0; j < kPieces; ++j)
            wreg[j] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(wb[j >= kPieces / 2], voff[j], soff, 0));
#pragma unroll
        for (int j = 0; j < NT; ++j)
            xreg[j] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(xb, xoff[j], 128 * t, 0));
    };
    auto store = [&](int buf, int t) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int r = (tid >> 3) + 32 * j;
            xl[buf][r * 8 + ((tid & 7) ^ (r & 7))] = xreg[j];
        }
#pragma unroll
        for (int j = 0; j < kPieces; ++j) {
            uint4 *row = wl[buf] + wr[j] * 8;
            const int x7 = wr[j] & 7;
            if constexpr (W16) {
                row[wc[j] ^ x7] = wreg[j];
            } else if constexpr (SA == MI_I8_ROW_SCALES) {
                const float4 *f = (const float4 *)(sp[j >= kPieces / 2] + kDgCols * t + 8 * wc[j]);
                row[wc[j] ^ x7] = __builtin_bit_cast(uint4, i8_weights8_rs(wreg[j].x, wreg[j].y, f[0], f[1]));
                row[(wc[j] + 1) ^ x7] = __builtin_bit_cast(uint4, i8_weights8_rs(wreg[j].z, wreg[j].w, f[2], f[3]));
            } else {
                row[wc[j] ^ x7] = __builtin_bit_cast(uint4, i8_weights8(wreg[j].x, wreg[j].y, sc[j], ns128[j]));
                row[(wc[j] + 1) ^ x7] = __builtin_bit_cast(uint4, i8_weights8(wreg[j].z, wreg[j].w, sc[j], ns128[j]));
            }
        }
    };

    f32x4 acc[4][NT];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[r][t] = (f32x4){0.f, 0.f, 0.f, 0.f};
    // row tile r of this wavefront in the LDS tile: PAIR 0, 1 = gate, 2, 3 = up of the same rows
    const int i = lane & 15, q = lane >> 4;
    auto tile_row = [&](int r) { return PAIR ? (r >> 1) * 64 + wm * 32 + (r & 1) * 16 : wm * 64 + 16 * r; };
    auto compute = [&](int buf) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int c = (4 * ks + q) ^ (i & 7);
            uint4 A[4], Bv[NT];
#pragma unroll
            for (int r = 0; r < 4; ++r) A[r] = wl[buf][(tile_row(r) + i) * 8 + c];
#pragma unroll
            for (int t = 0; t < NT; ++t) Bv[t] = xl[buf][(16 * (NT * wn + t) + i) * 8 + c];
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, A[r]),
                                                                        __builtin_bit_cast(bf16x8, Bv[t]), acc[r][t],
                                                                        0, 0, 0);
        }
    };
    load(t0);
    store(0, t0);
    if (t0 + 1 < t1) load(t0 + 1);
    lds_barrier();
    for (int t = t0; t < t1; ++t) {
        const int buf = (t - t0) & 1;
        compute(buf);
        if (t + 1 < t1) {
            store(buf ^ 1, t + 1);               // every wavefront left that buffer one barrier ago
            load(min(t + 2, t1 - 1));
            lds_barrier();
        }
    }

    // lane (i, q) holds outputs 4 q .. 4 q + 3 of each row tile for token 16 t + i
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int b = tok0 + 16 * (NT * wn + t) + i;
        if (b >= a.B) continue;
        if constexpr (PAIR) {
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const int o = row0 + wm * 32 + r * 16 + 4 * q;
                const f32x4 gv = acc[r][t], uv = acc[2 + r][t];
                if (a.S > 1) {
                    const size_t e = ((size_t)split * a.B + b) * a.n_out + o;
                    *(f32x4 *)(a.part[0] + e) = gv;
                    *(f32x4 *)(a.part[1] + e) = uv;
                } else {
                    float hv[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) hv[e] = swiglu_clamped(round_bf16(gv[e]), round_bf16(uv[e]), a.limit);
                    uint2 v;
                    v.x = f32_to_bf16_rne(hv[0]) | (f32_to_bf16_rne(hv[1]) << 16);
                    v.y = f32_to_bf16_rne(hv[2]) | (f32_to_bf16_rne(hv[3]) << 16);
                    *(uint2 *)(a.h + (size_t)b * a.n_out + o) = v;
                }
            }
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int o = row0 + wm * 64 + r * 16 + 4 * q;
                const f32x4 v = acc[r][t];
                if (a.S > 1) {
                    *(f32x4 *)(a.part[0] + ((size_t)split * a.B + b) * a.n_out + o) = v;
                    continue;
                }
                if (a.y_f32) *(f32x4 *)(a.y_f32 + (size_t)b * a.n_out + o) = v;
                if (a.y_bf16) {
                    uint2 p;
                    p.x = f32_to_bf16_rne(v[0]) | (f32_to_bf16_rne(v[1]) << 16);
                    p.y = f32_to_bf16_rne(v[2]) | (f32_to_bf16_rne(v[3]) << 16);
                    *(uint2 *)(a.y_bf16 + (size_t)b * a.n_out + o) = p;
                }
            }
        }
    }
}

}  // namespace mi

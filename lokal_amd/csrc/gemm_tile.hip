// gemm_tile.hip -- the multi-row GEMM for many activation rows (prefill
// chunks, full Batcher steps, the lm_head): Y[b][n] = sum_k X[b][k] W[n][k]
// on v_mfma_f32_16x16x32_f16 with f32-level accuracy, Linear::forward
// (src/model.rs:27-35) over many tokens at once.
//
// Two launches.  x_planes_kernel scales each activation row by a power of
// two (its largest |x| brought into [2^14, 2^15): exact) and splits it once into
// f16 hi + lo, stored in the order the matrix cores read: elements down to 2^-15 of
// the row's largest are held to 2^-24 of themselves, smaller ones to 2^-39 of the
// largest (a row with many of those is marked and takes f32 operands, f32_tile).
// gemm_tile_kernel then multiplies weight tiles against those planes.
// gemm16_kernel, which this replaces for large products, converts the same X
// chunk again in every one of its N / 64 column blocks: that conversion, not
// the MFMAs, bounded it (4864 x 896 Q8_0, 512 rows: 47.6 us = 94 TFLOP/s; here
// 20.4 us + 5.0 for the planes = 176 TFLOP/s).
//
// gemm_tile_kernel: a block of NW waves takes 16 NT NW weight rows x 16 MT
// activation rows over a range of K, 64 columns (a stage) at a time; KG such
// groups of waves share a block's tile, each with every KG-th pair of stages, and
// add up through LDS (four groups, 896 x 896 Q8_0, 512 rows: 9.3 -> 8.2 us).  Every
// load goes straight to LDS (global_load_lds, no registers, RING stages deep):
// the X planes shared by the block, and each wave's own weight rows and scales
// in the order it reads them back.  X is the MFMA's A operand and W its B, so a
// lane's column is one weight row and the block scale is one scalar of it.
// What bounds it: the chain of barrier, LDS reads, widening (ten vector
// instructions per 8 weights, spread over MT tiles), products and scaling (four
// FMAs per MFMA pair), which two to three waves per SIMD go through one after
// another at 1.9-2.2 GHz.  No unit is saturated (counters, 4864 x 896 Q8_0, 512 rows:
// vector instructions issue in 39% of the cycles, MFMAs run in 28%, LDS in 31% without
// bank conflicts; 2048 x 5632 Q4_K, 203 rows: 43 / 30 / 21%).
#include "gemm_impl.h"
#include "gemm_tile.h"

#include <type_traits>

namespace lkt {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 hh2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef unsigned int u4 __attribute__((ext_vector_type(4)));
typedef unsigned int u2 __attribute__((ext_vector_type(2)));

// Column order inside a 32-column block: lane (j = lane >> 4) of an MFMA
// operand holds columns 16 (j & 1) + 8 (j >> 1) .. +7.  A weight lane loads 16
// contiguous bytes (lanes j = 0, 1 one 32-byte block, j = 2, 3 the next), and
// two permlane32_swaps turn the pair of blocks into two operands in this order.
__device__ __forceinline__ void swap_blocks(u4& q) {
    const auto a = __builtin_amdgcn_permlane32_swap(q[0], q[2], false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(q[1], q[3], false, false);
    q[0] = a[0], q[2] = a[1], q[1] = b[0], q[3] = b[1];  // block 0: q[0], q[1]; block 1: q[2], q[3]
}

// 8 bytes + `off` as exact f16: the byte is the low mantissa byte of 1024 + u
__device__ __forceinline__ h8 bytes_h8(uint32_t w0, uint32_t w1, float off) {
    const hh2 bias = {(_Float16)off, (_Float16)off};
    const hh2 q0 = __builtin_bit_cast(hh2, __builtin_amdgcn_perm(0x64646464u, w0, 0x04010400u)) - bias;
    const hh2 q1 = __builtin_bit_cast(hh2, __builtin_amdgcn_perm(0x64646464u, w0, 0x04030402u)) - bias;
    const hh2 q2 = __builtin_bit_cast(hh2, __builtin_amdgcn_perm(0x64646464u, w1, 0x04010400u)) - bias;
    const hh2 q3 = __builtin_bit_cast(hh2, __builtin_amdgcn_perm(0x64646464u, w1, 0x04030402u)) - bias;
    return h8{q0[0], q0[1], q1[0], q1[1], q2[0], q2[1], q3[0], q3[1]};
}

template <int WT>
__device__ __forceinline__ uint32_t row_bytes(uint32_t K) {
    return WT == LK_Q8_0 || WT == LK_Q8_SM ? K : WT == LK_F16 ? 2 * K : K / 2;
}
template <int WT>
__device__ __forceinline__ uint32_t aux_bytes(uint32_t K) {
    return WT == LK_Q8_SM ? K / 2 : WT == LK_F16 ? 0 : K / 16;
}

// 16 (4) bytes per lane from global memory straight to LDS: lane l's to dst + 16 l (4 l)
typedef const __attribute__((address_space(1))) uint32_t* gptr;
typedef __attribute__((address_space(3))) uint32_t* lptr;
__device__ __forceinline__ void dma16(const void* src, void* dst) {
    __builtin_amdgcn_global_load_lds((gptr)src, (lptr)dst, 16, 0, 0);
}
__device__ __forceinline__ void dma4(const void* src, void* dst) {
    __builtin_amdgcn_global_load_lds((gptr)src, (lptr)dst, 4, 0, 0);
}

// A 16 x 16 tile of Y on f32 operands (v_mfma_f32_16x16x4_f32): activation row xr and
// weight row r of this lane (c16), chunks c0 .. c1 of K in sums of their own.  For
// the rows that the planes cannot hold; at an eighth of their rate and without LDS,
// so for nothing else (Q6_K 5632 x 2048, 256 rows: 47 us a call with no row marked, 58
// with one, 168 with all; Q8_0 4864 x 896, 512 rows: 25 / 33 / 116).  One tile at a
// time: four that share a weight load were no faster, and their registers slowed the
// products above (Q6_K 42.5 -> 44.4 us).
template <int WT>
__device__ __forceinline__ f4 f32_tile(const LkDevW& w, uint32_t r, const float* xr, uint32_t K, uint32_t c0,
                                       uint32_t c1, uint32_t j) {
    f4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (uint32_t c = c0; c < c1; c++) {
        const uint32_t k = c * 128 + 32 * j, kb = k < K ? k : K - 32;  // past K: in range, times zero
        lkg::Raw<WT> raw;
        lkg::raw_load(raw, w, r, kb);
        f4 x[8], acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 8; q++) x[q] = *lk_g((const f4*)(xr + kb + 4 * q));
#pragma unroll
        for (int s = 0; s < 4; s++) {
            float wv[8];
            lkg::dequant8<WT>(raw, s, kb, k < K, wv);
#pragma unroll
            for (int e = 0; e < 8; e++)
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(k < K ? x[2 * s + e / 4][e % 4] : 0.f, wv[e], acc, 0, 0, 0);
        }
        sum += acc;
    }
    return sum;
}

template <int WT, int NW, int NT, int MT, bool SW, uint32_t RING, int KG>
// two blocks' waves per SIMD: 256 registers, which also keeps the products out of the accumulation
// registers (moving them back cost 64 instructions a stage)
__global__ __launch_bounds__(64 * NW * KG, 2) void gemm_tile_kernel(const LkGemmArgs a, int mode) {
    constexpr int NO = SW ? NT / 2 : NT;  // output tiles of a wave
    // LDS of one 64-column stage: X planes [row tile][block of 2][plane][lane] for the
    // block, then each wave's own weights in operand order, block scales or
    // super-block heads, and (types with mins) the rows' sums; a ring of RING stages
    constexpr bool SM = WT == LK_Q8_SM, MIN = WT == LK_Q4_K || SM;
    constexpr int WP = WT == LK_Q8_0 || SM ? NT : WT == LK_F16 ? 2 * NT : (NT + 1) / 2;  // weight loads of a wave per stage
    constexpr int AUX = WT == LK_Q8_0 ? 16 : MIN ? 64 + 16 : 0;              // u4 per wave
    constexpr int XU = MT * 256, WU = NW * WP * 64, SU = XU + WU + NW * AUX, XI = MT * 4 / NW;
    constexpr int OPS = XI + WP + (WT == LK_Q8_0 ? 1 : MIN ? 2 : 0);  // loads of a wave per stage
    static_assert(16 * NT <= 64 && XI >= 1 && (!SM || NT <= 2), "one lane per weight row; an X load per wave");
    static_assert((RING & (RING - 1)) == 0 && (RING - 2) * OPS <= 63, "slots by mask; vmcnt holds 6 bits");
    __shared__ __align__(16) u4 rings[KG][RING][SU];
    const int lane = threadIdx.x & 63;
    // KG groups of NW waves take the block's chunks in turn, each with a ring of its own
    const uint32_t kg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) / NW;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) % NW;
    u4(*const ring)[SU] = rings[kg];
    const uint32_t j = (uint32_t)lane >> 4, c16 = (uint32_t)lane & 15;
    const uint32_t K = a.K, nck = (K + 127) / 128, nst = (K + 63) / 64;
    const uint32_t per = (nck + a.ks - 1) / a.ks;
    const uint32_t s_begin = 2 * blockIdx.z * per;
    const uint32_t s_end = s_begin + 2 * per < nst ? s_begin + 2 * per : nst;
    const uint32_t ST = s_begin < s_end ? s_end - s_begin : 0;  // the block's stages
    // the group's i-th pair of stages is the block's pair kg + i KG
    auto stage_of = [&](uint32_t s) { return KG == 1 ? s : (s >> 1) * (2 * KG) + 2 * kg + (s & 1); };
    uint32_t S = ST;
    if constexpr (KG > 1) {
        const uint32_t pairs = ST / 2, left = ST % 2;  // an odd last stage goes to the group next in turn
        S = pairs / KG * 2 + (pairs % KG > kg ? 2 : 0) + (left && pairs % KG == kg ? 1 : 0);
    }
    const uint32_t SI = KG == 1 ? S : (ST + 2 * KG - 1) / (2 * KG) * 2;  // iterations of every group (barriers)
    const uint32_t RT = (a.n_rows + 15) / 16, rt0 = blockIdx.y * MT;

    // The wave's tiles: a uniform base (the tile's first row) and this lane's
    // offset from it for each weight load.  Rows past the last re-read the last
    // one; their outputs are not stored.
    const uint8_t* wd[NT];
    uint32_t ow[NT], on[NT];
    const uint8_t* wa = nullptr;  // this lane's scale / head load: row lane % (16 NT) of the wave's
    uint64_t wq[WT == LK_Q4_K ? WP : 1];  // Q4_K: this lane's source of each two-tile load
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const uint32_t n0 = ((blockIdx.x * NW + wave) * NO + (SW ? t % NO : t)) * 16;
        uint32_t nb = 0;
        const LkSeg* sg = &a.seg[0];
        if constexpr (SW) {
            if (t >= NO) sg = &a.seg[1];
        } else {
            const uint32_t e0 = a.seg[0].w.rows, e1 = e0 + a.seg[1].w.rows;
            if (a.nseg > 1 && n0 >= e0) sg = &a.seg[1], nb = e0;
            if (a.nseg > 2 && n0 >= e1) sg = &a.seg[2], nb = e1;
        }
        const uint32_t rows = sg->w.rows, l0 = n0 - nb < rows ? n0 - nb : rows - 1;
        const uint32_t lr = c16 < rows - l0 ? c16 : rows - 1 - l0;
        wd[t] = sg->w.data + (size_t)l0 * row_bytes<WT>(K);
        on[t] = n0;
        if constexpr (WT == LK_Q4_K) {
            // one load takes two tiles: lanes 32.. the second; 16 of a row's 32 bytes each
            const uint64_t v = (uint64_t)(wd[t] + lr * row_bytes<WT>(K) + 16 * (j & 1));
            if (t % 2 == 0 || lane >= 32) wq[t / 2] = v;
            ow[t] = 0;
        } else {
            ow[t] = lr * row_bytes<WT>(K) + (WT == LK_F16 ? 32 * (j & 1) + 16 * (j >> 1) : 16 * j);
        }
        if constexpr (AUX != 0) {
            const uint8_t* v = sg->w.aux + (size_t)l0 * aux_bytes<WT>(K) + lr * aux_bytes<WT>(K);
            if constexpr (SM) {  // 32 bytes (4 groups) of a row per stage: 16 per lane, lanes 32.. the second tile
                if (t == 0 || lane >= 32) wa = v + 16 * (j & 1);
            } else {
                if (t == 0 || j % NT == (uint32_t)t) wa = v;
            }
        }
    }
    // row tile of the wave's i-th X load, and (types with mins) the source of the rows' sums: row tile wave % MT
    const uint8_t* xb[XI];
#pragma unroll
    for (int i = 0; i < XI; i++) {
        const uint32_t q = wave * XI + i, rt = rt0 + q / 4 < RT ? rt0 + q / 4 : RT - 1;
        xb[i] = (const uint8_t*)a.xp + ((size_t)rt * nck * 8 + q % 4) * 1024;
    }
    const float* xq = nullptr;
    if constexpr (MIN) {
        const uint32_t rt = rt0 + wave % MT < RT ? rt0 + wave % MT : RT - 1;
        xq = a.xsum + (size_t)rt * nck * 128 + lane;
    }
    const uint32_t l16 = lane * 16;
    // all loads of stage s (of this block's range) into its ring slot
    auto stage_load = [&](uint32_t s, u4* slot) {
        const uint32_t g = s_begin + stage_of(s);  // 64-column group
#pragma unroll
        for (int i = 0; i < XI; i++) dma16(xb[i] + (size_t)g * 4096 + l16, slot + (wave * XI + i) * 64);
        u4* const ws = slot + XU + wave * WP * 64;
        u4* const as = slot + XU + WU + wave * AUX;
        if constexpr (WT == LK_F16) {
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (uint32_t b = 0; b < 2; b++) {
                    const uint32_t k = g * 64 + 32 * b;  // past K: column 0, multiplied by zero planes
                    dma16(wd[t] + (size_t)2 * (k < K ? k : 0) + ow[t], ws + (2 * t + b) * 64);
                }
        } else if constexpr (WT == LK_Q8_0 || SM) {
#pragma unroll
            for (int t = 0; t < NT; t++) dma16(wd[t] + (size_t)g * 64 + ow[t], ws + t * 64);
            if constexpr (SM) {
                dma16(wa + g * 32, as);
                dma4(xq + (size_t)g * 64, as + 64);
            } else {
                dma4(wa + g * 4, as);
            }
        } else {
#pragma unroll
            for (int t = 0; t < WP; t++) dma16((const uint8_t*)wq[t] + g * 32, ws + t * 64);
            dma16(wa + (g >> 2) * 16, as);
            dma4(xq + (size_t)g * 64, as + 64);
        }
    };

    f4 y[NT][MT];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int m = 0; m < MT; m++) y[t][m] = f4{0.f, 0.f, 0.f, 0.f};
    // -m and the rows' sums: Q4_K of sub-block j of the chunk, Q8_SM of 16-column group j of the stage
    float mn[NT], xs[MIN ? MT : 1];
#pragma unroll
    for (uint32_t s = 0; s < RING - 1; s++)
        if (s < S) stage_load(s, ring[s]);
    // Stage s has landed when only the loads of the RING - 2 stages after it are
    // in flight (vmcnt counts in order, and every load of the loop is one of
    // OPS per stage); the barrier then says so for every wave, and that all
    // have read the slot that is refilled next.
    auto stage = [&](uint32_t s, auto half) {
        constexpr uint32_t h = decltype(half)::value;
        if (RING > 2 && s + RING - 2 < S) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((RING - 2) * OPS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (s + RING - 1 < S) stage_load(s + RING - 1, ring[RING == 2 ? h ^ 1 : (s + RING - 1) % RING]);
        if (KG > 1 && s >= S) return;  // the barrier only
        const u4* const slot = ring[RING == 2 ? h : s % RING];
        const u4* const ws = slot + XU + wave * WP * 64;
        const u4* const as = slot + XU + WU + wave * AUX;
        float d[NT][SM ? 4 : 2];  // scale of each 32-column block (Q8_SM: of each 16 columns)
        u4 q[NT][WT == LK_F16 ? 2 : 1];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            if constexpr (WT == LK_Q8_0) {
                q[t][0] = ws[t * 64 + lane];
                const uint32_t v = ((const uint32_t*)as)[t * 16 + c16];
                d[t][0] = lk_h2f((uint16_t)(v & 0xFFFF)), d[t][1] = lk_h2f((uint16_t)(v >> 16));
                swap_blocks(q[t][0]);
            } else if constexpr (SM) {
                q[t][0] = ws[t * 64 + lane];
                const u4 g0 = as[t * 32 + c16], g1 = as[t * 32 + 16 + c16];  // (s, m) of groups 0, 1 and 2, 3
                d[t][0] = __uint_as_float(g0[0]), d[t][1] = __uint_as_float(g0[2]);
                d[t][2] = __uint_as_float(g1[0]), d[t][3] = __uint_as_float(g1[2]);
                const uint32_t me = j < 2 ? ((j & 1) ? g0[3] : g0[1]) : ((j & 1) ? g1[3] : g1[1]);
                mn[t] = -__uint_as_float(me);
                swap_blocks(q[t][0]);
            } else if constexpr (WT == LK_F16) {
                q[t][0] = ws[2 * t * 64 + lane];
                q[t][1] = ws[(2 * t + 1) * 64 + lane];
            } else {
                const u2 b = ((const u2*)ws)[2 * ((t / 2) * 64 + (t & 1) * 32 + (j & 1) * 16 + c16) + (j >> 1)];
                q[t][0][0] = b[0], q[t][0][1] = b[1];
                // d1 = d * sc of the stage's two sub-blocks, m1 = dmin * m, each
                // rounded once as dequant_row_ref does (src/gguf/dequant.rs:462-483)
                const u4 hd = as[t * 16 + c16];
                const float ds = lk_h2f((uint16_t)(hd[0] & 0xFFFF)), dm = lk_h2f((uint16_t)(hd[0] >> 16));
                uint32_t sc0, sc1, m0, m1;
                lk::scale_min_k4_pair((s_begin + stage_of(s)) & 3, hd[1], hd[2], hd[3], sc0, m0, sc1, m1);
                d[t][0] = __fmul_rn(ds, (float)sc0), d[t][1] = __fmul_rn(ds, (float)sc1);
                const float mv = -__fmul_rn(dm, (float)((j & 1) ? m1 : m0));
                mn[t] = h == 0 || j >= 2 ? mv : mn[t];  // stage h holds sub-blocks 2h, 2h + 1
            }
        }
        if constexpr (MIN) {
#pragma unroll
            for (int m = 0; m < MT; m++) {
                const float* sm = (const float*)(slot + XU + WU + m * AUX + 64);  // sums of 16 columns: [group][row]
                if constexpr (SM) {
                    xs[m] = sm[j * 16 + c16];
                } else {
                    const float v = sm[(j & 1) * 32 + c16] + sm[(j & 1) * 32 + 16 + c16];
                    xs[m] = h == 0 || j >= 2 ? v : xs[m];
                }
            }
        }
        // both blocks' X operands are read before the first product, so LDS
        // answers while the matrix cores work
        h8 xf[2][MT][2];
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int p = 0; p < 2; p++)
                    xf[b][m][p] = __builtin_bit_cast(h8, slot[(m * 4 + b * 2 + p) * 64 + lane]);
        f4 D[MT][NT];
#pragma unroll
        for (int b = 0; b < 2; b++) {
            h8 w[NT];
#pragma unroll
            for (int t = 0; t < NT; t++) {
                if constexpr (WT == LK_Q8_0 || SM)
                    w[t] = bytes_h8(q[t][0][2 * b] ^ 0x80808080u, q[t][0][2 * b + 1] ^ 0x80808080u, 1152.0f);
                else if constexpr (WT == LK_F16)
                    w[t] = __builtin_bit_cast(h8, q[t][b]);
                else
                    w[t] = bytes_h8((q[t][0][0] >> (4 * b)) & 0x0F0F0F0Fu, (q[t][0][1] >> (4 * b)) & 0x0F0F0F0Fu, 1024.0f);
            }
            if constexpr (SM) {
                // a 32-column block holds two groups with scales of their own: lanes j = 0, 2 the
                // first, 1, 3 the second, the other's weights zero
                const uint32_t keep0 = (j & 1) ? 0u : ~0u;
#pragma unroll
                for (int gq = 0; gq < 2; gq++) {
                    h8 wg[NT];
#pragma unroll
                    for (int t = 0; t < NT; t++) {
                        u4 v = __builtin_bit_cast(u4, w[t]);
#pragma unroll
                        for (int e = 0; e < 4; e++) v[e] &= gq ? ~keep0 : keep0;
                        wg[t] = __builtin_bit_cast(h8, v);
                    }
#pragma unroll
                    for (int m = 0; m < MT; m++)
#pragma unroll
                        for (int p = 0; p < 2; p++)
#pragma unroll
                            for (int t = 0; t < NT; t++)
                                D[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[b][m][p], wg[t], p ? D[m][t] : f4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                    for (int m = 0; m < MT; m++)
#pragma unroll
                        for (int t = 0; t < NT; t++)
#pragma unroll
                            for (int i = 0; i < 4; i++) y[t][m][i] = fmaf(d[t][2 * b + gq], D[m][t][i], y[t][m][i]);
                }
                continue;
            }
#pragma unroll
            for (int m = 0; m < MT; m++) {
#pragma unroll
                for (int p = 0; p < 2; p++)
#pragma unroll
                    for (int t = 0; t < NT; t++)
                        D[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                            xf[b][m][p], w[t], p || (WT == LK_F16 && b) ? D[m][t] : f4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            }
            if constexpr (WT != LK_F16) {
#pragma unroll
                for (int m = 0; m < MT; m++)
#pragma unroll
                    for (int t = 0; t < NT; t++)
#pragma unroll
                        for (int i = 0; i < 4; i++) y[t][m][i] = fmaf(d[t][b], D[m][t][i], y[t][m][i]);
            }
        }
        // F16 has no scales, but a stage's sums of their own keep the error of an unsplit deep
        // K down (1536 columns: 3.4e-7 with one running product, 1.3e-7 so)
        if constexpr (WT == LK_F16) {
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (int i = 0; i < 4; i++) y[t][m][i] += D[m][t][i];
        }
        // the sums stay where they are: sunk to a later block by the
        // compiler, every product would be held until then
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int m = 0; m < MT; m++) asm volatile("" : "+v"(y[t][m]));
        if constexpr (SM || (WT == LK_Q4_K && h == 1)) {
            // minus m * sum(x) per sub-block or group: four of them are one f32 MFMA
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int t = 0; t < NT; t++)
                    y[t][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(xs[m], mn[t], y[t][m], 0, 0, 0);
        }
    };
#pragma unroll 1
    for (uint32_t s = 0; s < SI; s += 2) {
        stage(s, std::integral_constant<uint32_t, 0>{});
        if (KG > 1 || s + 1 < S) stage(s + 1, std::integral_constant<uint32_t, 1>{});
    }
    if constexpr (KG > 1) {
        // the groups' sums, through LDS, into group 0's in turn
        f4* const acc = (f4*)&rings[0][0][0];
        static_assert(sizeof(rings) >= (size_t)(KG - 1) * NW * NT * MT * 64 * 16, "the sums fit the rings");
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (kg)
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int m = 0; m < MT; m++) acc[((((kg - 1) * NW + wave) * NT + t) * MT + m) * 64 + lane] = y[t][m];
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (kg) return;
#pragma unroll
        for (int g = 0; g < KG - 1; g++)
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int m = 0; m < MT; m++) y[t][m] += acc[(((g * NW + wave) * NT + t) * MT + m) * 64 + lane];
    }

    // lane: rows 4j + i of each row tile, output on[t] + c16.  A K split leaves
    // its partial sums, else the bias, residual or SwiGLU epilogue runs here
    // (src/model.rs:27-35, :235-237, :247-249).
    const bool part = a.ks > 1;
    const size_t np = part ? (SW ? 2 * (size_t)a.N : a.N) : a.ldy;
    const uint32_t r0 = rt0 * 16;
    f4 s4[MT];
#pragma unroll
    for (int m = 0; m < MT; m++) {
        const uint32_t rt = rt0 + m < RT ? rt0 + m : RT - 1;
        s4[m] = *lk_g((const f4*)(a.xsc + rt * 16 + 4 * j));
    }
    // row tiles with marked rows, by scalar loads
    uint32_t marked = 0;
#pragma unroll
    for (int m = 0; m < MT; m++) {
        const uint32_t rt = rt0 + m < RT ? rt0 + m : RT - 1;
        const auto mk = (const __attribute__((address_space(4))) uint64_t*)(uintptr_t)(a.xmark + (size_t)rt * 16);
        if (mk[0] | mk[1]) marked |= 1u << m;
    }
    if (marked) {  // those rows again on f32 operands, whose sums need no scale
#pragma unroll 1
        for (uint32_t q = 0; q < NT * MT; q++) {
            const uint32_t t = q / MT, m = q % MT;
            if (!(marked >> m & 1)) continue;
            const uint32_t n0 = ((blockIdx.x * NW + wave) * NO + (SW ? t % NO : t)) * 16;
            const uint32_t rt = rt0 + m < RT ? rt0 + m : RT - 1, row = rt * 16 + c16;
            uint32_t si = SW && t >= NO ? 1 : 0, nb = 0;
            while (!SW && si + 1 < a.nseg && n0 >= nb + a.seg[si].w.rows) nb += a.seg[si++].w.rows;
            const LkDevW& w = a.seg[si].w;
            const uint32_t wr = n0 - nb + c16, mk = *lk_g((const uint32_t*)(a.xmark + rt * 16 + 4 * j));
            const f4 v = f32_tile<WT>(w, wr < w.rows ? wr : w.rows - 1,
                                      a.x + (size_t)(row < a.n_rows ? row : a.n_rows - 1) * a.ldx, K, s_begin / 2,
                                      (s_end + 1) / 2, j);
#pragma unroll
            for (int mm = 0; mm < MT; mm++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if (m != (uint32_t)mm || !(mk >> 8 * i & 1)) continue;
                    s4[mm][i] = 1.f;
#pragma unroll
                    for (int tt = 0; tt < NT; tt++) y[tt][mm][i] = t == (uint32_t)tt ? v[i] : y[tt][mm][i];
                }
        }
    }
    const bool acc = !SW && !part && mode == LK_MV_ACC;
    // GUARD: the block's last rows lie past n_rows
    auto store = [&](auto guard) {
        constexpr bool GUARD = decltype(guard)::value;
#pragma unroll
        for (int t = 0; t < NO; t++) {
            uint32_t nb = 0;
            const LkSeg* sg = &a.seg[0];
            if constexpr (!SW) {
                const uint32_t e0 = a.seg[0].w.rows, e1 = e0 + a.seg[1].w.rows;
                if (a.nseg > 1 && on[t] >= e0) sg = &a.seg[1], nb = e0;
                if (a.nseg > 2 && on[t] >= e1) sg = &a.seg[2], nb = e1;
            }
            // this lane's first row and output; the other rows are uniform steps of np from it, in 64
            // bits: 63 rows of 68.2 million floats (ldy is the caller's) pass 2^32
            float* const base = (part ? a.part + (size_t)blockIdx.z * a.n_rows * np + on[t] : sg->out + (on[t] - nb)) +
                                (size_t)(r0 + 4 * j) * np + c16;
            if (on[t] + c16 >= a.N) continue;
            const float bias = !part && sg->bias ? sg->bias[on[t] - nb + c16] : 0.f;
            float old[MT][4];
            if (acc) {
#pragma unroll
                for (int m = 0; m < MT; m++)
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        old[m][i] = !GUARD || r0 + 16 * m + 4 * j + i < a.n_rows ? *lk_g(base + (16 * m + i) * np) : 0.f;
            }
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if (GUARD && r0 + 16 * m + 4 * j + i >= a.n_rows) continue;
                    float* const ob = base + (16 * m + i) * np;
                    float v = y[t][m][i] * s4[m][i];
                    if constexpr (SW) {
                        const float u = y[t + NO][m][i] * s4[m][i];
                        if (part) ob[a.N] = u;
                        else v = lkg::silu_mul(v, u);
                    } else {
                        v += bias;
                        if (acc) v += old[m][i];
                    }
                    *ob = v;
                }
        }
    };
    if (r0 + 16 * MT <= a.n_rows) store(std::false_type{});
    else store(std::true_type{});
}

// One lane's 8 scaled columns (group g) to the planes, and with `xsum` their sum with
// the neighbour's; all lanes of the wave call it (the sums cross lanes)
__device__ __forceinline__ void store_group(const float* o, uint32_t g, uint32_t rt, uint32_t rr, uint32_t nck,
                                            u4* xp, float* xsum) {
    if (g < nck * 16) lk_store_planes(xp, rt, rr, nck, g, o);
    if (xsum) {
        float s = ((o[0] + o[1]) + (o[2] + o[3])) + ((o[4] + o[5]) + (o[6] + o[7]));
        s += __shfl_xor(s, 1, 64);
        if (g % 2 == 0 && g < nck * 16) xsum[((size_t)rt * nck * 8 + g / 2) * 16 + rr] = s;
    }
}

// Four activation rows per block, WPR waves each (rows past the last, up to a
// whole 16-row tile, are zero): the row's power-of-two scale, its f16 planes
// in MFMA order [row tile][chunk][block][plane][lane], the scale that undoes
// it, its mark (lk_row_score), and with `xsum` the row's scaled sum over every 16 columns (the Q4_K and Q8_SM
// min terms).  A lane holds its G groups of 8 columns from the load to the
// store (G = 0: a row too wide for that is read twice).  The four rows' 16-byte
// pieces of a 64-byte line leave one CU together; one row per block
// wrote each line from four XCDs.  512 rows of 4864: 11.0 -> 7.6 us.
template <int WPR, int G>
__global__ __launch_bounds__(256 * WPR) void x_planes_kernel(const float* __restrict__ x, uint32_t ldx, uint32_t n_rows,
                                                             uint32_t K, u4* __restrict__ xp, float* __restrict__ xsc,
                                                             float* __restrict__ xsum, uint8_t* __restrict__ xmark) {
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t r = blockIdx.x * 4 + wave / WPR, nck = (K + 127) / 128, rt = r / 16, rr = r % 16;
    const uint32_t t = (wave % WPR) * 64 + (threadIdx.x & 63);  // lane of the row's 64 * WPR
    __shared__ float red[4][WPR];
    __shared__ int cnt[4][WPR];
    const bool live = r < n_rows;
    const float* xr = x + (size_t)(live ? r : 0) * ldx;
    float v[G ? G : 1][8];
    auto load = [&](float* o, uint32_t g) {
        const uint32_t k = 8 * g;  // K is a multiple of 32: a group is whole or past it
        const f4 a = *lk_g((const f4*)(xr + (k < K ? k : 0))), b = *lk_g((const f4*)(xr + (k < K ? k : 0) + 4));
#pragma unroll
        for (int e = 0; e < 4; e++) {
            o[e] = live && k < K ? a[e] : 0.f;
            o[4 + e] = live && k < K ? b[e] : 0.f;
        }
    };
    auto most = [&](const float* o, float mx) {
#pragma unroll
        for (int e = 0; e < 8; e++) mx = fmaxf(mx, fabsf(o[e]));
        return mx;
    };
    float mx = 0.f;
    if constexpr (G != 0) {
#pragma unroll
        for (int i = 0; i < G; i++) load(v[i], t + 64 * WPR * i);
#pragma unroll
        for (int i = 0; i < G; i++) mx = most(v[i], mx);
    } else {
        for (uint32_t g = t; g < nck * 16; g += 64 * WPR) {
            load(v[0], g);
            mx = most(v[0], mx);
        }
    }
    mx = lk_wave_max(mx);
    if constexpr (WPR > 1) {
        if ((threadIdx.x & 63) == 0) red[wave / WPR][wave % WPR] = mx;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < WPR; i++) mx = fmaxf(mx, red[wave / WPR][i]);
    }
    float inv, sc;
    lk_row_scale(mx, inv, sc);
    int score = 0;
    auto store = [&](float* o, uint32_t g) {
#pragma unroll
        for (int e = 0; e < 8; e++) o[e] *= inv;
        store_group(o, g, rt, rr, nck, xp, xsum);
        score += lk_row_score(o);
    };
    if constexpr (G != 0) {
#pragma unroll
        for (int i = 0; i < G; i++) store(v[i], t + 64 * WPR * i);
    } else {
        for (uint32_t g0 = 0; g0 < nck * 16; g0 += 64 * WPR) {  // uniform: the sums cross lanes
            load(v[0], g0 + t);
            store(v[0], g0 + t);
        }
    }
    if constexpr (WPR > 1) {
        if ((threadIdx.x & 63) == 0) cnt[wave / WPR][wave % WPR] = score;
        __syncthreads();
        score = 0;
#pragma unroll
        for (int i = 0; i < WPR; i++) score += cnt[wave / WPR][i];
    }
    if (t == 0) {
        xsc[r] = sc;
        xmark[r] = lk_row_marked(mx, score);
    }
}

// rows_accnorm_kernel's work -- x += the split-K partials, then RMSNorm -- with
// the normalised row written as planes only, RPB rows per block, WPR waves per
// row, a lane holding its 8 columns throughout.  The float row that
// x_planes_kernel would read back is stored (y) for marked rows only: 512 rows of 896, 5.4 us for
// rows_accnorm_kernel + 4.5 for the planes -> 5.6 (3.3 without partials, 7-8 with
// eight, whose 14.7 MB then bound it).  Four rows per block, as their pieces make whole
// 64-byte lines (two: 5.9 us); wider rows two, which keeps a block to 1024 threads.
template <int RPB, int WPR>
__global__ __launch_bounds__(64 * RPB * WPR) void rows_accnorm_planes_kernel(
    float* __restrict__ x, const float* __restrict__ part, uint32_t ks, uint32_t n_rows, uint32_t K,
    const float* __restrict__ w, float eps, float* __restrict__ y, u4* __restrict__ xp, float* __restrict__ xsc,
    float* __restrict__ xsum, uint8_t* __restrict__ xmark) {
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), row = wave / WPR;
    const uint32_t r = blockIdx.x * RPB + row, nck = (K + 127) / 128;
    const uint32_t g = (wave % WPR) * 64 + (threadIdx.x & 63), k = 8 * g < K ? 8 * g : 0;  // K is a multiple of 32
    const bool in = r < n_rows && 8 * g < K;
    __shared__ float red[3][RPB][WPR];
    const size_t at = (size_t)(r < n_rows ? r : 0) * K + k;
    f4 v[2], wt[2];
#pragma unroll
    for (int c = 0; c < 2; c++) {
        v[c] = *lk_g((const f4*)(x + at + 4 * c));
        wt[c] = *lk_g((const f4*)(w + k + 4 * c));
    }
    if (ks) {  // in split order, as gemm_reduce_kernel would, eight splits' loads in flight
        const size_t stride = (size_t)n_rows * K;
        f4 a[2] = {};
        for (uint32_t z0 = 0; z0 < ks; z0 += 8) {
            f4 p[8][2];
#pragma unroll
            for (uint32_t z = 0; z < 8; z++)
#pragma unroll
                for (int c = 0; c < 2; c++)
                    p[z][c] = *lk_g((const f4*)(part + at + (size_t)(z0 + z < ks ? z0 + z : z0) * stride + 4 * c));
#pragma unroll
            for (uint32_t z = 0; z < 8; z++)
                if (z0 + z < ks) a[0] += p[z][0], a[1] += p[z][1];
        }
#pragma unroll
        for (int c = 0; c < 2; c++) {
            v[c] += a[c];
            if (in) *(f4*)(x + at + 4 * c) = v[c];
        }
    }
    auto across = [&](float u, float* rd, auto op) {  // the row's WPR waves
        if constexpr (WPR > 1) {
            if ((threadIdx.x & 63) == 0) rd[wave % WPR] = u;
            __syncthreads();
            u = rd[0];
#pragma unroll
            for (int i = 1; i < WPR; i++) u = op(u, rd[i]);
        }
        return u;
    };
    float o[8], ss = 0.f, mx = 0.f;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        o[e] = in ? v[e / 4][e % 4] : 0.f;
        ss = fmaf(o[e], o[e], ss);
    }
    ss = across(lk_wave_sum(ss), red[0][row], [](float a, float b) { return a + b; });
    const float scale = 1.0f / sqrtf(ss / (float)K + eps);
#pragma unroll
    for (int e = 0; e < 8; e++) {
        o[e] = in ? __fmul_rn(__fmul_rn(o[e], scale), wt[e / 4][e % 4]) : 0.f;
        mx = fmaxf(mx, fabsf(o[e]));
    }
    mx = across(lk_wave_max(mx), red[1][row], [](float a, float b) { return fmaxf(a, b); });
    float inv, sc;
    lk_row_scale(mx, inv, sc);
    float p[8];
#pragma unroll
    for (int e = 0; e < 8; e++) p[e] = o[e] * inv;
    store_group(p, g, r / 16, r % 16, nck, xp, xsum);
    const float score = across((float)lk_row_score(p), red[2][row], [](float a, float b) { return a + b; });
    const bool mark = lk_row_marked(mx, (int)score);
    if (g == 0) {
        xsc[r] = sc;
        xmark[r] = mark;
    }
    if (mark && in) {
        *(f4*)(y + at) = f4{o[0], o[1], o[2], o[3]};
        *(f4*)(y + at + 4) = f4{o[4], o[5], o[6], o[7]};
    }
}

template <int WT, int NW, int NT, int MT, bool SW, uint32_t RING, int KG = 1>
static hipError_t launch(const LkGemmArgs& a, int mode, hipStream_t st) {
    constexpr uint32_t BN = 16 * NW * (SW ? NT / 2 : NT);
    const dim3 grid((a.N + BN - 1) / BN, (a.n_rows + 16 * MT - 1) / (16 * MT), a.ks);
    hipLaunchKernelGGL((gemm_tile_kernel<WT, NW, NT, MT, SW, RING, KG>), grid, dim3(64 * NW * KG), 0, st, a, mode);
    return hipGetLastError();
}

// The instances tile_plan chooses from, by its names for them.
template <int WT>
static hipError_t launch_t(const LkGemmArgs& a, int mode, uint32_t kind, hipStream_t st) {
    constexpr bool ONE = WT == LK_F16;  // no wave groups
    if (mode == LK_MV_SWIGLU) {
        if (kind == LK_TILE_SMALL) return launch<WT, 4, 2, 2, true, 2, ONE ? 1 : 2>(a, mode, st);
        if (kind == LK_TILE_DEEP) return launch<WT, 2, 2, 2, true, 2, 4>(a, mode, st);
        return launch<WT, 4, 2, 4, true, 2>(a, mode, st);
    }
    switch (kind) {
    case LK_TILE_SMALL: return launch<WT, 4, 1, 2, false, ONE ? 4 : 2, ONE ? 1 : 2>(a, mode, st);
    case LK_TILE_MID:
        if constexpr (WT != LK_Q8_SM) return launch<WT, 4, 1, 4, false, 2>(a, mode, st);
        return hipErrorInvalidValue;
    case LK_TILE_LARGE: return launch<WT, 4, 2, 4, false, 2>(a, mode, st);
    case LK_TILE_SPLIT: return launch<WT, 8, 2, 4, false, 2>(a, mode, st);
    case LK_TILE_DEEP:
        if constexpr (!ONE) return launch<WT, 4, 1, 2, false, 2, 4>(a, mode, st);
        return hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
    }
}

}  // namespace lkt

hipError_t lk_planes_launch(const float* x, uint32_t ldx, uint32_t n_rows, uint32_t K, bool sums, void* planes,
                            hipStream_t st) {
    const LkPlanes p = lk_planes_at(planes, n_rows, K);
    const uint32_t groups = (K + 127) / 128 * 16;
    const dim3 grid((n_rows + 15) / 16 * 4);
    float* const xsum = sums ? p.xsum : nullptr;
#define LK_XP(wpr, g)                                                                                                \
    hipLaunchKernelGGL((lkt::x_planes_kernel<wpr, g>), grid, dim3(256 * wpr), 0, st, x, ldx, n_rows, K, (lkt::u4*)p.xp, \
                       p.xsc, xsum, p.mark)
    if (groups <= 64) LK_XP(1, 1);
    else if (groups <= 128) LK_XP(1, 2);
    else if (groups <= 256) LK_XP(4, 1);
    else if (groups <= 512) LK_XP(4, 2);
    else if (groups <= 768) LK_XP(4, 3);
    else LK_XP(4, 0);
#undef LK_XP
    return hipGetLastError();
}

hipError_t lk_rows_accnorm_planes_launch(float* x, const float* part, uint32_t ks, uint32_t rows, uint32_t n,
                                         const float* w, float eps, float* y, bool sums, void* planes,
                                         hipStream_t st) {
    if (rows == 0) return hipSuccess;
    if (!lk_accnorm_planes_ok(n)) return hipErrorInvalidValue;
    const LkPlanes p = lk_planes_at(planes, rows, n);
    const uint32_t groups = (n + 127) / 128 * 16, up = (rows + 15) / 16 * 16;
    float* const xsum = sums ? p.xsum : nullptr;
#define LK_NP(rpb, wpr)                                                                                     \
    hipLaunchKernelGGL((lkt::rows_accnorm_planes_kernel<rpb, wpr>), dim3(up / rpb), dim3(64 * rpb * wpr), 0, st, x, \
                       part, ks, rows, n, w, eps, y, (lkt::u4*)p.xp, p.xsc, xsum, p.mark)
    if (groups <= 64) LK_NP(4, 1);
    else if (groups <= 128) LK_NP(4, 2);
    else if (groups <= 256) LK_NP(2, 4);
    else LK_NP(2, 8);
#undef LK_NP
    return hipGetLastError();
}

hipError_t lk_tile_launch(LkGemmArgs a, int mode, const LkTilePlan& p, hipStream_t st) {
    const LkPlanes pl = lk_planes_at(a.planes, a.n_rows, a.K);
    a.xp = pl.xp;
    a.xsc = pl.xsc;
    a.xsum = pl.xsum;
    a.xmark = pl.mark;
    switch (a.seg[0].w.type) {
    case LK_Q8_0: return lkt::launch_t<LK_Q8_0>(a, mode, p.kind, st);
    case LK_F16: return lkt::launch_t<LK_F16>(a, mode, p.kind, st);
    case LK_Q4_K: return lkt::launch_t<LK_Q4_K>(a, mode, p.kind, st);
    case LK_Q8_SM: return lkt::launch_t<LK_Q8_SM>(a, mode, p.kind, st);
    default: return hipErrorInvalidValue;
    }
}

// gemm.hip -- the M > 1 GEMM of the packed matrices: the MFMA slab GEMM
// (k_gemm_mfma) and the K-split GEMMs for up to 16 rows (k_gemm_sk,
// k_gemm_skp), with their launch planning.
//
// Numerics contract: every kernel reproduces the fp32 operation order of the
// reference CPU path (dpuf_avx2.c / dpuf_engine.c in dulePan/dpuf) so that
// results are bit-identical, not merely close:
//   * integer parts (nibble x int8 dots) are exact in any order, so they are
//     spread over lanes and reduced with DPP;
//   * every floating-point reduction whose order the reference fixes (the
//     per-row FMA chain over 32-blocks, RMSNorm's 8 FMA lanes + hsum tree,
//     attention's hadd tree, softmax sums, the P.V chain) runs in that order;
//   * build with -ffp-contract=off; fused multiply-adds are explicit fmaf.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "hip_layer.h"
#include "dev_common.h"
#include "hip_internal.h"

// M > 16 GEMM on the matrix cores (slab path, dpuf_avx2.c:2643-2676): k_gemm_mfma
// (16 x 16 tiles) and k_gemm_x32 (32 x 32 tiles).
//
// For every (row, token) the reference accumulates every block:
//   acc = fma(float(D - sum8), fp16(ws) * xs, acc), blocks ascending,
// with D the u4 x i8 dot of the block and sum8 = 8 * sum(q).  D - sum8 =
// sum((u - 8) * q), so one int8 MFMA per block and tile gives it exactly; the
// epilogue is the reference's two rounded operations with the chains in
// registers across the block loop, so the block order is the reference's.
//
// What bounds both is instructions per tile and block (the chains leave 12
// per 256 outputs that no matrix instruction can take) and, in order in a
// wave, the latencies between them.  So:
//   * A = 16 (u - 8), one v_bitop3 per 4 nibbles (the nibble's top bit
//     flipped, in a byte's upper half), 3 instructions per nibble word where
//     u - 8 as fp16 took 11;
//   * the MFMA's C is the bit pattern of a float in every element (gm_base: 1.5
//     2^19, whose last mantissa bit is worth 1 / 16; modes 13 / 14, whose u
//     needs no offset and no factor, 1.5 2^23, whose last bit is worth 1).
//     Sums of magnitude up to 2^19 stay inside that binade, so the result read
//     as a float is the base plus the dot exactly, and one exact subtraction
//     gives the dot at full rate (v_cvt_f32_i32 issues at half);
//   * mode 12's products ws * xs come from 4 x 4 outer-product MFMAs (one for
//     256 outputs in place of 4 v_mul_f32; gm_outer4), issued with the dots
//     before any result is read: the chains are left with one subtraction and
//     one FMA per output.  (With the products on the vector unit down M = 29
//     32 us, 27 so, M = 512 119 and 108.  Left to the compiler's order, which
//     waits for each product in turn, they gained nothing.)
//   * weight scales are widened to float once per workgroup when they are
//     staged (v_fma_mix_f32 issues at half rate).
// Dots, products and chains have the reference's own values, so they overflow
// where its do.
//
// Activations (int8, token scales) and weight scales are staged in LDS a
// stage of several blocks at a time, double-buffered, one barrier per stage.
// LDS rows of a block are padded so that the staging writes of consecutive
// blocks fall into different banks (unpadded: 8-way conflicts).  Weight
// nibbles are read straight into a register ring several quads ahead, 16
// bytes per lane, and exchanged between the wave's lane rows into the MFMA
// layout.  MFMA lane layouts (gfx950, checked on the device): 16x16x32: A / B
// lane l = row / token l % 16, k = 8 (l / 16) + e; D lane l = token l % 16,
// rows 4 (l / 16) + v.  32x32x32: A / B lane l = row l % 32, k = 16 (l / 32) +
// e; D lane l = column l % 32, rows 8 (v / 4) + 4 (l / 32) + v % 4.
//
// us per launch at the 8B widths, before (one 16-row x 64-token fp16 tile per
// wave for every M) -> now: down M = 29 85 -> 27, M = 90 93 -> 37, M = 512 144
// -> 108; O 30 -> 11, 31 -> 15, 47.5 -> 38; mode 14 down M = 90 135 -> 50, M =
// 512 223 -> 145; gate + up with the SwiGLU M = 512 202 -> 178.
// ---------------------------------------------------------------------------

#define GM_SWI_ROWS 16384  // gate + up rows from which the fused SwiGLU launch pays
#define GM_RSRC3 0x00020000  // buffer descriptor word 3 (gfx9 family): 32-bit raw data

struct GmJob {
    const uint8_t* g;  // dense groups of the matrix
    int g0, g1;        // groups computed
    int rows;
    const uint16_t* h;  // activations as fp16 [M][K] (K-split kernels)
    const int8_t* q;    // activations as int8 [M][K]
    const float* s;     // block scales [M][K/32]
    const int32_t* m;   // 8 * block sums of q [M][K/32] (modes 13 / 14)
    float* out;        // out[m * ldo + row]
    int ldo;
};

struct GmArgs {
    GmJob j[3];
    int n_jobs;
    int tb[4];  // prefix sums of the jobs' row tiles (workgroups or fragments of the kernel)
    int K, M;
    int gy;     // token tiles
    // rows [z0, z1) of zo (row stride zld) set to 0 by zt extra row tiles of
    // 64 rows placed after the jobs' tiles
    float* zo;
    int zld, z0, z1, zt;
    int32_t* err;  // device error word: set when a bounded wait of k_gemm_sk runs out
    // gate + up with the SwiGLU (the SWI instances): the prep of the
    // down projection's input [M][swI] goes to swo, with the down input's
    // sign bits swsign and dead zone swdz
    DpufPrep swo;
    const uint8_t* swsign;
    float swdz;
    int swI;
};


// A fragment from one nibble word (row i, columns 8 kc .. 8 kc + 7 of a
// block: low nibbles = columns +0..+3, high nibbles = +4..+7): u - 8 as f16.
DEV gm_h8 gm_unpack_a(uint32_t w) {
    const uint32_t lo = w & 0x0F0F0F0Fu, hi = (w >> 4) & 0x0F0F0F0Fu;
    const uint32_t r0 = gm_sub(gm_pair(lo, 0x04010400u), (_Float16)1032.0f);
    const uint32_t r1 = gm_sub(gm_pair(lo, 0x04030402u), (_Float16)1032.0f);
    const uint32_t r2 = gm_sub(gm_pair(hi, 0x04010400u), (_Float16)1032.0f);
    const uint32_t r3 = gm_sub(gm_pair(hi, 0x04030402u), (_Float16)1032.0f);
    return __builtin_bit_cast(gm_h8, make_uint4(r0, r1, r2, r3));
}

// The same for modes 13 / 14: u itself (no offset) as f16, with bits 4..5
// from h (bits 0-1 of byte k for the low half, 2-3 for the high half; 0 for
// mode 13).
DEV gm_h8 gm_unpack_a_asym(uint32_t w, uint32_t h) {
    const uint32_t lo = (w & 0x0F0F0F0Fu) | ((h & 0x03030303u) << 4);
    const uint32_t hi = ((w >> 4) & 0x0F0F0F0Fu) | (((h >> 2) & 0x03030303u) << 4);
    const uint32_t r0 = gm_sub(gm_pair(lo, 0x04010400u), (_Float16)1024.0f);
    const uint32_t r1 = gm_sub(gm_pair(lo, 0x04030402u), (_Float16)1024.0f);
    const uint32_t r2 = gm_sub(gm_pair(hi, 0x04010400u), (_Float16)1024.0f);
    const uint32_t r3 = gm_sub(gm_pair(hi, 0x04030402u), (_Float16)1024.0f);
    return __builtin_bit_cast(gm_h8, make_uint4(r0, r1, r2, r3));
}


// ---------------------------------------------------------------------------
// Sixteen 4 x 4 outer products a b^T in one fp32 MFMA, each product rounded
// once (the FMA's addend is +0: a product of zero may lose its sign, which
// cannot reach an accumulator that is never -0): lane l = (block l / 4, column
// l % 4) gives a for row l % 4 and b for its column, and gets the block's 4 rows.
DEV gm_f4 gm_outer4(float a, float b) {
    return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, (gm_f4){0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
}

// The float whose bit pattern the dots accumulate onto, and the dot from the
// accumulated pattern.  (With the base in a scalar register in place of the
// subtraction's literal, prefill of 512 tokens was 0.9 % slower.)
template <int MODE>
constexpr float gm_base = MODE == 12 ? 0x1.8p19f : 0x1.8p23f;

template <int MODE>
DEV float gm_dot(int d) {
    return __builtin_bit_cast(float, d) - gm_base<MODE>;
}

// k_gemm_mfma: NW waves of 16 rows each, TT 16-token tiles per workgroup, for
// launches with few tiles: a wave of one tile (TT = 1) leaves the most waves,
// and a tile's serial chain over K is then all of the launch's length.
template <int TT, int MODE, int NW, bool SWI>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW == 8 ? 4 : TT == 1 ? 2 : 3))) void
k_gemm_mfma(GmArgs A) {
    constexpr int NT = 16 * TT;              // tokens per workgroup
    constexpr int NTH = 64 * NW;             // threads per workgroup
    constexpr int GPW = 2 * NW;              // 8-row groups per workgroup
    constexpr int SB = 32 / TT;              // blocks per LDS stage
    constexpr int QS = SB / 4;               // 4-block quads per stage
    constexpr int PF = TT == 1 ? 8 : 4;      // quads of nibbles in flight
    constexpr int G = TT == 1 ? 4 : 2;       // blocks per LDS read set
    constexpr int NX = NT * SB;              // token scales per stage (512)
    constexpr bool ASYM = MODE != 12;
    static_assert((NW == 4 || NW == 8) && (TT == 1 || TT == 2), "4 or 8 waves, 16 or 32 tokens");
    static_assert((2 * QS) % PF == 0, "ring slots are static over two stages");
    static_assert(!SWI || (NW == 8 && MODE == 12), "the SwiGLU pairing: 4 + 4 waves");
    __shared__ __align__(16) uint8_t bq[2][SB][NT * 32 + 32];          // int8 activations [stage][block][token][k]
    __shared__ __align__(16) float bs[2][NT][SB + 4];            // token scales [stage][token][block], rows padded
    __shared__ __align__(16) float bm[ASYM ? 2 : 1][NT][SB / 2 + 4];  // xm_s of the 64-blocks (modes 13 / 14)
    __shared__ __align__(16) float bw[2][SB][GPW * 8 + 8];           // weight scales [stage][block][row]
    // Workgroups go to the 8 XCDs round-robin by linear id L.  L = xcd +
    // 8 j with j = gy r + ty puts row tile 8 r + xcd of every token tile ty on
    // one XCD, dispatched back to back, so the gy workgroups that read the
    // same weights run together and share them through that XCD's L2.
    const int jx = blockIdx.x >> 3, ty = jx % A.gy;
    const int rt = (jx / A.gy) * 8 + (blockIdx.x & 7);
    if (rt >= A.tb[A.n_jobs]) {
        // zeroing tiles, then padding of the grid (whole workgroups)
        const int zi = rt - A.tb[A.n_jobs];
        if (zi < A.zt) {
            const int r = A.z0 + 64 * zi + (threadIdx.x & 63);
            for (int t = threadIdx.x >> 6; t < NT; t += NW) {
                const int m = ty * NT + t;
                if (m < A.M && r < A.z1) A.zo[(size_t)m * A.zld + r] = 0.0f;
            }
        }
        return;
    }
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, i16 = l & 15, kc = l >> 4;
    // SWI: waves 0-3 compute job 0 (gate), waves 4-7 job 1 (up), the same 64
    // rows (8 groups) of each, and the activations are the jobs' shared input
    int ji = 0;
    if (SWI) {
        ji = w >> 2;
    } else {
        if (A.n_jobs > 1 && rt >= A.tb[1]) ji = 1;
        if (A.n_jobs > 2 && rt >= A.tb[2]) ji = 2;
    }
    // the job's fields picked from the kernel arguments by uniform selects,
    // so they stay in scalar registers through the loop
    const GmJob& J = ji == 0 ? A.j[0] : ji == 1 ? A.j[1] : A.j[2];
    const int8_t* const Jq = ji == 0 ? A.j[0].q : ji == 1 ? A.j[1].q : A.j[2].q;
    const float* const Js = ji == 0 ? A.j[0].s : ji == 1 ? A.j[1].s : A.j[2].s;
    const int32_t* const Jm = ji == 0 ? A.j[0].m : ji == 1 ? A.j[1].m : A.j[2].m;
    // first group of the workgroup (SWI: of the wave's job), and the wave's
    // place among the waves of that job
    const int gb = SWI ? J.g0 + rt * (GPW / 2) : J.g0 + (rt - A.tb[ji]) * GPW;
    const int wl = SWI ? (w & 3) : w;
    const int m0 = ty * NT;
    const int K = A.K, M = A.M, n_blk = K >> 5, n_st = (n_blk + SB - 1) / SB;
    const size_t gstride = (size_t)n_blk * (MODE == 14 ? 208 : 144);

    // Every load is a buffer load with its whole offset in the lane: past the
    // descriptor's range it reads 0, and what lies in range past a row's or a
    // group's last block is never computed, so no load has a clamp or a
    // branch around it.  Rows and tokens are clamped once.
    const auto rsrc = [](const void* p, size_t n) {
        return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)(n < 0xFFFFFFFFu ? n : 0xFFFFFFFFu), GM_RSRC3);
    };
    const int gw0 = min(gb + 2 * wl, J.g1 - 1);
    const __amdgpu_buffer_rsrc_t rw = rsrc(J.g + (size_t)gw0 * gstride, (size_t)(J.g1 - gw0) * gstride);
    const int ga = min(gb + 2 * wl + (i16 >> 3), J.g1 - 1);
    // nibbles: lane (row i16, kc) reads the row's 16 bytes of block 4 q + kc;
    // mode 14: its 8 bytes of high bits of that block
    const uint32_t on = (uint32_t)((size_t)(ga - gw0) * gstride + (size_t)n_blk * 16 + (i16 & 7) * 16 + kc * 128);
    const uint32_t oh = (uint32_t)((size_t)(ga - gw0) * gstride + (size_t)n_blk * 144 + (i16 & 7) * 8 + kc * 64);
    gm_u4 wn[PF];
    gm_u2 wh[PF];
    auto wload = [&](int q, int slot) {
        wn[slot] = __builtin_bit_cast(gm_u4, __builtin_amdgcn_raw_buffer_load_b128(rw, on + (uint32_t)q * 512u, 0, 0));
        if (MODE == 14)
            wh[slot] = __builtin_bit_cast(gm_u2, __builtin_amdgcn_raw_buffer_load_b64(rw, oh + (uint32_t)q * 256u, 0, 0));
    };
    // Staging.  16-byte piece c = tid + NTH k: token c / (2 SB), half c & 1 of
    // block (c / 2) % SB, so consecutive threads read a token's contiguous
    // bytes.  Scale i = tid + NTH k: token i / SB, block i % SB (modes 13 / 14
    // pair i: its two scales and sums).  Weight scales: 16 bytes per (group,
    // block), group-major, addressed from the workgroup's first group (SWI:
    // groups 0-7 are job 0's, 8-15 job 1's, a whole wave in one job).
    constexpr int CPT = 2 * NX / NTH, SPT = (ASYM ? NX / 2 : NX) / NTH > 0 ? (ASYM ? NX / 2 : NX) / NTH : 1;
    static_assert(2 * NX % NTH == 0 && (!ASYM || NX / 2 % NTH == 0) && NX % NTH == 0, "whole shares per thread");
    constexpr int WS = GPW * SB;
    static_assert(WS <= NTH && WS % 64 == 0, "at most one weight scale piece per thread");
    const int jg = SWI ? (tid % WS) / (WS / 2) : ji;
    const int jgu = SWI ? __builtin_amdgcn_readfirstlane(jg) : ji;
    const GmJob& JG = jgu == 0 ? A.j[0] : jgu == 1 ? A.j[1] : A.j[2];
    const int gbg = SWI ? JG.g0 + rt * (GPW / 2) : gb;
    const __amdgpu_buffer_rsrc_t rg = rsrc(JG.g + (size_t)gbg * gstride, (size_t)(JG.g1 - gbg) * gstride);
    const int wg = (tid % WS) / SB, wb = tid % SB;
    const uint32_t og = (uint32_t)((size_t)(min(gbg + (SWI ? (wg & 7) : wg), JG.g1 - 1) - gbg) * gstride + wb * 16);
    const __amdgpu_buffer_rsrc_t rq = rsrc(Jq, (size_t)M * K);
    const __amdgpu_buffer_rsrc_t rs = rsrc(Js, (size_t)M * n_blk * 4);
    const __amdgpu_buffer_rsrc_t rm = rsrc(ASYM ? (const void*)Jm : (const void*)Js, (size_t)M * n_blk * 4);
    gm_u4 sq[CPT];
    float ss[SPT][2];
    int32_t sm[SPT][2];
    gm_u4 sw;
    uint32_t qo[CPT], so[SPT];
#pragma unroll
    for (int k = 0; k < CPT; k++) {
        const int c = tid + NTH * k;
        qo[k] = (uint32_t)(min(m0 + c / (2 * SB), M - 1) * K + 16 * (c % (2 * SB)));
    }
#pragma unroll
    for (int k = 0; k < SPT; k++) {
        const int i = tid + NTH * k;
        so[k] = ASYM ? (uint32_t)(4 * (min(m0 + i / (SB / 2), M - 1) * n_blk + 2 * (i % (SB / 2))))
                     : (uint32_t)(4 * (min(m0 + i / SB, M - 1) * n_blk + i % SB));
    }
    auto stage_load = [&](int st) {
#pragma unroll
        for (int k = 0; k < CPT; k++)
            sq[k] = __builtin_bit_cast(gm_u4,
                                       __builtin_amdgcn_raw_buffer_load_b128(rq, qo[k] + (uint32_t)st * (SB * 32u), 0, 0));
#pragma unroll
        for (int k = 0; k < SPT; k++) {
            const uint32_t o = so[k] + (uint32_t)st * (SB * 4u);
            if (ASYM) {
                const gm_u2 a = __builtin_bit_cast(gm_u2, __builtin_amdgcn_raw_buffer_load_b64(rs, o, 0, 0));
                const gm_u2 b = __builtin_bit_cast(gm_u2, __builtin_amdgcn_raw_buffer_load_b64(rm, o, 0, 0));
                const uint32_t a0 = a[0], a1 = a[1];
                ss[k][0] = __builtin_bit_cast(float, a0);
                ss[k][1] = __builtin_bit_cast(float, a1);
                sm[k][0] = (int32_t)b[0];
                sm[k][1] = (int32_t)b[1];
            } else {
                const uint32_t a = __builtin_amdgcn_raw_buffer_load_b32(rs, o, 0, 0);
                ss[k][0] = __builtin_bit_cast(float, a);
            }
        }
        sw = __builtin_bit_cast(gm_u4, __builtin_amdgcn_raw_buffer_load_b128(rg, og + (uint32_t)st * (SB * 16u), 0, 0));
    };
    auto stage_store = [&](int buf) {
#pragma unroll
        for (int k = 0; k < CPT; k++) {
            const int c = tid + NTH * k;
            *(gm_u4*)&bq[buf][(c >> 1) % SB][32 * (c / (2 * SB)) + 16 * (c & 1)] = sq[k];
        }
#pragma unroll
        for (int k = 0; k < SPT; k++) {
            const int i = tid + NTH * k;
            if (ASYM) {
                const int t = i / (SB / 2), p = i % (SB / 2);
                bs[buf][t][2 * p] = ss[k][0];
                bs[buf][t][2 * p + 1] = ss[k][1];
                const float pa = (float)sm[k][0] * ss[k][0], pb = (float)sm[k][1] * ss[k][1];
                bm[ASYM ? buf : 0][t][p] = (pa + pb) * 0.125f;
            } else {
                bs[buf][i / SB][i % SB] = ss[k][0];
            }
        }
        if (WS == NTH || tid < WS) {
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const uint32_t x = sw[2 * q], y = sw[2 * q + 1];
                const gm_h2 hx = __builtin_bit_cast(gm_h2, x), hy = __builtin_bit_cast(gm_h2, y);
                *(gm_f4*)&bw[buf][wb][8 * wg + 4 * q] = (gm_f4){(float)hx[0], (float)hx[1], (float)hy[0], (float)hy[1]};
            }
        }
    };

    gm_f4 acc[TT];
#pragma unroll
    for (int t = 0; t < TT; t++) acc[t] = (gm_f4){0.0f, 0.0f, 0.0f, 0.0f};

    // LDS operands of G blocks, read one set ahead of their MFMAs; the token
    // scales (and xm_s) of a quad are read with its first set
    long bf[2][G][TT];
    float wsr[2][G][ASYM ? 4 : 1];
    constexpr int BASE = __builtin_bit_cast(int, gm_base<MODE>);
    gm_i4 c0 = {BASE, BASE, BASE, BASE};
    asm("" : "+v"(c0));  // loop-invariant registers
    float xs[2][TT][4];
    float xm[2][TT][2];
    auto lds_set = [&](int buf, int b, int slot, int xslot) {
#pragma unroll
        for (int g = 0; g < G; g++) {
            if (ASYM) {
                const gm_f4 y = *(const gm_f4*)&bw[buf][b + g][16 * w + 4 * kc];
#pragma unroll
                for (int v = 0; v < 4; v++) wsr[slot][g][ASYM ? v : 0] = y[v];
            } else {
                wsr[slot][g][0] = bw[buf][b + g][16 * w + 4 * kc + (l & 3)];
            }
#pragma unroll
            for (int t = 0; t < TT; t++) bf[slot][g][t] = *(const long*)&bq[buf][b + g][32 * (16 * t + i16) + 8 * kc];
        }
        if (b % 4 == 0) {
#pragma unroll
            for (int t = 0; t < TT; t++) {
                const gm_f4 x = *(const gm_f4*)&bs[buf][16 * t + i16][b];
#pragma unroll
                for (int j = 0; j < 4; j++) xs[xslot][t][j] = x[j];
                if (ASYM) {
                    const float* y = &bm[ASYM ? buf : 0][16 * t + i16][b / 2];
                    xm[xslot][t][0] = y[0];
                    xm[xslot][t][1] = y[1];
                }
            }
        }
    };
    gm_f4 dk[TT];   // modes 13 / 14: the even block's dots and the pair's d,
    float dsk[4];   // held across the odd block
    // one quad: nibbles of ring slot s, blocks b .. b + 3 of stage buffer buf
    // (nb of them in range), the next quad's first set from LDS when there is
    // one in the stage
    auto quad = [&](int s, int buf, int b, int nb, int x, bool more) {
        uint32_t t0 = wn[s][0], t1 = wn[s][1], t2 = wn[s][2], t3 = wn[s][3];
        skp_transpose(t0, t1, t2, t3);
        const uint32_t tw[4] = {t0, t1, t2, t3};
        uint32_t th[4] = {0u, 0u, 0u, 0u};
        if (MODE == 14) {
            th[0] = wh[s][0];
            th[1] = th[0] >> 4;
            th[2] = wh[s][1];
            th[3] = th[2] >> 4;
            skp_transpose(th[0], th[1], th[2], th[3]);
        }
        // the quad's weight operands
        long wa[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            uint32_t lo, hi;
            if (!ASYM) {
                // 16 (u - 8) as int8: the nibble with its top bit flipped, in
                // the byte's upper half
                lo = ((tw[j] << 4) ^ 0x80808080u) & 0xF0F0F0F0u;
                hi = (tw[j] ^ 0x80808080u) & 0xF0F0F0F0u;
            } else {
                lo = tw[j] & 0x0F0F0F0Fu;
                hi = (tw[j] >> 4) & 0x0F0F0F0Fu;
                if (MODE == 14) {
                    lo |= (th[j] << 4) & 0x30303030u;
                    hi |= (th[j] << 2) & 0x30303030u;
                }
            }
            wa[j] = (long)(((uint64_t)hi << 32) | lo);
        }
        // G blocks at a time: their dots (and mode 12's products) are all
        // issued before the first is read, so their latencies overlap
#pragma unroll
        for (int j0 = 0; j0 < 4; j0 += G) {
            const int slot = G == 4 ? x : (j0 / G) & 1;
            // the set after this one
            if (j0 + G < 4)
                lds_set(buf, b + j0 + G, slot ^ 1, x);
            else if (more)
                lds_set(buf, b + 4, slot ^ 1, x ^ 1);
            if (j0 >= nb) break;  // uniform
            gm_i4 di[G][TT];
            gm_f4 pr[G][TT];
#pragma unroll
            for (int g = 0; g < G; g++)
#pragma unroll
                for (int t = 0; t < TT; t++) {
                    di[g][t] = __builtin_amdgcn_mfma_i32_16x16x32_i8(wa[j0 + g], bf[slot][g][t], c0, 0, 0, 0);
                    // rows 4 kc + 0 .. 3, the lane's token
                    if (!ASYM) pr[g][t] = gm_outer4(wsr[slot][g][0], xs[x][t][j0 + g]);
                }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int g = 0; g < G; g++) {
                const int j = j0 + g;
                if (j >= nb) break;  // uniform
#pragma unroll
                for (int t = 0; t < TT; t++) {
                    const float sx = xs[x][t][j];
                    float d[4];
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        d[v] = gm_dot<MODE>(di[g][t][v]);
                    }
                    if (!ASYM) {
#pragma unroll
                        for (int v = 0; v < 4; v++) acc[t][v] = fmaf(d[v], pr[g][t][v], acc[t][v]);
                    } else if ((j & 1) == 0) {
#pragma unroll
                        for (int v = 0; v < 4; v++) dk[t][v] = d[v];
                    } else {
                        const float sx0 = xs[x][t][j - 1], sm_ = xm[x][t][j >> 1];
#pragma unroll
                        for (int v = 0; v < 4; v++) {
                            const float p1 = d[v] * sx;
                            const float fd = fmaf(dk[t][v], sx0, p1);
                            acc[t][v] = fmaf(fd, dsk[v], acc[t][v]);
                            acc[t][v] = fmaf(wsr[slot][g][ASYM ? v : 0], sm_, acc[t][v]);
                        }
                    }
                }
                if (ASYM && (j & 1) == 0) {
#pragma unroll
                    for (int v = 0; v < 4; v++) dsk[v] = wsr[slot][g][ASYM ? v : 0];
                }
            }
        }
    };

    stage_load(0);
#pragma unroll
    for (int q = 0; q < PF; q++) wload(q, q);
    stage_store(0);
    __syncthreads();
    for (int st0 = 0; st0 < n_st; st0 += 2) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int st = st0 + h;
            if (st >= n_st) break;  // uniform
            stage_load(st + 1);
            lds_set(h, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < QS; i++) {
                const int b = st * SB + 4 * i, s = (h * QS + i) % PF;
                if (b < n_blk) quad(s, h, 4 * i, n_blk - b, i & 1, i + 1 < QS);
                wload(st * QS + i + PF, s);
            }
            if (st + 1 < n_st) stage_store(h ^ 1);
            __syncthreads();
        }
    }
    if constexpr (SWI) {
        // SwiGLU + prep of the down input for the workgroup's 64 columns
        // (one 64-block, blk) of the tokens m0 .. m0 + NT - 1 below M.  Lane l of wave
        // w holds acc[t][v] for column c = 16 (w & 3) + 4 (l / 16) + v and
        // token 16 t + l % 16; x[w & 3][t][v][l] in the LDS of the stage
        // buffers (free once every wave is past its last block) exchanges
        // them: the up waves write theirs, the gate waves replace them by
        // swiglu1(gate, up) (swiglu_prep_lane's arithmetic), then each 16-lane
        // row preps one token's block as swiglu_prep_lane does.
        float* x = (float*)&bq[0][0][0];
        static_assert(sizeof(bq) >= 4 * TT * 4 * 64 * sizeof(float), "the exchange fits the stage buffers");
        auto xi = [&](int ww, int t, int v, int ln) { return ((ww * TT + t) * 4 + v) * 64 + ln; };
        const int blk = (gb * 8) >> 6;  // gb: the wave's first group; a block is 8 groups
        __syncthreads();
        if (w >= 4) {
#pragma unroll
            for (int t = 0; t < TT; t++)
#pragma unroll
                for (int v = 0; v < 4; v++) x[xi(wl, t, v, l)] = acc[t][v];
        }
        __syncthreads();
        if (w < 4) {
            const uint8_t* sg = A.swsign ? A.swsign + 8 * blk : nullptr;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int c = 16 * wl + 4 * kc + v;
                const uint32_t neg = sg ? (sg[c >> 3] >> (c & 7)) & 1u : 0u;
#pragma unroll
                for (int t = 0; t < TT; t++) x[xi(wl, t, v, l)] = swiglu1(acc[t][v], x[xi(wl, t, v, l)], A.swdz, neg);
            }
        }
        __syncthreads();
        const int R = tid >> 4, r = tid & 15, I = A.swI, nbI = I >> 5;
#pragma unroll
        for (int pass = 0; pass < (NT + 31) / 32; pass++) {
            const int tok = R + 32 * pass, mt = m0 + tok;
            if (tok < NT && mt < M) {  // uniform over the 16-lane row
                float v4[4];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const int c = 4 * r + k;
                    v4[k] = x[xi(c >> 4, tok >> 4, c & 3, 16 * ((c >> 2) & 3) + (tok & 15))];
                }
                row_prep64(v4, r, blk, A.swo.q + (size_t)mt * I, A.swo.s + (size_t)mt * nbI,
                           A.swo.m + (size_t)mt * nbI, A.swo.h ? A.swo.h + (size_t)mt * I : nullptr);
            }
        }
        return;
    }
    // rows 16 w + 4kc + v of the workgroup, token m0 + 16t + i16
    const int grp = gb + 2 * w + (kc >> 1);
    if (grp >= J.g1) return;
#pragma unroll
    for (int t = 0; t < TT; t++) {
        const int m = m0 + 16 * t + i16;
        if (m >= M) continue;
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int r = grp * 8 + (kc & 1) * 4 + v;
            if (r < J.rows) J.out[(size_t)m * J.ldo + r] = acc[t][v];
        }
    }
}

// ---------------------------------------------------------------------------
// k_gemm_x32: 32 x 32 tiles, for launches with tiles enough to fill the chip.
// A 32x32x32 MFMA costs 8.2 cycles per 16 x 16 outputs where a 16x16x32 one
// costs 17, and a fragment read from LDS feeds twice the outputs.  The tokens
// are the MFMA's A and the weights its B, so a lane holds one weight row: one
// weight scale per lane and block, and stores of 32 consecutive rows.
//
// Workgroup of 4 waves = 2 row waves x 2 token waves: 64 RF weight rows x 64
// tokens; a wave holds RF 32-row fragments x 32 tokens.  SWI: fragment 0 is
// 32 rows of gate and fragment 1 the same rows of up, so the SwiGLU needs no
// exchange and the workgroup's 64 columns are one 64-block of the down input.
template <int RF, int MODE, bool SWI>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(RF == 1 && MODE == 12 ? 3 : 2))) void k_gemm_x32(GmArgs A) {
    constexpr int NT = 64, SB = 8;           // tokens per workgroup, blocks per LDS stage
    constexpr int PS = SB / 2;               // block pairs per stage
    constexpr int GPW = 8 * RF;              // 8-row groups per workgroup
    constexpr bool ASYM = MODE != 12;
    static_assert(!SWI || (RF == 2 && MODE == 12), "fragment 0 gate, fragment 1 up");
    __shared__ __align__(16) uint8_t aq[2][SB][NT * 32 + 32];  // int8 activations [stage][block][token][k]
    __shared__ __align__(16) float xl[2][SB][NT + 8];        // token scales
    __shared__ __align__(16) float ml[ASYM ? 2 : 1][SB / 2][NT + 8];  // xm_s of the 64-blocks (modes 13 / 14)
    __shared__ __align__(16) float wl[2][SB][GPW * 8 + 8];   // weight scales
    const int jx = blockIdx.x >> 3, ty = jx % A.gy;
    const int rt = (jx / A.gy) * 8 + (blockIdx.x & 7);
    if (rt >= A.tb[A.n_jobs]) {
        const int zi = rt - A.tb[A.n_jobs];
        if (zi < A.zt) {
            const int r = A.z0 + 64 * zi + (threadIdx.x & 63);
            for (int t = threadIdx.x >> 6; t < NT; t += 4) {
                const int m = ty * NT + t;
                if (m < A.M && r < A.z1) A.zo[(size_t)m * A.zld + r] = 0.0f;
            }
        }
        return;
    }
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, r32 = l & 31, h = l >> 5;
    const int wr = w & 1, wt = w >> 1;
    int ji = 0;
    if (!SWI) {
        if (A.n_jobs > 1 && rt >= A.tb[1]) ji = 1;
        if (A.n_jobs > 2 && rt >= A.tb[2]) ji = 2;
    }
    const GmJob& J = ji == 0 ? A.j[0] : ji == 1 ? A.j[1] : A.j[2];
    const int8_t* const Jq = ji == 0 ? A.j[0].q : ji == 1 ? A.j[1].q : A.j[2].q;
    const float* const Js = ji == 0 ? A.j[0].s : ji == 1 ? A.j[1].s : A.j[2].s;
    const int32_t* const Jm = ji == 0 ? A.j[0].m : ji == 1 ? A.j[1].m : A.j[2].m;
    const int gb = SWI ? rt * 8 : J.g0 + (rt - A.tb[ji]) * GPW;  // first group of the workgroup
    const int m0 = ty * NT;
    const int K = A.K, M = A.M, n_blk = K >> 5, n_st = (n_blk + SB - 1) / SB;
    const size_t gstride = (size_t)n_blk * (MODE == 14 ? 208 : 144);
    const auto rsrc = [](const void* p, size_t n) {
        return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)(n < 0xFFFFFFFFu ? n : 0xFFFFFFFFu), GM_RSRC3);
    };
    // a fragment's first group (fragment f: rows 32 (RF wr + f) of the
    // workgroup; SWI: rows 32 wr of job f), its descriptor and lane offset
    __amdgpu_buffer_rsrc_t rw[RF];
    uint32_t on[RF], oh[RF];
#pragma unroll
    for (int f = 0; f < RF; f++) {
        const GmJob& Jf = SWI ? A.j[f] : J;
        const int gf = min(gb + (SWI ? 4 * wr : 4 * (RF * wr + f)), Jf.g1 - 1);
        rw[f] = rsrc(Jf.g + (size_t)gf * gstride, (size_t)(Jf.g1 - gf) * gstride);
        const int ga = min(gb + (SWI ? 4 * wr : 4 * (RF * wr + f)) + (r32 >> 3), Jf.g1 - 1);
        on[f] = (uint32_t)((size_t)(ga - gf) * gstride + (size_t)n_blk * 16 + (r32 & 7) * 16 + h * 128);
        oh[f] = (uint32_t)((size_t)(ga - gf) * gstride + (size_t)n_blk * 144 + (r32 & 7) * 8 + h * 64);
    }
    constexpr int PF = ASYM && RF == 2 ? 2 : 4;  // block pairs of nibbles in flight
    static_assert((2 * PS) % PF == 0, "ring slots are static over two stages");
    gm_u4 wn[PF][RF];
    gm_u2 wh[PF][RF];
    auto wload = [&](int p, int slot) {
#pragma unroll
        for (int f = 0; f < RF; f++) {
            wn[slot][f] = __builtin_bit_cast(
                gm_u4, __builtin_amdgcn_raw_buffer_load_b128(rw[f], on[f] + (uint32_t)p * 256u, 0, 0));
            if (MODE == 14)
                wh[slot][f] = __builtin_bit_cast(
                    gm_u2, __builtin_amdgcn_raw_buffer_load_b64(rw[f], oh[f] + (uint32_t)p * 128u, 0, 0));
        }
    };
    // staging: 16-byte piece c = tid + 256 k of a token's SB 32 contiguous
    // bytes; scale i: token i / SB, block i % SB (modes 13 / 14: token, pair)
    constexpr int CPT = NT * SB * 2 / 256, SPT = NT * SB / 256;  // 4, 2
    gm_u4 sq[CPT];
    float ss[SPT];
    int32_t sm[2];
    gm_u4 sw;
    const __amdgpu_buffer_rsrc_t rq = rsrc(Jq, (size_t)M * K);
    const __amdgpu_buffer_rsrc_t rs = rsrc(Js, (size_t)M * n_blk * 4);
    const __amdgpu_buffer_rsrc_t rm = rsrc(ASYM ? (const void*)Jm : (const void*)Js, (size_t)M * n_blk * 4);
    // weight scales: thread t < 8 GPW stages the 16 bytes of group t / SB,
    // block t % SB (SWI: groups 8 .. 15 are job 1's, threads 64 .. 127)
    constexpr int WS = GPW * SB;
    const int wg = (tid % WS) / SB, wb = tid % SB;
    const GmJob& JG = SWI ? (w & 1 ? A.j[1] : A.j[0]) : J;
    const __amdgpu_buffer_rsrc_t rg = rsrc(JG.g + (size_t)gb * gstride, (size_t)(JG.g1 - gb) * gstride);
    const uint32_t og = (uint32_t)((size_t)(min(gb + (SWI ? (wg & 7) : wg), JG.g1 - 1) - gb) * gstride + wb * 16);
    uint32_t qo[CPT], so[SPT];
#pragma unroll
    for (int k = 0; k < CPT; k++) {
        const int c = tid + 256 * k;
        qo[k] = (uint32_t)(min(m0 + c / (2 * SB), M - 1) * K + 16 * (c % (2 * SB)));
    }
#pragma unroll
    for (int k = 0; k < SPT; k++) {
        const int i = tid + 256 * k;
        so[k] = ASYM ? (uint32_t)(4 * (min(m0 + tid / PS, M - 1) * n_blk + 2 * (tid % PS)))
                     : (uint32_t)(4 * (min(m0 + i / SB, M - 1) * n_blk + i % SB));
    }
    auto stage_load = [&](int st) {
#pragma unroll
        for (int k = 0; k < CPT; k++)
            sq[k] = __builtin_bit_cast(gm_u4,
                                       __builtin_amdgcn_raw_buffer_load_b128(rq, qo[k] + (uint32_t)st * (SB * 32u), 0, 0));
        if (ASYM) {
            const uint32_t o = so[0] + (uint32_t)st * (SB * 4u);
            const gm_u2 a = __builtin_bit_cast(gm_u2, __builtin_amdgcn_raw_buffer_load_b64(rs, o, 0, 0));
            const gm_u2 b = __builtin_bit_cast(gm_u2, __builtin_amdgcn_raw_buffer_load_b64(rm, o, 0, 0));
            const uint32_t a0 = a[0], a1 = a[1];
            ss[0] = __builtin_bit_cast(float, a0);
            ss[1] = __builtin_bit_cast(float, a1);
            sm[0] = (int32_t)b[0];
            sm[1] = (int32_t)b[1];
        } else {
#pragma unroll
            for (int k = 0; k < SPT; k++) {
                const uint32_t a = __builtin_amdgcn_raw_buffer_load_b32(rs, so[k] + (uint32_t)st * (SB * 4u), 0, 0);
                ss[k] = __builtin_bit_cast(float, a);
            }
        }
        sw = __builtin_bit_cast(gm_u4, __builtin_amdgcn_raw_buffer_load_b128(rg, og + (uint32_t)st * (SB * 16u), 0, 0));
    };
    auto stage_store = [&](int buf) {
#pragma unroll
        for (int k = 0; k < CPT; k++) {
            const int c = tid + 256 * k;
            *(gm_u4*)&aq[buf][(c >> 1) % SB][32 * (c / (2 * SB)) + 16 * (c & 1)] = sq[k];
        }
        if (ASYM) {
            const int t = tid / PS, p = tid % PS;
            xl[buf][2 * p][t] = ss[0];
            xl[buf][2 * p + 1][t] = ss[1];
            const float pa = (float)sm[0] * ss[0], pb = (float)sm[1] * ss[1];
            ml[ASYM ? buf : 0][p][t] = (pa + pb) * 0.125f;
        } else {
#pragma unroll
            for (int k = 0; k < SPT; k++) {
                const int i = tid + 256 * k, t = i / SB;
                xl[buf][i % SB][(t & 32) + ((t >> 2) & 1) * 16 + (t & 3) * 4 + ((t >> 3) & 3)] = ss[k];
            }
        }
        if (tid < WS) {
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const uint32_t a = sw[2 * q], b = sw[2 * q + 1];
                const gm_h2 x = __builtin_bit_cast(gm_h2, a), y = __builtin_bit_cast(gm_h2, b);
                *(gm_f4*)&wl[buf][wb][wg * 8 + 4 * q] = (gm_f4){(float)x[0], (float)x[1], (float)y[0], (float)y[1]};
            }
        }
    };

    float acc[RF][16];
#pragma unroll
    for (int f = 0; f < RF; f++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[f][v] = 0.0f;
    const bool live = m0 + 32 * wt < M;  // uniform: the wave has a token to compute

    // LDS operands of one block
    gm_i4 af[2];
    float xs[2][ASYM ? 16 : 4];
    float ws[2][RF];
    auto lds_blk = [&](int buf, int b, int slot) {
        af[slot] = *(const gm_i4*)&aq[buf][b][32 * (32 * wt + r32) + 16 * h];
        if (ASYM) {
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const gm_f4 x = *(const gm_f4*)&xl[buf][b][32 * wt + 8 * g + 4 * h];
#pragma unroll
                for (int v = 0; v < 4; v++) xs[slot][ASYM ? 4 * g + v : 0] = x[v];
            }
        } else {
            // tokens 8 g + 4 h + l % 4, g = 0 .. 3
            const gm_f4 x = *(const gm_f4*)&xl[buf][b][32 * wt + 16 * h + 4 * (l & 3)];
#pragma unroll
            for (int g = 0; g < 4; g++) xs[slot][g] = x[g];
        }
#pragma unroll
        for (int f = 0; f < RF; f++) ws[slot][f] = wl[buf][b][(SWI ? 64 * f + 32 * wr : 32 * (RF * wr + f)) + r32];
    };
    float dk[RF][16];  // modes 13 / 14: the even block's dots, d and token scales
    float dd[RF];
    float xk[16];
    gm_i16 c0;  // loop-invariant, so that the MFMAs share one set of registers
#pragma unroll
    for (int v = 0; v < 16; v++) c0[v] = __builtin_bit_cast(int, gm_base<MODE>);
    asm("" : "+v"(c0));
    // block pair p of a stage (blocks 2 p, 2 p + 1; nb of them in range)
    auto pair = [&](int s, int buf, int p, int nb, bool more) {
        gm_i4 wa[2][RF];
#pragma unroll
        for (int f = 0; f < RF; f++) {
            uint32_t w0 = wn[s][f][0], w1 = wn[s][f][1], w2 = wn[s][f][2], w3 = wn[s][f][3];
            // chunks 2 h, 2 h + 1 of both blocks
            const auto e0 = __builtin_amdgcn_permlane32_swap(w0, w2, false, false);
            const auto e1 = __builtin_amdgcn_permlane32_swap(w1, w3, false, false);
            const uint32_t c[2][2] = {{e0[0], e1[0]}, {e0[1], e1[1]}};
            uint32_t hb[2] = {0u, 0u};
            if (MODE == 14) {
                // the block's high-bit word h (chunks 2 h: low nibbles, 2 h + 1: high)
                const auto eh = __builtin_amdgcn_permlane32_swap(wh[s][f][0], wh[s][f][1], false, false);
                hb[0] = eh[0];
                hb[1] = eh[1];
            }
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    uint32_t lo, hi;
                    if (!ASYM) {
                        lo = ((c[b][q] << 4) ^ 0x80808080u) & 0xF0F0F0F0u;
                        hi = (c[b][q] ^ 0x80808080u) & 0xF0F0F0F0u;
                    } else {
                        lo = c[b][q] & 0x0F0F0F0Fu;
                        hi = (c[b][q] >> 4) & 0x0F0F0F0Fu;
                        if (MODE == 14) {
                            lo |= (q ? hb[b] : hb[b] << 4) & 0x30303030u;
                            hi |= (q ? hb[b] >> 2 : hb[b] << 2) & 0x30303030u;
                        }
                    }
                    wa[b][f][2 * q] = (int)lo;
                    wa[b][f][2 * q + 1] = (int)hi;
                }
        }
#pragma unroll
        for (int b = 0; b < 2; b++) {
            if (b == 0 || more) lds_blk(buf, 2 * p + b + 1, b ^ 1);
            if (b >= nb) break;  // uniform
            gm_i16 d[RF];
#pragma unroll
            for (int f = 0; f < RF; f++) {
                d[f] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[b], wa[b][f], c0, 0, 0, 0);
            }
            // products xs ws of tokens 8 g + 4 h + 0 .. 3 and the lane's row, all
            // issued before the first dot is read: their latencies overlap
            gm_f4 pr[RF][4];
            if (!ASYM) {
#pragma unroll
                for (int f = 0; f < RF; f++)
#pragma unroll
                    for (int g = 0; g < 4; g++) pr[f][g] = gm_outer4(xs[b][g], ws[b][f]);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int f = 0; f < RF; f++) {
                if (!ASYM) {
#pragma unroll
                    for (int v = 0; v < 16; v++) {
                        const float x = gm_dot<MODE>(d[f][v]);
                        acc[f][v] = fmaf(x, pr[f][v >> 2][v & 3], acc[f][v]);
                    }
                } else if (b == 0) {
#pragma unroll
                    for (int v = 0; v < 16; v++) {
                        dk[f][v] = gm_dot<MODE>(d[f][v]);
                        xk[v] = xs[0][ASYM ? v : 0];
                    }
                    dd[f] = ws[0][f];
                } else {
#pragma unroll
                    for (int v = 0; v < 16; v++) {
                        const float x = gm_dot<MODE>(d[f][v]);
                        const float p1 = x * xs[1][ASYM ? v : 0];
                        const float fd = fmaf(dk[f][v], xk[v], p1);
                        acc[f][v] = fmaf(fd, dd[f], acc[f][v]);
                    }
                }
            }
            if (ASYM && b == 1) {
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const gm_f4 y = *(const gm_f4*)&ml[ASYM ? buf : 0][p][32 * wt + 8 * g + 4 * h];
#pragma unroll
                    for (int f = 0; f < RF; f++)
#pragma unroll
                        for (int v = 0; v < 4; v++) acc[f][4 * g + v] = fmaf(ws[1][f], y[v], acc[f][4 * g + v]);
                }
            }
        }
    };

    stage_load(0);
#pragma unroll
    for (int p = 0; p < PF; p++) wload(p, p);
    stage_store(0);
    __syncthreads();
    for (int st0 = 0; st0 < n_st; st0 += 2) {
#pragma unroll
        for (int hh = 0; hh < 2; hh++) {
            const int st = st0 + hh;
            if (st >= n_st) break;  // uniform
            stage_load(st + 1);
            if (live) {
                lds_blk(hh, 0, 0);
#pragma unroll
                for (int i = 0; i < PS; i++) {
                    const int b = st * SB + 2 * i, s = (hh * PS + i) % PF;
                    if (b < n_blk) pair(s, hh, i, n_blk - b, i + 1 < PS);
                    wload(st * PS + i + PF, s);
                }
            }
            if (st + 1 < n_st) stage_store(hh ^ 1);
            __syncthreads();
        }
    }

    if constexpr (SWI) {
        constexpr int XS = 68;
        float* x = (float*)&aq[0][0][0];  // [token][column], rows padded
        static_assert(sizeof(aq) >= NT * XS * sizeof(float), "the exchange fits the stage buffers");
        const int col = 32 * wr + r32;
        const uint32_t neg = A.swsign ? (A.swsign[8 * rt + (col >> 3)] >> (col & 7)) & 1u : 0u;
        if (live) {
#pragma unroll
            for (int v = 0; v < 16; v++)
                x[(32 * wt + 8 * (v >> 2) + 4 * h + (v & 3)) * XS + col] = swiglu1(acc[0][v], acc[1][v], A.swdz, neg);
        }
        __syncthreads();
        const int R = tid >> 4, r = tid & 15, I = A.swI, nbI = I >> 5;
#pragma unroll
        for (int pass = 0; pass < NT / 16; pass++) {
            const int tok = R + 16 * pass, mt = m0 + tok;
            if (mt < M) {  // uniform over the 16-lane row
                float v4[4];
                const gm_f4 y = *(const gm_f4*)&x[tok * XS + 4 * r];
#pragma unroll
                for (int k = 0; k < 4; k++) v4[k] = y[k];
                row_prep64(v4, r, rt, A.swo.q + (size_t)mt * I, A.swo.s + (size_t)mt * nbI, A.swo.m + (size_t)mt * nbI,
                           A.swo.h ? A.swo.h + (size_t)mt * I : nullptr);
            }
        }
        return;
    }
#pragma unroll
    for (int f = 0; f < RF; f++) {
        const int row = (gb + 4 * (RF * wr + f)) * 8 + r32;
        if (row >= J.g1 * 8 || row >= J.rows) continue;
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int m = m0 + 32 * wt + 8 * (v >> 2) + 4 * h + (v & 3);
            if (m < M) J.out[(size_t)m * J.ldo + row] = acc[f][v];
        }
    }
}

// ---------------------------------------------------------------------------
// M <= 16 GEMM (one 16-token tile): the chains of k_gemm_mfma with K split
// across the waves of a workgroup.
//
// With one token tile k_gemm_mfma has one wave per 16 rows, each streaming
// all of K: a 4096-row matrix keeps only 256 waves busy.  Here a workgroup
// computes one 16-row fragment (2 groups) for the M tokens.  SK_NP producer
// waves take the blocks of a round (SKP_RB consecutive blocks each, SKP_RS
// per round): one v_mfma_f32_16x16x32_f16 per block gives float(D - sum8) of
// the 16 x 16 tile exactly, stored to LDS.  SK_NC = 4 chain waves run the
// fp32 chains one round behind: chain wave c owns output (token l % 16, row
// 4 (l / 16) + c) of the MFMA D layout and applies the round's blocks in
// ascending order, acc = fma(d, fp16(ws) * xs, acc), the same two rounded
// operations as k_gemm_mfma, so every output is bit-identical to it.  One
// barrier per round hands the (double-buffered) D tiles over.
//
// A producer wave reads its 4 blocks with one 16-byte load per lane (lane
// (row i, kc): row i's 16 bytes of block b0 + kc) and a 4 x 4 lane transpose
// restores the MFMA A layout (skp_transpose).  Weights, scales and
// activations are loaded SK_P - 1 rounds ahead into a register ring, the
// round loop unrolled by SK_P so every slot index is static: all in one ring
// because the wait counter retires loads in issue order, so activations
// loaded later than the weights would hold every wait to the newest weights.
// The scales ride in the same ring: 32 lanes of each producer wave load the
// weight-scale dwords of the wave's blocks and store them transposed,
// [row][block], so a chain lane reads its row's scales of a round with 16-byte
// LDS reads, and every lane a token scale, [token][block]; the chains read
// LDS only, so no memory latency sits between two barriers.
// ---------------------------------------------------------------------------
#define SK_NP 8   // producer waves
#define SK_NC 4   // chain waves (one per D component)
#define SK_P 4    // load ring depth in rounds (even; fastest of 4..10 in a sweep of the dword-load version)
static_assert(SK_P % 2 == 0, "the D buffers alternate with the round");
#ifndef SK_NB
#define SK_NB 4   // k_gemm_sk round buffers in LDS (producers run up to SK_NB rounds ahead of the chains)
#endif

#define SKP_P 8  // ring depth in rounds: a multiple of every NR (4 in one instance)
#define SKP_RB 4                 // blocks per producer wave per round
#define SKP_RS (SK_NP * SKP_RB)  // 32 blocks per round

// One round of a chain wave: every block's sp = fp16(ws) * xs first (they
// do not depend on the chain), then acc = fma(d, sp, acc) over the round's
// blocks in order; a full round runs the chain with no per-block guard, so
// each block adds one dependent instruction, not three (product, fma and a
// select).
DEV float sk_round_chain(float acc, const float (&d)[SKP_RS], const uint32_t (&wv)[SKP_RS / 2],
                         const gm_f4 (&xr)[SKP_RS / 4], int nj) {
    float sp[SKP_RS];
#pragma unroll
    for (int j = 0; j < SKP_RS; j++) {
        const gm_h2 hw = __builtin_bit_cast(gm_h2, wv[j >> 1]);
        sp[j] = __builtin_fmaf((float)hw[j & 1], xr[j >> 2][j & 3], 0.0f);
    }
    if (nj >= SKP_RS) {
#pragma unroll
        for (int j = 0; j < SKP_RS; j++) acc = fmaf(d[j], sp[j], acc);
    } else {
#pragma unroll
        for (int j = 0; j < SKP_RS; j++)
            if (j < nj) acc = fmaf(d[j], sp[j], acc);
    }
    return acc;
}

// The same for the 64-block pairs of modes 13 / 14 (dpuf_avx2.c:2871-2882): fd
// is fma(float(D0), xs0, float(D1) * xs1), wv the pair's fp16 (d, m), xm its
// xm_s, and np the pairs of the round:
//   acc = fma(fd, d, acc); acc = fma(m, xm_s, acc)
DEV float sk_round_chain_asym(float acc, const float (&fd)[SKP_RS / 2], const uint32_t (&wv)[SKP_RS / 2],
                              const gm_f4 (&xm)[SKP_RS / 8], int np) {
#pragma unroll
    for (int j = 0; j < SKP_RS / 2; j++) {
        const gm_h2 hw = __builtin_bit_cast(gm_h2, wv[j]);
        if (j < np) {  // uniform
            acc = __builtin_fmaf(fd[j], (float)hw[0], acc);
            acc = __builtin_fmaf((float)hw[1], xm[j >> 2][j & 3], acc);
        }
    }
    return acc;
}

// Polls an LDS counter until it reaches want, at most 2^22 polls (false when
// it ran out); the polled value is wave-uniform, so the loop is scalar.
DEV bool sk_wait(uint32_t* p, uint32_t want) {
    int spins = 0;
#pragma clang loop unroll(disable)
    while ((uint32_t)__builtin_amdgcn_readfirstlane(
               (int)__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) < want) {
        if (++spins >= (1 << 22)) return false;
        __builtin_amdgcn_s_sleep(1);
    }
    return true;
}

// Scales and sums of the two 64-blocks b0, b0 + 2 of a token (pairs clamped
// into the row; n_blk is even in modes 13 / 14).
DEV void sk_xs_load(__amdgpu_buffer_rsrc_t rs, __amdgpu_buffer_rsrc_t rm, int xt, int b0, int n_blk, gm_u4& xs,
                    gm_u4& xm) {
#pragma unroll
    for (int p = 0; p < 2; p++) {
        const uint32_t o = (uint32_t)(4 * (xt + min(b0 + 2 * p, n_blk - 2)));
        const gm_u2 a = __builtin_bit_cast(gm_u2, __builtin_amdgcn_raw_buffer_load_b64(rs, o, 0, 0));
        const gm_u2 b = __builtin_bit_cast(gm_u2, __builtin_amdgcn_raw_buffer_load_b64(rm, o, 0, 0));
        xs[2 * p] = a[0];
        xs[2 * p + 1] = a[1];
        xm[2 * p] = b[0];
        xm[2 * p + 1] = b[1];
    }
}

// Modes 13 / 14: a producer wave's two 64-block pairs of a round.  tw / th are
// the transposed nibble and high-bit words of its 4 blocks, xs / xm the lane's
// token scales and sums of them; fd of each pair goes to LDS in place of the
// two D tiles (half the traffic, and the chains' products with xs are taken
// off them) and the lanes of kc 0 store the pairs' xm_s.
DEV void sk_pairs(const uint32_t (&tw)[4], const uint32_t (&th)[4], const gm_u4 (&ax)[SKP_RB], gm_u4 xs, gm_u4 xm,
                  float (*dq)[4][64], float* xml, int l) {
#pragma unroll
    for (int p = 0; p < 2; p++) {
        // through scalars: this compiler's bit cast of a vector element reads element 0
        const uint32_t s0 = xs[2 * p], s1 = xs[2 * p + 1];
        const float xs0 = __builtin_bit_cast(float, s0), xs1 = __builtin_bit_cast(float, s1);
        const gm_f4 d0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(gm_unpack_a_asym(tw[2 * p], th[2 * p]),
                                                               __builtin_bit_cast(gm_h8, ax[2 * p]),
                                                               (gm_f4){0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
        const gm_f4 d1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(gm_unpack_a_asym(tw[2 * p + 1], th[2 * p + 1]),
                                                               __builtin_bit_cast(gm_h8, ax[2 * p + 1]),
                                                               (gm_f4){0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const float p1 = d1[v] * xs1;
            dq[p][v][l] = fmaf(d0[v], xs0, p1);
        }
        const float pa = (float)(int32_t)xm[2 * p] * xs0, pb = (float)(int32_t)xm[2 * p + 1] * xs1;
        if (l < 16) xml[p] = (pa + pb) * 0.125f;
    }
}

// Modes 13 / 14 on this kernel against one wave per 16 rows of k_gemm_mfma
// (which a 4-token pass leaves bound by one stage's load latency at a time):
// down [12288 -> 4096] in mode 14 at M = 4, 41 MB, 103.7 -> 20.4 us.
template <int MODE>
__global__ __launch_bounds__(64 * (SK_NP + SK_NC)) void k_gemm_sk(GmArgs A) {
    constexpr bool ASYM = MODE != 12;
    constexpr int ND = ASYM ? SKP_RS / 2 : SKP_RS;              // tiles handed over per round
    __shared__ __align__(16) float dq[SK_NB][ND][4][64];        // D (fd of a pair) tiles [buf][block][v][lane]
    __shared__ __align__(16) uint16_t wsl[SK_NB][16][SKP_RS];   // weight scales [buf][row][block]
    __shared__ __align__(16) float xsl[SK_NB][16][ND + 4];      // token scales (xm_s of a pair) [buf][token][block], rows padded
    // hand-off counters per buffer, cumulative: full[b] counts producer waves
    // done with a round in b, freed[b] chain waves done reading one
    __shared__ uint32_t full[SK_NB], freed[SK_NB];
    const int fr = blockIdx.x;
    // the wave index through readfirstlane: uniform for the compiler, so the
    // role branch and every scalar block offset stay scalar
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
    const int M = A.M;
    if (fr >= A.tb[A.n_jobs]) {
        const int zi = fr - A.tb[A.n_jobs];
        if (zi < A.zt) {
            const int r = A.z0 + 64 * zi + l;
            for (int t = w; t < M; t += SK_NP + SK_NC)
                if (r < A.z1) A.zo[(size_t)t * A.zld + r] = 0.0f;
        }
        return;
    }
    int ji = 0;
    if (A.n_jobs > 1 && fr >= A.tb[1]) ji = 1;
    if (A.n_jobs > 2 && fr >= A.tb[2]) ji = 2;
    const GmJob& J = ji == 0 ? A.j[0] : ji == 1 ? A.j[1] : A.j[2];
    const uint16_t* const Jh = ji == 0 ? A.j[0].h : ji == 1 ? A.j[1].h : A.j[2].h;
    const float* const Js = ji == 0 ? A.j[0].s : ji == 1 ? A.j[1].s : A.j[2].s;
    const int32_t* const Jm = ji == 0 ? A.j[0].m : ji == 1 ? A.j[1].m : A.j[2].m;
    const int gf = J.g0 + 2 * (fr - A.tb[ji]);  // first group of the fragment
    const int K = A.K, n_blk = K >> 5, n_r = (n_blk + SKP_RS - 1) / SKP_RS;
    const size_t gstride = (size_t)n_blk * (MODE == 14 ? 208 : 144);
    const int i16 = l & 15, kc = l >> 4;
    if (tid < SK_NB) {
        full[tid] = 0;
        freed[tid] = 0;
    }
    __syncthreads();

    if (w < SK_NP) {
        // ---- producer: 4 blocks per round, one 16-byte weight load per lane
        // (row i16, block b0 + kc) and the lane transpose, as in k_gemm_skp;
        // groups and blocks clamped per lane ----
        const size_t wbytes = (size_t)(J.g1 - gf) * gstride;
        const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(J.g + (size_t)gf * gstride), 0, (int)(wbytes < 0xFFFFFFFFu ? wbytes : 0xFFFFFFFFu), GM_RSRC3);
        const int ga = min(gf + (i16 >> 3), J.g1 - 1);
        const uint32_t on = (uint32_t)((size_t)(ga - gf) * gstride + (size_t)n_blk * 16 + (i16 & 7) * 16);
        const int sj = (l >> 2) & 3, sd = l & 3, sg = min(gf + ((l >> 4) & 1), J.g1 - 1);
        const uint32_t os = (uint32_t)((size_t)(sg - gf) * gstride + sd * 4);
        // mode 14: the row's 8 bytes of high bits of block b0 + kc
        const uint32_t oh = (uint32_t)((size_t)(ga - gf) * gstride + (size_t)n_blk * 144 + (i16 & 7) * 8);
        const __amdgpu_buffer_rsrc_t rm =
            __builtin_amdgcn_make_buffer_rsrc(ASYM ? (void*)Jm : (void*)Js, 0, M * n_blk * 4, GM_RSRC3);
        const __amdgpu_buffer_rsrc_t rh = __builtin_amdgcn_make_buffer_rsrc((void*)Jh, 0, M * K * 2, GM_RSRC3);
        const uint32_t ho = (uint32_t)(2 * (min(i16, M - 1) * K + 8 * kc));
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)Js, 0, M * n_blk * 4, GM_RSRC3);
        const int xt = min(i16, M - 1) * n_blk;
        uint32_t wq[SK_P][4], wsq[SK_P];
        gm_u4 ax[SK_P][SKP_RB];
        gm_u4 xsq[SK_P], xmq[SK_P];  // mode 12: xsq[..][0] is block b0 + kc's scale; else blocks b0 .. b0 + 3
        uint32_t hq[SK_P][2];
        // weights, scales and activations of round r in one ring slot (the
        // wait counter retires loads in issue order)
        auto load = [&](int r, int u) {
            uint32_t(&q)[4] = wq[u];
            gm_u4(&a)[SKP_RB] = ax[u];
            const int b0 = r * SKP_RS + w * SKP_RB;
            const gm_u4 v = __builtin_bit_cast(
                gm_u4, __builtin_amdgcn_raw_buffer_load_b128(rw, on + (uint32_t)min(b0 + kc, n_blk - 1) * 128u, 0, 0));
            q[0] = v[0];
            q[1] = v[1];
            q[2] = v[2];
            q[3] = v[3];
            if (MODE == 14) {
                const gm_u2 h = __builtin_bit_cast(
                    gm_u2, __builtin_amdgcn_raw_buffer_load_b64(rw, oh + (uint32_t)min(b0 + kc, n_blk - 1) * 64u, 0, 0));
                hq[u][0] = h[0];
                hq[u][1] = h[1];
            }
            wsq[u] = __builtin_amdgcn_raw_buffer_load_b32(rw, os + (uint32_t)min(b0 + sj, n_blk - 1) * 16u, 0, 0);
#pragma unroll
            for (int j = 0; j < SKP_RB; j++)
                a[j] = __builtin_bit_cast(gm_u4,
                                          __builtin_amdgcn_raw_buffer_load_b128(rh, ho, min(b0 + j, n_blk - 1) * 64, 0));
            if (ASYM)
                sk_xs_load(rs, rm, xt, b0, n_blk, xsq[u], xmq[u]);
            else
                xsq[u][0] =
                    __builtin_amdgcn_raw_buffer_load_b32(rs, (uint32_t)(4 * (xt + min(b0 + kc, n_blk - 1))), 0, 0);
        };
#pragma unroll
        for (int u = 0; u < SK_P - 1; u++) load(u, u);
        for (int it0 = 0; it0 < n_r; it0 += SK_P) {
#pragma unroll
            for (int u = 0; u < SK_P; u++) {
                const int it = it0 + u;
                if (it >= n_r) break;  // uniform
                const int un = (u + SK_P - 1) % SK_P;
                load(it + SK_P - 1, un);
                {
                    // round it goes to buffer it % SK_NB once the chains have
                    // read round it - SK_NB from it
                    const int buf = it % SK_NB;
                    if (it >= SK_NB) {
                        if (!sk_wait(&freed[buf], (uint32_t)(SK_NC * (it / SK_NB))) && l == 0) atomicOr(A.err, 1);
                        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
                    }
                    uint32_t t0 = wq[u][0], t1 = wq[u][1], t2 = wq[u][2], t3 = wq[u][3];
                    skp_transpose(t0, t1, t2, t3);
                    const uint32_t tw[4] = {t0, t1, t2, t3};
                    if (ASYM) {
                        uint32_t th[4] = {0u, 0u, 0u, 0u};
                        if (MODE == 14) {
                            // word kc / 2 of the row's high bits, the odd chunk's in the upper nibbles
                            th[0] = hq[u][0];
                            th[1] = hq[u][0] >> 4;
                            th[2] = hq[u][1];
                            th[3] = hq[u][1] >> 4;
                            skp_transpose(th[0], th[1], th[2], th[3]);
                        }
                        sk_pairs(tw, th, ax[u], xsq[u], xmq[u],
                                 &dq[buf][2 * w], &xsl[buf][i16][2 * w], l);
                    } else {
#pragma unroll
                        for (int j = 0; j < SKP_RB; j++) {
                            const gm_f4 d = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                                gm_unpack_a(tw[j]), __builtin_bit_cast(gm_h8, ax[u][j]),
                                (gm_f4){0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
                            for (int v = 0; v < 4; v++) dq[buf][w * SKP_RB + j][v][l] = d[v];
                        }
                    }
                    if (l < 32) {
                        const int row = ((l >> 4) & 1) * 8 + 2 * sd;
                        wsl[buf][row][w * SKP_RB + sj] = (uint16_t)(wsq[u] & 0xFFFFu);
                        wsl[buf][row + 1][w * SKP_RB + sj] = (uint16_t)(wsq[u] >> 16);
                    }
                    if (!ASYM) xsl[buf][i16][w * SKP_RB + kc] = __builtin_bit_cast(float, xsq[u][0]);
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
                    if (l == 0) __hip_atomic_fetch_add(&full[buf], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                }
            }
        }
        return;
    }

    // ---- chain wave c: output (token l % 16, row 4 (l / 16) + c) ----
    const int c = w - SK_NP, rr = 4 * kc + c;
    float acc = 0.0f;
    for (int it = 1; it <= n_r; it++) {
        {
            // round it - 1, once every producer wave has written it
            const int buf = (it - 1) % SK_NB, b0 = (it - 1) * SKP_RS;
            if (!sk_wait(&full[buf], (uint32_t)(SK_NP * ((it - 1) / SK_NB + 1))) && l == 0) atomicOr(A.err, 1);
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
            const int nj = min(SKP_RS, n_blk - b0);  // uniform
            float d[ND];
#pragma unroll
            for (int j = 0; j < ND; j++) d[j] = dq[buf][j][c][l];
            // scale words as separate 32-bit values (see k_gemm_skp)
            uint32_t wv[SKP_RS / 2];
#pragma unroll
            for (int q = 0; q < SKP_RS / 8; q++) {
                const gm_u4 t = *(const gm_u4*)&wsl[buf][rr][8 * q];
                wv[4 * q] = t[0];
                wv[4 * q + 1] = t[1];
                wv[4 * q + 2] = t[2];
                wv[4 * q + 3] = t[3];
            }
            gm_f4 xr[ND / 4];
#pragma unroll
            for (int q = 0; q < ND / 4; q++) xr[q] = *(const gm_f4*)&xsl[buf][i16][4 * q];
            if constexpr (ASYM)
                acc = sk_round_chain_asym(acc, d, wv, xr, nj >> 1);
            else
                acc = sk_round_chain(acc, d, wv, xr, nj);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
            if (l == 0) __hip_atomic_fetch_add(&freed[buf], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
    }
    const int grp = gf + (rr >> 3);
    const int r = grp * 8 + (rr & 7);
    if (i16 < M && grp < J.g1 && r < J.rows) J.out[(size_t)i16 * J.ldo + r] = acc;
}

// The same for K <= 32 NR blocks (NR rounds of 32 blocks per fragment, NR
// <= 4), with persistent workgroups: job j gets tb[j + 1] - tb[j]
// workgroups, sized to the chip, and workgroup lb walks the job's fragments
// lb, lb + nwg, ... with one load ring running across fragment boundaries,
// so the ring fills once per workgroup instead of once per fragment.  The
// activations and token scales a producer wave needs are the same for every
// fragment: they are loaded once, before the loop, and the ring holds only
// weight nibbles and weight scales, SKP_P - 1 rounds ahead.  Rounds past the
// matrix's last (K < 1024 NR) compute nothing.
//
// A producer wave takes 4 consecutive blocks per round with one 16-byte load
// per lane: lane (row i, kc) reads row i's 16 bytes of block b0 + kc, 1 KB
// per load instruction (four times the bytes of a dword per lane, for the
// same number of load instructions in flight).  A 4 x 4 transpose across the
// four 16-lane rows of the wave (v_permlane32_swap, then v_permlane16_swap)
// turns that into the MFMA A layout: word kc of each of the 4 blocks in lane
// (i, kc).
// ---------------------------------------------------------------------------
template <int NR, int MODE>
__global__ __launch_bounds__(64 * (SK_NP + SK_NC)) void k_gemm_skp(GmArgs A) {
    constexpr bool ASYM = MODE != 12;
    constexpr int ND = ASYM ? SKP_RS / 2 : SKP_RS;  // tiles handed over per round
    constexpr int P = MODE == 14 && NR == 4 ? 4 : SKP_P;  // mode 14: its high bits would not fit 8 rounds in registers
    static_assert(P % NR == 0 && NR <= 4, "ring depth must be a multiple of the rounds per fragment");
    __shared__ __align__(16) float dq[2][ND][4][64];        // D (fd of a pair) tiles [buf][block][v][lane]
    __shared__ __align__(16) uint16_t wsl[2][16][SKP_RS];   // weight scales [buf][row][block]
    __shared__ __align__(16) float xsl[2][16][ND + 4];      // token scales (xm_s of a pair) [buf][token][block], rows padded
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
    const int M = A.M, bid = blockIdx.x;
    if (bid >= A.tb[A.n_jobs]) {
        const int zi = bid - A.tb[A.n_jobs];
        if (zi < A.zt) {
            const int r = A.z0 + 64 * zi + l;
            for (int t = w; t < M; t += SK_NP + SK_NC)
                if (r < A.z1) A.zo[(size_t)t * A.zld + r] = 0.0f;
        }
        return;
    }
    int ji = 0;
    if (A.n_jobs > 1 && bid >= A.tb[1]) ji = 1;
    if (A.n_jobs > 2 && bid >= A.tb[2]) ji = 2;
    const GmJob& J = ji == 0 ? A.j[0] : ji == 1 ? A.j[1] : A.j[2];
    const uint16_t* const Jh = ji == 0 ? A.j[0].h : ji == 1 ? A.j[1].h : A.j[2].h;
    const float* const Js = ji == 0 ? A.j[0].s : ji == 1 ? A.j[1].s : A.j[2].s;
    const int32_t* const Jm = ji == 0 ? A.j[0].m : ji == 1 ? A.j[1].m : A.j[2].m;
    const int lb = bid - A.tb[ji], nwg = A.tb[ji + 1] - A.tb[ji];
    const int nf = (J.g1 - J.g0 + 1) >> 1;              // fragments of the job
    const int n_my = (nf - lb + nwg - 1) / nwg;         // >= 1: nwg <= nf
    const int K = A.K, n_blk = K >> 5, S = n_my * NR;   // steps: NR rounds per fragment
    const uint32_t gstride = (uint32_t)n_blk * (MODE == 14 ? 208u : 144u);    // J.g1 gstride < 2^32 is checked at launch
    const int i16 = l & 15, kc = l >> 4;

    if (w < SK_NP) {
        // ---- producer: one descriptor over the job's groups up to g1; the
        // fragment's base goes into the scalar offset, which the range check
        // does not cover, so the lanes of a fragment's second group add it
        // only when it exists (a one-group fragment re-reads its first), and
        // block indices are clamped per lane ----
        const __amdgpu_buffer_rsrc_t rw =
            __builtin_amdgcn_make_buffer_rsrc((void*)J.g, 0, (int)((uint32_t)J.g1 * gstride), GM_RSRC3);
        const uint32_t on = (uint32_t)n_blk * 16u + (i16 & 7) * 16;
        const bool on_hi = i16 >= 8;
        // weight-scale dword of lane l < 32: group (l >> 4) & 1 of the
        // fragment, block (l >> 2) & 3 of the wave, rows 2 (l & 3), 2 (l & 3) + 1
        const int sj = (l >> 2) & 3, sd = l & 3;
        const bool os_hi = ((l >> 4) & 1) != 0;
        const uint32_t oh = (uint32_t)n_blk * 144u + (i16 & 7) * 8;  // mode 14: the row's 8 bytes of high bits
        uint32_t wq[P][4], wsq[P];
        uint32_t hq[P][2];
        gm_u4 ax[NR][SKP_RB];
        // token l & 15, per round: mode 12 block l >> 4 of the wave's scale in
        // [0], else the wave's 4 blocks' scales and sums
        gm_u4 xh[NR], xhm[NR];
        {
            const __amdgpu_buffer_rsrc_t rh = __builtin_amdgcn_make_buffer_rsrc((void*)Jh, 0, M * K * 2, GM_RSRC3);
            const __amdgpu_buffer_rsrc_t rs =
                __builtin_amdgcn_make_buffer_rsrc((void*)Js, 0, M * n_blk * 4, GM_RSRC3);
            const __amdgpu_buffer_rsrc_t rm =
                __builtin_amdgcn_make_buffer_rsrc(ASYM ? (void*)Jm : (void*)Js, 0, M * n_blk * 4, GM_RSRC3);
            const uint32_t ho = (uint32_t)(2 * (min(i16, M - 1) * K + 8 * kc));
            const int xt = min(i16, M - 1) * n_blk;
#pragma unroll
            for (int r = 0; r < NR; r++) {
                const int b0 = r * SKP_RS + w * SKP_RB;
#pragma unroll
                for (int j = 0; j < SKP_RB; j++)
                    ax[r][j] = __builtin_bit_cast(
                        gm_u4, __builtin_amdgcn_raw_buffer_load_b128(rh, ho, min(b0 + j, n_blk - 1) * 64, 0));
                if (ASYM) {
                    sk_xs_load(rs, rm, xt, b0, n_blk, xh[r], xhm[r]);
                } else {
                    const uint32_t xo = (uint32_t)(4 * (xt + min(b0 + kc, n_blk - 1)));
                    xh[r][0] = __builtin_amdgcn_raw_buffer_load_b32(rs, xo, 0, 0);
                }
            }
        }
        // loads of step s = NR fl + r: fragment lb + fl nwg, round r.  Steps
        // past the workgroup's last fragment re-read that fragment.
        const int fr_last = lb + (n_my - 1) * nwg;
        auto wload = [&](int fl, int r, int u) {
            uint32_t(&q)[4] = wq[u];
            const int fr = min(lb + fl * nwg, fr_last);
            const uint32_t gb = (uint32_t)(J.g0 + 2 * fr) * gstride;
            const uint32_t g2 = J.g0 + 2 * fr + 1 < J.g1 ? gstride : 0u;  // uniform
            const int b0 = r * SKP_RS + w * SKP_RB;
            const uint32_t von = on + (on_hi ? g2 : 0u) + (uint32_t)min(b0 + kc, n_blk - 1) * 128u;
            const gm_u4 v = __builtin_bit_cast(gm_u4, __builtin_amdgcn_raw_buffer_load_b128(rw, von, gb, 0));
            q[0] = v[0];
            q[1] = v[1];
            q[2] = v[2];
            q[3] = v[3];
            const uint32_t vos = (os_hi ? g2 : 0u) + (uint32_t)min(b0 + sj, n_blk - 1) * 16u + sd * 4;
            wsq[u] = __builtin_amdgcn_raw_buffer_load_b32(rw, vos, gb, 0);
            if (MODE == 14) {
                const uint32_t voh = oh + (on_hi ? g2 : 0u) + (uint32_t)min(b0 + kc, n_blk - 1) * 64u;
                const gm_u2 h = __builtin_bit_cast(gm_u2, __builtin_amdgcn_raw_buffer_load_b64(rw, voh, gb, 0));
                hq[u][0] = h[0];
                hq[u][1] = h[1];
            }
        };
#pragma unroll
        for (int u = 0; u < P - 1; u++) wload(u / NR, u % NR, u);
        for (int it0 = 0; it0 <= S; it0 += P) {
#pragma unroll
            for (int u = 0; u < P; u++) {
                const int it = it0 + u;
                if (it > S) break;  // uniform
                const int un = (u + P - 1) % P;
                wload((it0 + u + P - 1) / NR, un % NR, un);
                const int r = u % NR;
                if (it < S && r * SKP_RS < n_blk) {
                    const int buf = u & 1;
                    uint32_t t0 = wq[u][0], t1 = wq[u][1], t2 = wq[u][2], t3 = wq[u][3];
                    skp_transpose(t0, t1, t2, t3);
                    const uint32_t tw[4] = {t0, t1, t2, t3};
                    if (ASYM) {
                        uint32_t th[4] = {0u, 0u, 0u, 0u};
                        if (MODE == 14) {
                            // word kc / 2 of the row's high bits, the odd chunk's in the upper nibbles
                            th[0] = hq[u][0];
                            th[1] = hq[u][0] >> 4;
                            th[2] = hq[u][1];
                            th[3] = hq[u][1] >> 4;
                            skp_transpose(th[0], th[1], th[2], th[3]);
                        }
                        sk_pairs(tw, th, ax[r], xh[r], xhm[r],
                                 &dq[buf][2 * w], &xsl[buf][i16][2 * w], l);
                    } else {
#pragma unroll
                        for (int j = 0; j < SKP_RB; j++) {
                            const gm_f4 d = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                                gm_unpack_a(tw[j]), __builtin_bit_cast(gm_h8, ax[r][j]),
                                (gm_f4){0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
                            for (int v = 0; v < 4; v++) dq[buf][w * SKP_RB + j][v][l] = d[v];
                        }
                    }
                    if (l < 32) {
                        const int row = ((l >> 4) & 1) * 8 + 2 * sd;
                        wsl[buf][row][w * SKP_RB + sj] = (uint16_t)(wsq[u] & 0xFFFFu);
                        wsl[buf][row + 1][w * SKP_RB + sj] = (uint16_t)(wsq[u] >> 16);
                    }
                    if (!ASYM) xsl[buf][i16][w * SKP_RB + kc] = __builtin_bit_cast(float, xh[r][0]);
                }
                __syncthreads();
            }
        }
        return;
    }

    // ---- chain wave c: output (token l % 16, row 4 (l / 16) + c) ----
    const int c = w - SK_NP, rr = 4 * kc + c;
    float acc = 0.0f;
    for (int it0 = 0; it0 <= S; it0 += P) {
#pragma unroll
        for (int u = 0; u < P; u++) {
            const int it = it0 + u;
            if (it > S) break;  // uniform
            if (it >= 1) {
                // step it - 1: round r of local fragment fl
                const int um = (u + P - 1) % P, r = um % NR;
                const int fl = (u >= 1 ? it0 : it0 - P) / NR + um / NR;
                const int buf = (u + 1) & 1, b0 = r * SKP_RS;
                const int nj = min(SKP_RS, n_blk - b0);  // uniform, <= 0 past the last round
                if (nj > 0) {
                    float d[ND];
#pragma unroll
                    for (int j = 0; j < ND; j++) d[j] = dq[buf][j][c][l];
                    // the scale words as separate 32-bit values: this compiler
                    // selected the wrong register for words 1..3 when they
                    // went from a 4 x 32-bit vector into v_fma_mix_f32
                    uint32_t wv[SKP_RS / 2];
#pragma unroll
                    for (int q = 0; q < SKP_RS / 8; q++) {
                        const gm_u4 t = *(const gm_u4*)&wsl[buf][rr][8 * q];
                        wv[4 * q] = t[0];
                        wv[4 * q + 1] = t[1];
                        wv[4 * q + 2] = t[2];
                        wv[4 * q + 3] = t[3];
                    }
                    gm_f4 xr[ND / 4];
#pragma unroll
                    for (int q = 0; q < ND / 4; q++) xr[q] = *(const gm_f4*)&xsl[buf][i16][4 * q];
                    if constexpr (ASYM)
                        acc = sk_round_chain_asym(acc, d, wv, xr, nj >> 1);
                    else
                        acc = sk_round_chain(acc, d, wv, xr, nj);
                }
                if (r == NR - 1) {
                    const int fr = lb + fl * nwg;
                    const int grp = J.g0 + 2 * fr + (rr >> 3);
                    const int row = grp * 8 + (rr & 7);
                    if (fr < nf && i16 < M && grp < J.g1 && row < J.rows) J.out[(size_t)i16 * J.ldo + row] = acc;
                    acc = 0.0f;
                }
            }
            __syncthreads();
        }
    }
}


extern "C" {

typedef void (*GmKernel)(GmArgs);

// Workgroups of a K-split GEMM instance the device holds at once.
static int gm_capacity(GmKernel k, int threads) {
    static int n_cu = 0;
    static GmKernel c_k[9];
    static int c_cap[9], c_n = 0;
    for (int i = 0; i < c_n; i++)
        if (c_k[i] == k) return c_cap[i];
    if (n_cu == 0) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n_cu <= 0)
            n_cu = 1;
    }
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k, threads, 0) != hipSuccess || per_cu <= 0)
        per_cu = 1;
    const int cap = per_cu * n_cu;
    if (c_n < 9) {
        c_k[c_n] = k;
        c_cap[c_n++] = cap;
    }
    return cap;
}


extern "C++" {
template <int MODE>
static GmKernel gm_skp_of(int nr) {
    return nr == 1 ? k_gemm_skp<1, MODE> : nr == 2 ? k_gemm_skp<2, MODE> : k_gemm_skp<4, MODE>;
}
}

extern "C++" {
template <int MODE>
static GmKernel gm_of(bool x32, int rf, int tt) {
    if (!x32) return tt == 1 ? k_gemm_mfma<1, MODE, 4, false> : k_gemm_mfma<2, MODE, 4, false>;
    if constexpr (MODE != 14)
        if (rf == 2) return k_gemm_x32<2, MODE, false>;
    return k_gemm_x32<1, MODE, false>;
}
}

// Gate and up of M > 16 tokens with the SwiGLU + dead zone + prep of the down
// input in the same launch: the workgroup that computes 64 rows of gate and
// the same of up preps those 64 columns of its tokens into out.  -1 (nothing
// launched) when the shapes do not allow it: mode 12, one shared input, every
// row of equal gate / up matrices with 64 | rows, and out distinct from the
// input.  It pays at every M > 16: the fp32 gate and up rows are never written
// and a launch goes (pp512 20.7 -> 19.8 ms when it was introduced).
int32_t dpuf_hip_gemm_swiglu(void* s, int32_t M, const DpufGemvJob* jobs, float dz, const uint8_t* sign,
                             DpufPrep out) {
    const DpufGemvJob& a = jobs[0];
    const DpufGemvJob& b = jobs[1];
    const int I = a.w.rows;
    if (M <= 16 || a.w.mode != 12 || b.w.mode != 12 || a.w.cols != b.w.cols || b.w.rows != I || I % 64 ||
        2 * I < GM_SWI_ROWS || a.g0 != 0 || b.g0 != 0 || a.g1 != I / 8 || b.g1 != I / 8 || !a.p.q || a.p.q != b.p.q ||
        a.p.s != b.p.s || !out.q || !out.s || !out.m || out.q == a.p.q)
        return -1;
    if ((long long)M * a.w.cols >= (1ll << 30) || (long long)M * I >= (1ll << 30)) return -1;
    GmArgs G;
    memset(&G, 0, sizeof G);
    G.n_jobs = 2;
    G.K = a.w.cols;
    G.M = M;
    for (int i = 0; i < 2; i++) {
        G.j[i].g = jobs[i].w.g;
        G.j[i].g0 = 0;
        G.j[i].g1 = jobs[i].g1;
        G.j[i].rows = jobs[i].w.rows;
        G.j[i].h = jobs[i].p.h;
        G.j[i].q = jobs[i].p.q;
        G.j[i].s = jobs[i].p.s;
        G.j[i].m = jobs[i].p.m;
        G.j[i].out = jobs[i].out;
        G.j[i].ldo = jobs[i].ldo;
    }
    const int tiles = I / 64;
    G.tb[0] = 0;
    G.tb[1] = tiles;
    G.tb[2] = tiles;
    G.swo = out;
    G.swsign = sign;
    G.swdz = dz;
    G.swI = I;
    const int gx = (tiles + 7) & ~7;
    // up to 32 tokens two 16-token tiles, else 32 x 32 tiles (M = 29: 32 us against
    // 50, whose second token wave has nothing to do; M = 512: 204 against 178)
    const bool x32 = M > 32;
    const int nt = x32 ? 64 : 32;
    G.gy = (M + nt - 1) / nt;
    GmKernel k = x32 ? k_gemm_x32<2, 12, true> : k_gemm_mfma<2, 12, 8, true>;
    hipLaunchKernelGGL(k, dim3(gx * G.gy), dim3(x32 ? 256 : 512), 0, ST(s), G);
    LAUNCHED("k_gemm_mfma");
    return 0;
}

// The M > 1 GEMM; rows [z0, z1) of zo are zeroed by the same launch.
void dpuf_hip_gm_launch(void* s, int32_t M, int32_t n_jobs, const DpufGemvJob* jobs, float* zo, int32_t zld, int32_t z0,
                      int32_t z1) {
    {
        GmArgs G;
        memset(&G, 0, sizeof G);
        G.n_jobs = n_jobs;
        G.K = jobs[0].w.cols;
        G.M = M;
        int any = 0;
        for (int i = 0; i < n_jobs; i++) {
            G.j[i].g = jobs[i].w.g;
            G.j[i].g0 = jobs[i].g0;
            G.j[i].g1 = jobs[i].g1;
            G.j[i].rows = jobs[i].w.rows;
            G.j[i].h = jobs[i].p.h;
            G.j[i].q = jobs[i].p.q;
            if ((long long)M * G.K >= (1ll << 30)) {
                note(hipErrorInvalidValue, "dpuf_hip_gemv: M * K must stay below 2^30");
                return;
            }
            // the K-split kernels read the fp16 copy, the others the int8 one
            if (M <= 16 && !jobs[i].p.h) {
                note(hipErrorInvalidValue, "dpuf_hip_gemv: 2..16 tokens need the fp16 activations (DpufPrep.h)");
                return;
            }
            if (M > 16 && !jobs[i].p.q) {
                note(hipErrorInvalidValue, "dpuf_hip_gemv: more than 16 tokens need the int8 activations (DpufPrep.q)");
                return;
            }
            G.j[i].s = jobs[i].p.s;
            G.j[i].m = jobs[i].p.m;
            G.j[i].out = jobs[i].out;
            G.j[i].ldo = jobs[i].ldo;
            any += jobs[i].g1 > jobs[i].g0;
        }
        if (zo && z1 > z0) {
            G.zo = zo;
            G.zld = zld;
            G.z0 = z0;
            G.z1 = z1;
            G.zt = (z1 - z0 + 63) / 64;
        }
        if (any + G.zt <= 0) return;
        const int n_blk = G.K >> 5;
        const int mode = jobs[0].w.mode;  // one mode per launch (dpuf_hip_gemv groups them)
        long long gmax = 0;
        for (int i = 0; i < n_jobs; i++) gmax = gmax > jobs[i].g1 ? gmax : jobs[i].g1;
        // up to 16 tokens, every mode: K-split (modes 13 / 14 at M = 4 and the 8B
        // shapes: Q or O 34.0 -> 10.6 us, K + V 36.8 -> 11.1, down 103.7 -> 20.4
        // against k_gemm_mfma, whose waves are then one per 16 rows)
        if (M <= 16 && n_blk <= 128 && gmax * n_blk * dpuf_grp_unit(mode) < 0xFFFFFFFFll) {
            // one 16-token tile, K <= 4096: persistent K-split workgroups,
            // each job's share of the chip in proportion to its fragments
            const int NR = n_blk <= 32 ? 1 : n_blk <= 64 ? 2 : 4;
            GmKernel k = mode == 13 ? gm_skp_of<13>(NR) : mode == 14 ? gm_skp_of<14>(NR) : gm_skp_of<12>(NR);
            int cap = gm_capacity(k, 64 * (SK_NP + SK_NC));
            if (dpuf_hip_mv_max_wg() > 0 && cap > dpuf_hip_mv_max_wg()) cap = dpuf_hip_mv_max_wg();
            int nfr[3], ftot = 0;
            for (int i = 0; i < n_jobs; i++) {
                const int ng = jobs[i].g1 - jobs[i].g0;
                nfr[i] = ng > 0 ? (ng + 1) / 2 : 0;
                ftot += nfr[i];
            }
            int wgs = 0;
            for (int i = 0; i < n_jobs; i++) {
                G.tb[i] = wgs;
                int nw = ftot > 0 ? (int)(((long long)cap * nfr[i] + ftot - 1) / ftot) : 0;
                nw = nw < 1 ? 1 : nw;
                wgs += nfr[i] > 0 ? (nw < nfr[i] ? nw : nfr[i]) : 0;
            }
            G.tb[n_jobs] = wgs;
            hipLaunchKernelGGL(k, dim3(wgs + G.zt), dim3(64 * (SK_NP + SK_NC)), 0, ST(s), G);
            LAUNCHED("k_gemm_skp");
            return;
        }
        if (M <= 16) {
            // one 16-token tile: the K-split kernel, one workgroup per 16 rows
            int f = 0;
            for (int i = 0; i < n_jobs; i++) {
                G.tb[i] = f;
                const int ng = jobs[i].g1 - jobs[i].g0;
                f += ng > 0 ? (ng + 1) / 2 : 0;
            }
            G.tb[n_jobs] = f;
            G.err = dpuf_hip_error_word();
            if (!G.err) {
                note(hipErrorInvalidValue, "dpuf_hip_gemv: no device error word bound");
                return;
            }
            hipLaunchKernelGGL(mode == 13 ? k_gemm_sk<13> : mode == 14 ? k_gemm_sk<14> : k_gemm_sk<12>, dim3(f + G.zt), dim3(64 * (SK_NP + SK_NC)), 0, ST(s), G);
            LAUNCHED("k_gemm_sk");
            return;
        }
        // The tile by the number of 16 x 16 tiles per SIMD (each a serial
        // chain over K).  Measured, us (16 x 16 | 16 x 32 | 32 x 32 | 64 x 32
        // per wave; before the outer-product MFMAs), mode 12: 4 096 rows, K = 12 288: 2 per SIMD 43 | 61 | 88 |
        // 126; 4 per SIMD 86 | 81 | 90 | 126; 8 per SIMD 179 | 160 | 119 | 136.
        // 6 144 rows, K = 4 096: 3 per SIMD 26 | 29 | 32 | 46; 6 per SIMD 46 |
        // 39 | 37 | 47.  24 576 rows: 12 per SIMD 86 | 72 | 52 | 62; 48 per SIMD
        // 312 | 254 | 200 | 190.  In mode 13 the wider wave is ahead sooner
        // (24 576 rows, 9 per SIMD: 65 | 71 | 64; 6 per SIMD 42 | 43 | 53); in
        // mode 14 its registers do not fit.
        const int tm = (M + 15) / 16, simds = 4 * dpuf_hip_cu_count();
        long long tiles = 0;
        for (int i = 0; i < n_jobs; i++) {
            const int ng = jobs[i].g1 - jobs[i].g0;
            tiles += ng > 0 ? (long long)((ng + 1) / 2) * tm : 0;
        }
        const bool x32 = tiles >= 6ll * simds;
        const int rf = x32 && mode != 14 && tiles >= (mode == 13 ? 8ll : 32ll) * simds ? 2 : 1;
        const int tt = tiles >= 4ll * simds ? 2 : 1;
        const int nt = x32 ? 64 : 16 * tt, gpw = 8 * rf;
        int t = 0;
        for (int i = 0; i < n_jobs; i++) {
            G.tb[i] = t;
            const int ng = jobs[i].g1 - jobs[i].g0;
            t += ng > 0 ? (ng + gpw - 1) / gpw : 0;
        }
        G.tb[n_jobs] = t;
        // a multiple of 8 row tiles keeps a row tile's token tiles on one XCD
        const int gx = (t + G.zt + 7) & ~7;
        G.gy = (M + nt - 1) / nt;
        GmKernel k = mode == 13 ? gm_of<13>(x32, rf, tt) : mode == 14 ? gm_of<14>(x32, rf, tt) : gm_of<12>(x32, rf, tt);
        hipLaunchKernelGGL(k, dim3(gx * G.gy), dim3(256), 0, ST(s), G);
        LAUNCHED("k_gemm_mfma");
    }
}


}  // extern "C"

// attn_tile.hip -- attention of several tokens (prompts and prompt chunks) on
// the fp32 matrix instructions, over the fp32 and the int8 KV cache, for even
// query-head groups: scores (k_attn_scm, k_attn_q8_scm), then softmax + P.V +
// the prep of the O projection's input (k_attn_pvm).
//
// Numerics contract: bit-identical to gqa_attn_head_pair_f32 /
// gqa_attn_head_pair_q8 (dpuf_engine.c:341-577, 579-752).  Every fp32 MFMA of
// gfx950 computes each of its outputs as one chain of fused multiply-adds
// over k in ascending order, rounded after each, denormals kept (compared bit
// for bit with fmaf chains on the device over normal, denormal, overflowing,
// infinite and NaN operands), so a chain of v_mfma_f32_16x16x4_f32 with the
// accumulator as C is the reference's FMA chain whenever the k index of the
// operands runs through its elements in its order:
//   * scores: the reference's eight accumulators j, each a chain over
//     q[8i + j] k[8i + j]: eight accumulator tiles, k = i;
//   * P.V: a chain over the keys per output, k = key;
//   * int8 scores: per 32-block and lane L the four-term chain
//     8 + L, L, 24 + L, 16 + L (one MFMA, C = 0), then fma(t, k_scale, s).
// The horizontal sums, the softmax and the last keys of a tile (which only
// some of its rows reach) run on the vector unit as in the other kernels.
// Operand layout of the 16x16x4 instruction (lane l, c = l % 16, g = l / 16):
// A lane = row c, k = g; B lane = column c, k = g; D register i = row
// 4 g + i, column c.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include "hip_layer.h"
#include "dev_common.h"
#include "hip_internal.h"
#include "attn_common.h"

#define ATL_SLOTS DPUF_HIP_ATTN_SLOTS
#define ATL_RSRC3 0x00020000  // buffer descriptor word 3 (gfx9 family): 32-bit raw data

DEV gm_f4 mfma4(float a, float b, gm_f4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// Row r of a tile of qt tokens x G heads starting at token m0: its kv_len (0
// past the last row or token).
DEV int tile_len(int r, int G, int qt, int m0, int M, int pos0) {
    const int mi = r / G;
    return mi < qt && m0 + mi < M ? pos0 + m0 + mi + 1 : 0;
}

// Stores one lane's four scores (keys t .. t + 3 of one row, t % 4 == 0) and
// takes those below kv_len L into the lane's maximum.
DEV void score_store4(float* row, int t, int L, int max_seq, const float (&s)[4], float& mx) {
    if (t >= L) return;
    if (t + 3 < max_seq) {
        // past L but inside the row: never read as a score
        __builtin_memcpy(row + t, s, 16);
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (t + i < L) row[t + i] = s[i];
    }
#pragma unroll
    for (int i = 0; i < 4; i++)
        if (t + i < L) mx = fmaxf(mx, s[i]);
}

// The maximum of each row's scores over the wave's keys into its slot (lanes
// c of the four lane groups hold the same row).
DEV void score_max_slot(float mx, int L, float* slot, int g) {
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    if (g == 0 && L > 0) *slot = mx;
}

// ---------------------------------------------------------------------------
// Scores over the fp32 cache.  A wave keeps XT x 16 query rows (qt tokens x G
// heads) in registers and walks tpw tiles of 16 keys: K as the A operand, q
// as B, so a lane ends with four consecutive keys of one query row.  Lane
// (c, g) loads the 32 contiguous bytes 8 (4 s + g) .. + 7 of its key's (row's)
// head vector per step s: the k = g operands of step s of all eight
// accumulators, with no shuffle and no LDS.  Two waves per SIMD (the q rows,
// two K tiles and 8 XT accumulator tiles); the next K tile loads while this
// one's 64 (XT = 2, hd 128) MFMAs run.
// Bound: fp32 matrix rate (32 FMA per cycle and SIMD, twice the vector rate;
// fp32 MFMAs and vector instructions do not overlap).
// Every wave writes the maximum of its keys per row to smax[row][slot].
// Measured, 32 heads of 128 over 8 KV heads, against the vector kernel
// k_attn_sc it replaces here: 256 tokens at 4 096 keys 168 -> 102 us (53 us
// at the matrix rate), 512 tokens from an empty cache 30.6 -> 26.0, 29 tokens
// at 439 keys 7.8 -> 5.7.
// ---------------------------------------------------------------------------
template <int HD, int XT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_attn_scm(
    const float* __restrict__ q, const float* __restrict__ kc, const int32_t* __restrict__ pos0p, int M, int n_q,
    int n_kv, int max_seq, float scale, int qt, int tpw, float* __restrict__ S, float* __restrict__ smax) {
    constexpr int NS = HD / 32;
    const int kvh = blockIdx.x, m0 = blockIdx.y * qt, l = threadIdx.x & 63, c = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int G = n_q / n_kv, pos0 = *pos0p, slot = blockIdx.z * 4 + w;
    const int mlast = (m0 + qt < M ? m0 + qt : M) - 1, Lmax = pos0 + mlast + 1;
    int t0 = slot * 16 * tpw;
    const int t1 = min(t0 + 16 * tpw, Lmax);
    if (t0 >= t1) return;
    float qr[XT][NS][8];
    int L[XT];
    float* row[XT];
    float* slt[XT];
#pragma unroll
    for (int x = 0; x < XT; x++) {
        const int r = 16 * x + c;
        L[x] = tile_len(r, G, qt, m0, M, pos0);
        // a row past the tile repeats its first (never stored)
        const size_t rq = (size_t)(m0 + (L[x] ? r / G : 0)) * n_q + kvh * G + (L[x] ? r % G : 0);
        row[x] = S + rq * max_seq;
        slt[x] = smax + rq * ATL_SLOTS + slot;
#pragma unroll
        for (int s = 0; s < NS; s++) {
            *(float4*)&qr[x][s][0] = *(const float4*)(q + rq * HD + 8 * (4 * s + g));
            *(float4*)&qr[x][s][4] = *(const float4*)(q + rq * HD + 8 * (4 * s + g) + 4);
        }
    }
    const float* kh = kc + (size_t)kvh * max_seq * HD + 8 * g;
    float ka[NS][8], kb[NS][8];
    auto load = [&](int t, float (&k)[NS][8]) {
        const float* kp = kh + (size_t)min(t + c, max_seq - 1) * HD;
#pragma unroll
        for (int s = 0; s < NS; s++) {
            *(float4*)&k[s][0] = *(const float4*)(kp + 32 * s);
            *(float4*)&k[s][4] = *(const float4*)(kp + 32 * s + 4);
        }
    };
    float mx[XT];
#pragma unroll
    for (int x = 0; x < XT; x++) mx[x] = -1e30f;
    auto tile = [&](int t, const float (&k)[NS][8]) {
        gm_f4 acc[XT][8];
#pragma unroll
        for (int x = 0; x < XT; x++)
#pragma unroll
            for (int j = 0; j < 8; j++) acc[x][j] = (gm_f4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int j = 0; j < 8; j++)
#pragma unroll
                for (int x = 0; x < XT; x++) acc[x][j] = mfma4(k[s][j], qr[x][s][j], acc[x][j]);
        const int tq = t + 4 * g;
#pragma unroll
        for (int x = 0; x < XT; x++) {
            // hadd tree below kv_len & ~3, eng_hsum256 above it
            float sc[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float a[8];
#pragma unroll
                for (int j = 0; j < 8; j++) a[j] = acc[x][j][i];
                sc[i] = hsum8_hadd(a) * scale;
            }
            const bool hs = tq >= (L[x] & ~3) && tq < L[x];
            if (__any(hs)) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    float a[8];
#pragma unroll
                    for (int j = 0; j < 8; j++) a[j] = acc[x][j][i];
                    sc[i] = hs ? hsum8(a) * scale : sc[i];
                }
            }
            score_store4(row[x], tq, L[x], max_seq, sc, mx[x]);
        }
    };
    load(t0, ka);
    for (; t0 + 16 < t1; t0 += 32) {
        load(t0 + 16, kb);
        tile(t0, ka);
        load(t0 + 32, ka);
        tile(t0 + 16, kb);
    }
    if (t0 < t1) tile(t0, ka);
#pragma unroll
    for (int x = 0; x < XT; x++) score_max_slot(mx[x], L[x], slt[x], g);
}

// ---------------------------------------------------------------------------
// Scores over the int8 cache, the same tiling.  Lane group g holds the terms
// at 8, 0, 24, 16 (g = 0 .. 3) + L of each 32-block: the order of the pair
// path's four-term chain.  A row's last key when its kv_len is odd takes
// dot_f32_q8_blk32's two accumulators (terms L, 16 + L and 8 + L, 24 + L),
// which are the same operands with the other two lane groups' zeroed.
// Measured, 90 tokens at 790 keys: 41.8 us on the vector unit
// (k_attn_q8_sc), 18.2 here.
// ---------------------------------------------------------------------------
template <int HD, int XT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_attn_q8_scm(
    const float* __restrict__ q, DpufKvQ8 c8, const int32_t* __restrict__ pos0p, int M, int n_q, int n_kv, int max_seq,
    float scale, int qt, int tpw, float* __restrict__ S, float* __restrict__ smax) {
    constexpr int NB = HD / 32;
    const int kvh = blockIdx.x, m0 = blockIdx.y * qt, l = threadIdx.x & 63, c = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int G = n_q / n_kv, pos0 = *pos0p, slot = blockIdx.z * 4 + w;
    const int mlast = (m0 + qt < M ? m0 + qt : M) - 1, Lmax = pos0 + mlast + 1;
    int t0 = slot * 16 * tpw;
    const int t1 = min(t0 + 16 * tpw, Lmax);
    if (t0 >= t1) return;
    const int go = 8 * (g ^ 1);  // 8, 0, 24, 16
    float qr[XT][NB][8];
    int L[XT];
    float* row[XT];
    float* slt[XT];
#pragma unroll
    for (int x = 0; x < XT; x++) {
        const int r = 16 * x + c;
        L[x] = tile_len(r, G, qt, m0, M, pos0);
        const size_t rq = (size_t)(m0 + (L[x] ? r / G : 0)) * n_q + kvh * G + (L[x] ? r % G : 0);
        row[x] = S + rq * max_seq;
        slt[x] = smax + rq * ATL_SLOTS + slot;
#pragma unroll
        for (int b = 0; b < NB; b++) {
            *(float4*)&qr[x][b][0] = *(const float4*)(q + rq * HD + 32 * b + go);
            *(float4*)&qr[x][b][4] = *(const float4*)(q + rq * HD + 32 * b + go + 4);
        }
    }
    const int8_t* kh = c8.kq + (size_t)kvh * max_seq * HD + go;
    const float* sh = c8.ks + (size_t)kvh * max_seq * NB;
    struct KT {
        uint2 k[NB];
        float s[4][NB];  // scales of keys 4 g + i
    };
    auto load = [&](int t, KT& k) {
        const int8_t* kp = kh + (size_t)min(t + c, max_seq - 1) * HD;
#pragma unroll
        for (int b = 0; b < NB; b++) k.k[b] = *(const uint2*)(kp + 32 * b);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float* sp = sh + (size_t)min(t + 4 * g + i, max_seq - 1) * NB;
#pragma unroll
            for (int b = 0; b < NB; b++) k.s[i][b] = sp[b];
        }
    };
    float mx[XT];
#pragma unroll
    for (int x = 0; x < XT; x++) mx[x] = -1e30f;
    const gm_f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    auto tile = [&](int t, const KT& k) {
        const int tq = t + 4 * g;
        gm_f4 sa[XT][8];
#pragma unroll
        for (int x = 0; x < XT; x++)
#pragma unroll
            for (int j = 0; j < 8; j++) sa[x][j] = zero;
#pragma unroll
        for (int b = 0; b < NB; b++) {
            float kf[8];
#pragma unroll
            for (int j = 0; j < 8; j++) kf[j] = (float)(int8_t)((j < 4 ? k.k[b].x : k.k[b].y) >> (8 * (j & 3)));
#pragma unroll
            for (int j = 0; j < 8; j++)
#pragma unroll
                for (int x = 0; x < XT; x++) {
                    const gm_f4 d = mfma4(kf[j], qr[x][b][j], zero);
#pragma unroll
                    for (int i = 0; i < 4; i++) sa[x][j][i] = fmaf(d[i], k.s[i][b], sa[x][j][i]);
                }
            __builtin_amdgcn_sched_barrier(0);  // one block's products in registers at a time
        }
        float sc[XT][4];
        bool odd = false;
#pragma unroll
        for (int x = 0; x < XT; x++) {
            odd = odd || ((L[x] & 1) && tq <= L[x] - 1 && L[x] - 1 < tq + 4);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float a[8];
#pragma unroll
                for (int j = 0; j < 8; j++) a[j] = sa[x][j][i];
                sc[x][i] = hsum8_hadd(a) * scale;
            }
        }
        if (__any(odd)) {  // the tile holds some row's odd last key
#pragma unroll
            for (int x = 0; x < XT; x++) {
                gm_f4 tot[8];
#pragma unroll
                for (int j = 0; j < 8; j++) tot[j] = zero;
#pragma unroll
                for (int b = 0; b < NB; b++) {
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        // copies the compiler cannot trace back: it would keep
                        // every masked operand in registers across the key loop
                        uint32_t kw = j < 4 ? k.k[b].x : k.k[b].y;
                        float qv = qr[x][b][j];
                        asm volatile("" : "+v"(kw), "+v"(qv));
                        const float kv = (float)(int8_t)(kw >> (8 * (j & 3)));
                        const bool hi = (g & 1) != 0;
                        const gm_f4 a0 = mfma4(hi ? kv : 0.0f, hi ? qv : 0.0f, zero);
                        const gm_f4 a1 = mfma4(hi ? 0.0f : kv, hi ? 0.0f : qv, zero);
#pragma unroll
                        for (int i = 0; i < 4; i++) tot[j][i] = fmaf(a0[i] + a1[i], k.s[i][b], tot[j][i]);
                        asm volatile("" : "+v"(tot[j]));  // summed here, not sunk to where it is read
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    float a[8];
#pragma unroll
                    for (int j = 0; j < 8; j++) a[j] = tot[j][i];
                    if ((L[x] & 1) && tq + i == L[x] - 1) sc[x][i] = hsum8(a) * scale;
                }
            }
        }
#pragma unroll
        for (int x = 0; x < XT; x++) score_store4(row[x], tq, L[x], max_seq, sc[x], mx[x]);
    };
    KT ka, kb;
    load(t0, ka);
    for (; t0 + 16 < t1; t0 += 32) {
        load(t0 + 16, kb);
        tile(t0, ka);
        load(t0 + 32, ka);
        tile(t0 + 16, kb);
    }
    if (t0 < t1) tile(t0, ka);
#pragma unroll
    for (int x = 0; x < XT; x++) score_max_slot(mx[x], L[x], slt[x], g);
}

// ---------------------------------------------------------------------------
// Softmax and P.V.  Workgroup (kv head, tile of qt = 16 / G tokens): 16 score
// rows, HD / 32 waves, wave w the dims 32 w .. 32 w + 31 (for the int8 cache
// one 32-column block, so the reference's p * v_scale is one weight per key).
// The rows' scores stream through LDS in chunks of KC = HD / 2 keys, one
// float4 per thread:
//   pass A: e = exp(s - max) (the polynomial on the 8-aligned part, expf on
//     the tail) and the reference's eight sum lanes, one thread per (row,
//     lane), each chunk's 8 terms in order; then the reciprocal;
//   pass B: A operand p = e * inv (times v_scale), B operand V straight from
//     memory: lane (c, g) reads dims 32 w + 2 c, + 1 of key 4 i + g, 128
//     contiguous bytes per key, 8 steps ahead of their MFMAs.
// RES: every chunk keeps its LDS slot and pass B reads pass A's e; otherwise
// (rows too long for that) pass A stores e over the scores and pass B loads it
// (each thread its own elements), in two rotating slots.  A slot is [row][key % 4][key / 4 (+ 4 padding)], so four
// steps' A operands are one 16-byte read.  Keys from Lmin & ~3 on (at most
// qt + 2) are reached by some rows only and take one predicated FMA per
// output on the vector unit, so a masked key never multiplies V.
// Bound: fp32 matrix rate, then exp on the vector unit.  Measured at the 8B
// geometry against the vector kernels (softmax + P.V with the chains as FMAs
// from LDS): 256 tokens at 4 096 keys 1 433 -> 143 us (streamed), 512 tokens
// from an empty cache 48.0 -> 31.0 (resident), 29 tokens at 439 keys 40.3 ->
// 17.2, int8 cache with 90 tokens at 790 keys 86.9 + 5.0 (its O prep) -> 27.7.
// Resident rows up to 76 KB of LDS: two workgroups per CU; past that one
// workgroup per CU would leave the matrix cores to four waves, and streaming
// costs each score a store and a load.
// ---------------------------------------------------------------------------
template <int HD>
struct PvmGeo {
    static constexpr int KC = HD / 2, NI = KC / 4, GS = NI + 4, RS = 4 * GS, SLOT = 16 * RS;  // floats
    static constexpr size_t lds(int slots) {
        const size_t a = (size_t)slots * SLOT * 4, b = (size_t)16 * (HD + 4) * 4;
        return a > b ? a : b;
    }
};

template <int HD, bool Q8, bool RES>
__global__ __launch_bounds__(2 * HD) void k_attn_pvm(
    float* S, const float* __restrict__ smax, const float* __restrict__ vc, DpufKvQ8 c8,
    const int32_t* __restrict__ pos0p, int M, int n_q, int n_kv, int max_seq, int qt, int tpw,
    float* __restrict__ out, const uint8_t* __restrict__ o_sign, DpufPrep op) {
    using P = PvmGeo<HD>;
    constexpr int KC = P::KC, NI = P::NI, GS = P::GS, RS = P::RS, NB = HD / 32;
    constexpr int VS = 8;  // steps (of 4 keys) per register batch of V
    extern __shared__ __align__(16) float sm[];
    __shared__ float part[16][8], tail[16][8], rinv[16];
    const int kvh = blockIdx.x, m0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * qt;  // longest rows first
    const int tid = threadIdx.x, l = tid & 63, c = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int G = n_q / n_kv, pos0 = *pos0p;
    const int mq = (m0 + qt < M ? m0 + qt : M) - m0;
    const int Lmax = pos0 + m0 + mq, Lmin = pos0 + m0 + 1, nfull = Lmin & ~3;
    const int nch = (Lmax + KC - 1) / KC;

    // the thread's score row and its four keys of each chunk
    const int tr = tid / NI, ti = tid % NI;
    const int Lt = tile_len(tr, G, qt, m0, M, pos0), n8t = Lt & ~7;
    const size_t row0 = (size_t)m0 * n_q + kvh * G;  // score row of tile row 0
    const size_t rqt = (size_t)(Lt ? tr / G : 0) * n_q + (Lt ? tr % G : 0);
    // reads past the scores' end return 0, past a row's kv_len unused values
    const size_t left = ((size_t)M * n_q - row0) * max_seq * 4;
    const __amdgpu_buffer_rsrc_t rS = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(S + row0 * max_seq), 0, (int)(left < 0xFFFFFFFFu ? left : 0xFFFFFFFFu), ATL_RSRC3);
    const uint32_t so = (uint32_t)(rqt * max_seq + 4 * ti) * 4u;
    auto s_load = [&](int ch) {
        return __builtin_bit_cast(gm_f4, __builtin_amdgcn_raw_buffer_load_b128(rS, so + (uint32_t)(ch * KC * 4), 0, 0));
    };
    gm_f4 xn = s_load(0);
    float mx = -1e30f;
    {
        const float* mp = smax + (row0 + rqt) * ATL_SLOTS;
        const int ns = (Lt + 16 * tpw - 1) / (16 * tpw);
        for (int k = ti; k < ns; k += NI) mx = fmaxf(mx, mp[k]);
#pragma unroll
        for (int o = NI / 2; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    }
    float* const eo = sm + tr * RS + ti;
    auto l_store = [&](int sl, gm_f4 v) {
        float* e = eo + sl * P::SLOT;
#pragma unroll
        for (int k = 0; k < 4; k++) e[k * GS] = v[k];
    };
    auto e_store = [&](int ch, int sl, gm_f4 x) {
        const int t = ch * KC + 4 * ti;
        gm_f4 v;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            v[k] = exp_poly(x[k] - mx);
            if (t + k >= n8t) v[k] = t + k < Lt ? expf_libc(x[k] - mx) : 0.0f;
        }
        l_store(sl, v);
        if (!RES && Lt > 0) {
            // the thread's own scores again, for its pass B
            if (t + 3 < max_seq) {
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(gm_u4, v), rS, so + (uint32_t)(ch * KC * 4), 0, 0);
            } else {
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const float vk = v[k];
                    if (t + k < max_seq)
                        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, vk), rS,
                                                              so + (uint32_t)(ch * KC * 4) + 4 * k, 0, 0);
                }
            }
        }
    };

    // pass A
    const int cr = tid >> 3, cj = tid & 7;  // sum lane cj of row cr (the first 128 threads)
    const bool chain = tid < 128;
    const int n8c = chain ? tile_len(cr, G, qt, m0, M, pos0) & ~7 : 0;
    const float* ce = sm + (chain ? cr : 0) * RS + (cj & 3) * GS + (cj >> 2);
    float a = 0.0f;
    for (int ch = 0; ch < nch; ch++) {
        const gm_f4 x = xn;
        xn = s_load(ch + 1);
        const int sl = RES ? ch : ch & 1;
        e_store(ch, sl, x);
        __syncthreads();
        if (chain) {
            float v[KC / 8];
#pragma unroll
            for (int i = 0; i < KC / 8; i++) v[i] = ce[sl * P::SLOT + 2 * i];
#pragma unroll
            for (int i = 0; i < KC / 8; i++) a = a + (ch * KC + 8 * i < n8c ? v[i] : 0.0f);
        }
    }
    if (chain) {
        part[cr][cj] = a;
        // the row's last kv_len % 8 terms, from the last chunk(s) still in LDS
        const int t = n8c + cj, ch = t / KC, k = t % KC;
        const int Lc = tile_len(cr, G, qt, m0, M, pos0);
        tail[cr][cj] = t < Lc ? sm[(RES ? ch : ch & 1) * P::SLOT + cr * RS + (k & 3) * GS + (k >> 2)] : 0.0f;
    }
    if (!RES) xn = s_load(0);
    __syncthreads();
    if (tid < 16) {
        const int L = tile_len(tid, G, qt, m0, M, pos0);
        float sp = hsum8(part[tid]);
        for (int k = 0; k < (L & 7); k++) sp += tail[tid][k];
        rinv[tid] = 1.0f / (sp + 1e-12f);
    }
    __syncthreads();

    // pass B: wave w, dims d0 = 32 w + 2 c and d0 + 1
    const float inv = rinv[c];
    const int d0 = 32 * w + 2 * c;
    const float* Vh = Q8 ? nullptr : vc + (size_t)kvh * max_seq * HD + d0;
    const int8_t* Vq = Q8 ? c8.vq + (size_t)kvh * max_seq * HD + d0 : nullptr;
    const float* Vsc = Q8 ? c8.vs + (size_t)kvh * max_seq * NB + w : nullptr;
    struct VB {
        float2 v[Q8 ? 1 : VS];
        uint16_t b[Q8 ? VS : 1];
        float s[Q8 ? VS : 1];
    };
    // Buffer loads with the step in the scalar offset: no vector instruction
    // per load (they add to the MFMAs' time).  A step past the cache's last
    // whole one (never used) repeats that; the scalar offset is outside the
    // descriptor's range check, which covers the lane offsets of caches of
    // fewer than four rows.
    constexpr int VB1 = Q8 ? 1 : 4;  // bytes per element
    const __amdgpu_buffer_rsrc_t rV = __builtin_amdgcn_make_buffer_rsrc(
        Q8 ? (void*)(c8.vq + (size_t)kvh * max_seq * HD) : (void*)(vc + (size_t)kvh * max_seq * HD), 0,
        max_seq * HD * VB1, ATL_RSRC3);
    const __amdgpu_buffer_rsrc_t rVs = __builtin_amdgcn_make_buffer_rsrc(
        Q8 ? (void*)(c8.vs + (size_t)kvh * max_seq * NB) : (void*)S, 0, max_seq * NB * 4, ATL_RSRC3);
    const uint32_t vo = (uint32_t)(g * HD + d0) * VB1, vso = (uint32_t)(g * NB + w) * 4u;
    const int slast = max(max_seq / 4 - 1, 0);
    auto v_load = [&](int step, VB& B) {
#pragma unroll
        for (int i = 0; i < VS; i++) {
            const int st = min(step + i, slast);
            if (Q8) {
                B.b[i] = __builtin_amdgcn_raw_buffer_load_b16(rV, vo, st * 4 * HD, 0);
                const uint32_t x = __builtin_amdgcn_raw_buffer_load_b32(rVs, vso, st * 16 * NB, 0);
                B.s[i] = __builtin_bit_cast(float, x);
            } else {
                const gm_u2 x = __builtin_bit_cast(gm_u2, __builtin_amdgcn_raw_buffer_load_b64(rV, vo, st * 16 * HD, 0));
                const uint32_t x0 = x[0], x1 = x[1];
                B.v[i] = make_float2(__builtin_bit_cast(float, x0), __builtin_bit_cast(float, x1));
            }
        }
    };
    gm_f4 acc0 = {0.0f, 0.0f, 0.0f, 0.0f}, acc1 = acc0;
    const int nstep = nfull >> 2;
    const float* pa = sm + c * RS + g * GS;
    // VS steps from `step`: the A operands of the slot, MFMAs
    auto steps = [&](int step, const float* ps, const VB& B) {
        gm_f4 e4[VS / 4];
#pragma unroll
        for (int u = 0; u < VS / 4; u++) e4[u] = *(const gm_f4*)(ps + 4 * u);
        auto one = [&](int i) {
            float p = e4[i >> 2][i & 3] * inv;
            float v0, v1;
            if (Q8) {
                p = p * B.s[i];
                v0 = (float)(int8_t)(B.b[i] & 0xFF);
                v1 = (float)(int8_t)(B.b[i] >> 8);
            } else {
                v0 = B.v[i].x;
                v1 = B.v[i].y;
            }
            acc0 = mfma4(p, v0, acc0);
            acc1 = mfma4(p, v1, acc1);
        };
        if (step + VS <= nstep) {
#pragma unroll
            for (int i = 0; i < VS; i++) one(i);
        } else {
#pragma unroll
            for (int i = 0; i < VS; i++)
                if (step + i < nstep) one(i);  // uniform
        }
    };
    VB va, vb;
    v_load(0, va);
    for (int ch = 0; ch < nch; ch++) {
        const int sl = RES ? ch : ch & 1;
        if (!RES) {
            const gm_f4 x = xn;
            xn = s_load(ch + 1);
            l_store(sl, x);  // past a row's kv_len: never used
            __syncthreads();
        }
        const float* ps = pa + sl * P::SLOT;
        // NI / VS batches of steps per chunk (1, 2 or 4), two register sets
        if (NI / VS == 1) {
            v_load((ch + 1) * NI, vb);
            __builtin_amdgcn_sched_barrier(0);
            steps(ch * NI, ps, va);
            va = vb;
        } else {
#pragma unroll
            for (int u = 0; u < NI / VS; u += 2) {
                const int s0 = ch * NI + u * VS;
                v_load(s0 + VS, vb);
                __builtin_amdgcn_sched_barrier(0);
                steps(s0, ps + u * VS, va);
                v_load(s0 + 2 * VS, va);
                __builtin_amdgcn_sched_barrier(0);
                steps(s0 + VS, ps + u * VS + VS, vb);
            }
        }
        // the chunk's keys that only some rows reach
        for (int t = max(nfull, ch * KC); t < min(Lmax, (ch + 1) * KC); t++) {
            const int k = t - ch * KC;
            float v0, v1, vs = 1.0f;
            if (Q8) {
                const uint16_t b = *(const uint16_t*)(Vq + (size_t)t * HD);
                v0 = (float)(int8_t)(b & 0xFF);
                v1 = (float)(int8_t)(b >> 8);
                vs = Vsc[(size_t)t * NB];
            } else {
                const float2 v = *(const float2*)(Vh + (size_t)t * HD);
                v0 = v.x;
                v1 = v.y;
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int r = 4 * g + i;
                float p = sm[sl * P::SLOT + r * RS + (k & 3) * GS + (k >> 2)] * rinv[r];
                if (Q8) p = p * vs;
                if (t < tile_len(r, G, qt, m0, M, pos0)) {
                    acc0[i] = fmaf(p, v0, acc0[i]);
                    acc1[i] = fmaf(p, v1, acc1[i]);
                }
            }
        }
    }

    if (!op.q) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int r = 4 * g + i;
            if (tile_len(r, G, qt, m0, M, pos0) > 0)
                *(float2*)(out + (row0 + (size_t)(r / G) * n_q + r % G) * HD + d0) = make_float2(acc0[i], acc1[i]);
        }
        return;
    }
    // the prep of the O projection's input (k_prep's arithmetic): the tile to
    // LDS, then quad q = (row, 64-column block of the head), 16 columns a lane
    constexpr int LDT = HD + 4;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; i++) *(float2*)(sm + (4 * g + i) * LDT + d0) = make_float2(acc0[i], acc1[i]);
    __syncthreads();
    const int qd = n_q * HD, nb = qd >> 5;
    if (tid < HD) {
        const int bi = tid >> 2, qp = tid & 3, r = bi / (HD / 64), bh = bi % (HD / 64);
        if (tile_len(r, G, qt, m0, M, pos0) > 0) {  // whole quads
            float v[16];
            load16(sm + r * LDT + 64 * bh + 16 * qp, v);
            const int m = m0 + r / G, blk = (kvh * G + r % G) * (HD / 64) + bh;
            apply_sign_bits(v, quad_sign_bits(o_sign, blk, qp));
            quad_fwht64(v, qp);
            quad_quant_store(v, qp, blk, op.q + (size_t)m * qd, op.s + (size_t)m * nb, op.m + (size_t)m * nb,
                             op.h ? op.h + (size_t)m * qd : nullptr);
        }
    }
}

// ---------------------------------------------------------------------------

template <int HD, bool Q8>
static void launch(void* s, int M, int lmax, const float* q, const float* kc, const float* vc, DpufKvQ8 c8, float* out,
                   float* S, float* smax, const int32_t* pos0, int n_q, int n_kv, int max_seq, float scale,
                   const uint8_t* o_sign, DpufPrep op) {
    // 16-row fragments of query rows per scores wave: two where they fit two
    // waves per SIMD (int8 K is a quarter of the bytes, so one is enough)
    constexpr int XT = HD == 256 || Q8 ? 1 : 2;
    const int G = n_q / n_kv, qs = 16 * XT / G, qp = 16 / G;
    // key tiles per wave: as many as keep about two waves per SIMD, at most
    // 32 (512 keys: a wave's start, its q rows and first K tile, is paid once;
    // 256 tokens at 4 096 keys 111 us with at most 8, 102 so), and enough for
    // ATL_SLOTS slots to cover the keys
    const int kt = (lmax + 15) / 16, rt = (M + qs - 1) / qs;
    long long tpw = (long long)kt * rt * n_kv / (8 * dpuf_hip_cu_count());
    tpw = tpw < 1 ? 1 : tpw > 32 ? 32 : tpw;
    if (tpw * ATL_SLOTS < kt) tpw = (kt + ATL_SLOTS - 1) / ATL_SLOTS;
    const dim3 g1(n_kv, rt, (unsigned)((kt + 4 * tpw - 1) / (4 * tpw)));
    if (Q8)
        hipLaunchKernelGGL((k_attn_q8_scm<HD, 1>), g1, dim3(256), 0, ST(s), q, c8, pos0, M, n_q, n_kv, max_seq,
                           scale, qs, (int)tpw, S, smax);
    else
        hipLaunchKernelGGL((k_attn_scm<HD, XT>), g1, dim3(256), 0, ST(s), q, kc, pos0, M, n_q, n_kv, max_seq, scale,
                           qs, (int)tpw, S, smax);
    using P = PvmGeo<HD>;
    const int nch = (lmax + P::KC - 1) / P::KC;
    const dim3 g2(n_kv, (M + qp - 1) / qp);
    const size_t res = P::lds(nch);
    if (res <= 76 * 1024)  // two workgroups per CU at least
        hipLaunchKernelGGL((k_attn_pvm<HD, Q8, true>), g2, dim3(2 * HD), res, ST(s), S, smax, vc, c8, pos0, M, n_q,
                           n_kv, max_seq, qp, (int)tpw, out, o_sign, op);
    else {
        hipLaunchKernelGGL((k_attn_pvm<HD, Q8, false>), g2, dim3(2 * HD), P::lds(2), ST(s), S, smax, vc, c8, pos0, M,
                           n_q, n_kv, max_seq, qp, (int)tpw, out, o_sign, op);
        attn_path_note(6);
    }
}

int32_t attn_tile(void* s, int32_t M, int32_t lmax, const float* q, const float* kc, const float* vc,
                  const DpufKvQ8* c8, float* out, float* scores, const int32_t* pos0, int32_t n_q, int32_t n_kv,
                  int32_t hd, int32_t max_seq, float scale, const uint8_t* o_sign, DpufPrep op) {
    if (M < 2 || n_kv <= 0 || n_q % n_kv || (hd != 64 && hd != 128 && hd != 256)) return -1;
    const int G = n_q / n_kv;
    if ((G & 1) || G > 16) return -1;
    // 32-bit byte offsets from a tile's first score row
    if ((long long)(16 / G + 1) * n_q * max_seq * 4 >= (1ll << 31)) return -1;
    float* smax = scores + (size_t)M * n_q * max_seq;  // ATL_SLOTS floats per row
    DpufKvQ8 z;
    memset(&z, 0, sizeof z);
    if (c8) {
        if (hd == 64) launch<64, true>(s, M, lmax, q, kc, vc, *c8, out, scores, smax, pos0, n_q, n_kv, max_seq, scale, o_sign, op);
        else if (hd == 128) launch<128, true>(s, M, lmax, q, kc, vc, *c8, out, scores, smax, pos0, n_q, n_kv, max_seq, scale, o_sign, op);
        else launch<256, true>(s, M, lmax, q, kc, vc, *c8, out, scores, smax, pos0, n_q, n_kv, max_seq, scale, o_sign, op);
    } else {
        if (hd == 64) launch<64, false>(s, M, lmax, q, kc, vc, z, out, scores, smax, pos0, n_q, n_kv, max_seq, scale, o_sign, op);
        else if (hd == 128) launch<128, false>(s, M, lmax, q, kc, vc, z, out, scores, smax, pos0, n_q, n_kv, max_seq, scale, o_sign, op);
        else launch<256, false>(s, M, lmax, q, kc, vc, z, out, scores, smax, pos0, n_q, n_kv, max_seq, scale, o_sign, op);
    }
    LAUNCHED("k_attn_tile");
    return 0;
}

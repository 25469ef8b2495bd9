// Causal attention of many queries (prefill passes, prefill_attention_gpu):
// flare-core's cpu_grouped_query_attention (model.rs:9849-9966) for every
// token of a prompt.
//
// A contraction, so both products run on the matrix cores with f32 accuracy
// from split operands: binary16 caches are exact operands against q and p in
// two binary16 parts (22 bits); f32 keys and values are three bfloat16 parts
// (24 bits) against three-part q and p, the six products above 2^-24.
//
// Scores are formed transposed, S^T = K Q^T, with v_mfma_f32_32x32x16: a
// query is a lane, its 32 scores are that lane's 16 registers and those of
// lane ^ 32, so the softmax needs one cross-lane exchange, and the
// probabilities are already the operand layout of O^T = V^T P^T (the key rows
// of a tile enter with index bits 2 and 3 swapped to make it so): P never
// passes through LDS.
#pragma once

#include "attw_args.h"
#include "bgemm_args.h"
#include "bgemm_pack.h"

namespace fl {

typedef _Float16 wh8_t __attribute__((ext_vector_type(8)));
typedef __bf16 wb8_t __attribute__((ext_vector_type(8)));

template <int NP>
__device__ __forceinline__ f16x_t attw_mfma(u4x_t a, u4x_t b, f16x_t c) {
    if constexpr (NP == 1)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(wh8_t, a), __builtin_bit_cast(wh8_t, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(wb8_t, a), __builtin_bit_cast(wb8_t, b), c, 0, 0, 0);
}

// Part p of three bfloat16 parts (in the high half): the first truncated (no
// overflow), the second rounded to nearest, so the third takes either sign and
// the products that are dropped (second x third parts) have no bias.
__device__ __forceinline__ uint32_t attw_part(uint32_t u, int p) {
    return p == 1 ? u + 0x7FFFu + ((u >> 16) & 1u) : u;
}

// 8 floats as 2 binary16 parts (round toward zero, then the rest) or 3
// bfloat16 parts
template <int NP>
__device__ __forceinline__ void attw_split(const float *x, u4x_t *o) {
    if constexpr (NP == 1) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const auto h = __builtin_amdgcn_cvt_pkrtz(x[2 * i], x[2 * i + 1]);
            const auto l = __builtin_amdgcn_cvt_pkrtz(x[2 * i] - (float)h[0], x[2 * i + 1] - (float)h[1]);
            o[0][i] = __builtin_bit_cast(uint32_t, h);
            o[1][i] = __builtin_bit_cast(uint32_t, l);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            uint32_t a = __float_as_uint(x[2 * i]), b = __float_as_uint(x[2 * i + 1]);
#pragma unroll
            for (int p = 0; p < 3; p++) {
                const uint32_t ra = attw_part(a, p), rb = attw_part(b, p);
                o[p][i] = __builtin_amdgcn_perm(rb, ra, 0x07060302u);
                a = __float_as_uint(__uint_as_float(a) - __uint_as_float(ra & 0xFFFF0000u));
                b = __float_as_uint(__uint_as_float(b) - __uint_as_float(rb & 0xFFFF0000u));
            }
        }
    }
}

// 16-bit operand values (binary16, or bfloat16 planes)
template <int NP>
constexpr uint32_t kAttwExp = NP == 1 ? 0x7C00u : 0x7F80u;  // exponent of Inf and NaN
template <int NP>
__device__ __forceinline__ float attw_value(uint16_t b) {
    if constexpr (NP == 1) return h2f(b);
    else return __uint_as_float((uint32_t)b << 16);
}

// the other half's value (lane ^ 32)
__device__ __forceinline__ float attw_other(float v) { return __shfl_xor(v, 32, 64); }

// One workgroup: 4 items of one kv head (an item: 32 queries of one head;
// items of one query tile are neighbours) x 2 key lanes.  Iteration i covers
// 64 keys, key lane b its 32 from 64 i + 32 b; the two lanes' (max, sum, O)
// meet at the end.  The items share every K / V tile: K of iteration i + 1 is
// copied to LDS while the scores of i are formed, V of i + 1 while O of i is,
// in three rotating buffers.  Bound by the matrix and vector issue of each
// workgroup's chain of key tiles.  Measured on MI355X: 1531 f32 queries of 32
// heads x 128: the call, split into planes included, 4180 -> 172
// us against one query at a time on the vector units.
//
// Values that are not finite: a masked key has p = 0, but its V row is in the
// PV operand, and 0 * Inf is NaN; an Inf against the zero low part of p or q is
// NaN where the product is Inf.  Every such case leaves a NaN or Inf in O: the
// kernel then sets *a.flag (host memory), and the caller, which waits for the
// result in any case, does its work again with CAREFUL: values of V that are
// not finite are taken out of the operand and added for the queries that see
// them, and scores that came out NaN are formed again in plain f32.  Every other
// output is the same bits with and without CAREFUL.  (Both in one kernel, the
// second pass behind a vote of the workgroup, cost 1 to 3 us of every call: the
// registers of the first pass's loop fell differently.)
//
// SPLIT: few queries behind a long context have few workgroups, each a chain of
// key tiles as long as the context.  The range of keys is then cut over
// a.ksplit workgroups, which leave (max, sum, O) of theirs in memory for
// k_attw_merge.  A kernel of its own: the whole form's loop is as it was.
template <int NP, int D, bool CAREFUL, bool SPLIT>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_attw(AttwArgs a) {
    constexpr int QP = NP == 1 ? 2 : 3;  // parts of q and p
    constexpr int KS = D / 16, DT = D / 32, CH = D / 8;  // K = 16 steps, channel tiles, 16-B chunks per row
    constexpr int PLANE = 64 * D * 2, BUF = NP * PLANE;  // bytes of 64 keys
    constexpr int NL = BUF / 1024 / 8;                   // copies per wave and tile
    extern __shared__ __align__(16) char smem[];         // 3 buffers; at the end the lanes' exchange
    const int lane = threadIdx.x & 63, l31 = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), b = wave >> 2;
    const int kvh = blockIdx.x % a.nkv;
    const int ntile = (a.M + 31) / 32, items = ntile * a.group;
    const int nwg = (items + 3) / 4, ks = SPLIT ? blockIdx.x / a.nkv / nwg : 0;
    const int w = nwg - 1 - (blockIdx.x / a.nkv - ks * nwg);  // longest rows first
    const int item = min(4 * w + (wave & 3), items - 1), tile = item / a.group;
    const int head = kvh * a.group + item % a.group;
    const bool live = 4 * w + (wave & 3) < items;
    // keys: the workgroup's range ends with its last query's position
    const int last_tile = (min(4 * w + 4, items) - 1) / a.group;
    const int nkeys = a.pos0 + min(a.M, 32 * last_tile + 32);
    const int it0 = ks * a.chunk, nit = SPLIT ? min((nkeys + 63) / 64, it0 + a.chunk) : (nkeys + 63) / 64;
    if (SPLIT && it0 >= nit) return;
    const int t = 32 * tile + l31, qpos = a.pos0 + min(t, a.M - 1);
    const int tile_last = a.pos0 + min(a.M, 32 * tile + 32) - 1;  // last key any query of this item sees
    const uint16_t *kc = a.k + (size_t)kvh * a.head_stride, *vc = a.v + (size_t)kvh * a.head_stride;

    // LDS chunk p (16 B) of a K tile holds chunk c ^ g(row) of its row, g from
    // row bits 0, 1, 3 (the rows 8 lanes read together differ in those); of a V
    // tile, chunk c ^ (d >> 1 & 3) of channel row d
    auto copy_k = [&](int it, char *buf) {
#pragma unroll
        for (int u = 0; u < NL; u++) {
            const int kb = wave + 8 * u, pl = kb / (PLANE / 1024), p = (kb % (PLANE / 1024)) * 64 + lane;
            const int r = p / CH, g = (r & 3) | ((r >> 1) & 4);
            const int slot = min(64 * it + r, a.slots - 1);
            copy_to_lds((const char *)(kc + pl * a.plane + (size_t)slot * D + 8 * ((p % CH) ^ g)), buf + kb * 1024);
        }
    };
    auto copy_v = [&](int it, char *buf) {
#pragma unroll
        for (int u = 0; u < NL; u++) {
            const int kb = wave + 8 * u, pl = kb / (PLANE / 1024), p = (kb % (PLANE / 1024)) * 64 + lane;
            const int blk = min(2 * it + p / (4 * D), (a.slots >> 5) - 1), d = (p >> 2) % D;
            copy_to_lds((const char *)(vc + pl * a.plane + ((size_t)blk * D + d) * 32 + 8 * ((p & 3) ^ ((d >> 1) & 3))),
                        buf + kb * 1024);
        }
    };

    copy_k(SPLIT ? it0 : 0, smem);
    copy_v(SPLIT ? it0 : 0, smem + BUF);
    // q as operands: lane = query, part p of channels 16 k + 8 h + 0..7; binary16
    // parts are scaled by a power of two per query (their residual would
    // otherwise go subnormal for small q)
    u4x_t qf[KS][QP];
    float c = (float)(1.4426950408889634 / (D == 64 ? 8.0 : 11.313708498984761));  // log2(e) * the score scale
    float qmul = 1.0f;
    const float *qp = a.q + (size_t)min(t, a.M - 1) * a.qstride + head * D + 8 * h;
    {
        if constexpr (NP == 1) {
            float m = 0.0f;
#pragma unroll
            for (int k = 0; k < KS; k++)
#pragma unroll
                for (int j = 0; j < 8; j++) m = fmaxf(m, fabsf(qp[16 * k + j]));
            m = fmaxf(m, attw_other(m));
            // 2^e of m brought to 2^13 (zero, denormal and non-finite rows stay)
            const int e = (int)((__float_as_uint(m) >> 23) & 0xFF);
            if (e > 13 && e < 255) {
                const int s = min(max(140 - e, -100), 100);
                qmul = __uint_as_float((uint32_t)(127 + s) << 23);
                c *= __uint_as_float((uint32_t)(127 - s) << 23);
            }
        }
#pragma unroll
        for (int k = 0; k < KS; k++) {
            float x[8];
#pragma unroll
            for (int j = 0; j < 8; j++) x[j] = qp[16 * k + j] * qmul;
            attw_split<NP>(x, qf[k]);
        }
    }
    const f16x_t zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    f16x_t o[DT];
#pragma unroll
    for (int d = 0; d < DT; d++) o[d] = zero;
    float m_run = -INFINITY, l_run = 0.0f;
    // p is kept times 2^15, so its binary16 parts hold 22 bits down to 2^-18
    constexpr float kShift = NP == 1 ? 15.0f : 0.0f;
    // K row of this lane: index bits 2 and 3 swapped
    const int krow = (l31 & 0x13) | ((l31 & 4) << 1) | ((l31 & 8) >> 1);
    const int kg = (krow & 3) | ((krow >> 1) & 4);

    int bk = 0, bv = 1, bn = 2;
    for (int it = SPLIT ? it0 : 0; it < nit; it++) {
        // K of this iteration has landed (V's copies may be in flight) and
        // every wave's reads of the buffer copied to next are complete
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NL) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        copy_k(it + 1, smem + bn * BUF);  // past the end: clamped, not read
        const int kb = 64 * it + 32 * b;
        const bool work = kb <= tile_last;  // wave-uniform
        f16x_t s = zero;
        float al = 1.0f;
        if (work) {
            const char *kt = smem + bk * BUF + (size_t)(32 * b + krow) * D * 2;
            f16x_t rest = zero;  // the products of lower parts, summed apart
#pragma unroll
            for (int k = 0; k < KS; k++) {
                u4x_t kf[NP];
#pragma unroll
                for (int p = 0; p < NP; p++) kf[p] = *(const u4x_t *)(kt + p * PLANE + (((2 * k + h) ^ kg) * 16));
                if constexpr (NP == 3) {
                    rest = attw_mfma<NP>(kf[0], qf[k][2], rest);
                    rest = attw_mfma<NP>(kf[1], qf[k][1], rest);
                    rest = attw_mfma<NP>(kf[2], qf[k][0], rest);
                    rest = attw_mfma<NP>(kf[1], qf[k][0], rest);
                }
                rest = attw_mfma<NP>(kf[0], qf[k][1], rest);
                s = attw_mfma<NP>(kf[0], qf[k][0], s);
            }
#pragma unroll
            for (int i = 0; i < 16; i++) s[i] += rest[i];
            if (kb + 31 > a.pos0 + 32 * tile) {  // some query of the tile does not see every key
#pragma unroll
                for (int i = 0; i < 16; i++)
                    if (kb + 16 * (i >> 3) + 8 * h + (i & 7) > qpos) s[i] = -INFINITY;
            }
            if constexpr (CAREFUL) {
                // (one score at a time, indexed by selects: registers matter here, time does not)
                const float *qr = qp - 8 * h;
                const char *k0 = smem + bk * BUF + 32 * b * D * 2;
#pragma unroll 1
                for (int i = 0; i < 16; i++) {
                    float v = s[0];
#pragma unroll
                    for (int j = 1; j < 16; j++) v = i == j ? s[j] : v;
                    if (v == v) continue;
                    const int key = 16 * (i >> 3) + 8 * h + (i & 7), g = (key & 3) | ((key >> 1) & 4);
                    v = 0.0f;
#pragma unroll 1
                    for (int d = 0; d < D; d++) {
                        const char *kp = k0 + key * D * 2 + (((d >> 3) ^ g) * 16) + (d & 7) * 2;
                        float kv = attw_value<NP>(*(const uint16_t *)kp);
                        if constexpr (NP == 3)
                            kv += attw_value<NP>(*(const uint16_t *)(kp + PLANE)) +
                                  attw_value<NP>(*(const uint16_t *)(kp + 2 * PLANE));
                        v = __builtin_fmaf(qr[d] * qmul, kv, v);
                    }
#pragma unroll
                    for (int j = 0; j < 16; j++) s[j] = i == j ? v : s[j];
                }
            }
            float m = s[0];
#pragma unroll
            for (int i = 1; i < 16; i++) m = fmaxf(m, s[i]);
            m = fmaxf(m, attw_other(m)) * c;
            if (__any(m > m_run)) {
                const float mn = fmaxf(m_run, m);
                al = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - mn);
                m_run = mn;
            }
            // a query that has seen no key yet keeps p = 0
            const float off = m_run == -INFINITY ? -INFINITY : kShift - m_run;
            float ps = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const float x = __builtin_fmaf(s[i], c, off);
                const float p = __builtin_amdgcn_exp2f(x);
                s[i] = s[i] == -INFINITY ? 0.0f : p;
                ps += s[i];
            }
            l_run = __builtin_fmaf(l_run, al, ps);
        }
        // V of this iteration has landed
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NL) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        copy_v(it + 1, smem + bk * BUF);  // every wave is past its reads of K
        if (work) {
            const char *vt = smem + bv * BUF + 32 * b * D * 2;
            u4x_t pf[2][QP];
#pragma unroll
            for (int mm = 0; mm < 2; mm++) {
                float x[8];
#pragma unroll
                for (int j = 0; j < 8; j++) x[j] = s[8 * mm + j];
                attw_split<NP>(x, pf[mm]);
            }
            // a tile's products are summed by themselves, low parts first, so O
            // is rounded once per 32 keys
#pragma unroll
            for (int d = 0; d < DT; d++) {
                const int dd = 32 * d + l31;
                u4x_t vf[2][NP];
#pragma unroll
                for (int mm = 0; mm < 2; mm++)
#pragma unroll
                    for (int p = 0; p < NP; p++)
                        vf[mm][p] = *(const u4x_t *)(vt + p * PLANE + dd * 64 + (((2 * mm + h) ^ ((dd >> 1) & 3)) * 16));
                uint32_t bad = 0;  // CAREFUL: keys of the tile whose V row is not finite in these channels
                if constexpr (CAREFUL) {
                    constexpr uint32_t E = kAttwExp<NP>;
#pragma unroll
                    for (int mm = 0; mm < 2; mm++)
#pragma unroll
                        for (int j = 0; j < 8; j++) {
                            const uint32_t w = vf[mm][0][j >> 1], sh = 16 * (j & 1);
                            if (((w >> sh) & E) != E) continue;
                            vf[mm][0][j >> 1] = w & ~(0xFFFFu << sh);
                            bad |= 1u << (16 * mm + 8 * h + j);
                        }
#pragma unroll
                    for (int x = 1; x < 64; x <<= 1) bad |= __shfl_xor(bad, x, 64);
                }
                f16x_t pv = zero;
#pragma unroll
                for (int mm = 0; mm < 2; mm++) {
                    if constexpr (NP == 3) {
                        pv = attw_mfma<NP>(vf[mm][0], pf[mm][2], pv);
                        pv = attw_mfma<NP>(vf[mm][1], pf[mm][1], pv);
                        pv = attw_mfma<NP>(vf[mm][2], pf[mm][0], pv);
                        pv = attw_mfma<NP>(vf[mm][1], pf[mm][0], pv);
                    }
                    pv = attw_mfma<NP>(vf[mm][0], pf[mm][1], pv);
                }
#pragma unroll
                for (int mm = 0; mm < 2; mm++) pv = attw_mfma<NP>(vf[mm][0], pf[mm][0], pv);
#pragma unroll
                for (int i = 0; i < 16; i++) o[d][i] = __builtin_fmaf(o[d][i], al, pv[i]);
                if constexpr (CAREFUL) {
                    for (; bad; bad &= bad - 1) {  // uniform
                        const int key = __builtin_ctz(bad);
                        float p = s[0];
#pragma unroll
                        for (int i = 1; i < 16; i++) p = i == (((key >> 4) << 3) | (key & 7)) ? s[i] : p;
                        p = __shfl(p, l31 + 32 * ((key >> 3) & 1), 64);
                        if (kb + key > qpos) continue;
                        int h4 = 4 * h;
                        asm volatile("" : "+v"(h4));  // the addresses below are formed here, not kept
#pragma unroll
                        for (int i = 0; i < 16; i++) {
                            const int ch = 32 * d + 8 * (i >> 2) + h4 + (i & 3);
                            const uint16_t v =
                                *(const uint16_t *)(vt + ch * 64 + (((key >> 3) ^ ((ch >> 1) & 3)) * 16) + (key & 7) * 2);
                            if ((v & kAttwExp<NP>) == kAttwExp<NP>) o[d][i] = __builtin_fmaf(p, attw_value<NP>(v), o[d][i]);
                        }
                    }
                }
            }
        }
        const int x = bk;  // next: K in the free buffer, V in this K's, free this V's
        bk = bn;
        bn = bv;
        bv = x;
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // the clamped copies, before LDS is reused
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    l_run += attw_other(l_run);

    // key lane 1 hands (m, l, O) to lane 0 through LDS, two channel tiles at a
    // time: [4 items][64 lanes][32 + 2] floats
    float *ex = (float *)smem + (size_t)((wave & 3) * 64 + lane);
    float wa = 1.0f, wb = 0.0f;
#pragma unroll
    for (int d0 = 0; d0 < DT; d0 += 2) {
        if (b == 1) {
#pragma unroll
            for (int d = 0; d < 2; d++)
#pragma unroll
                for (int i = 0; i < 16; i++) ex[(16 * d + i) * 256] = o[d0 + d][i];
            if (d0 == 0) {
                ex[32 * 256] = m_run;
                ex[33 * 256] = l_run;
            }
        }
        __syncthreads();
        if (b == 0) {
            if (d0 == 0) {
                const float m1 = ex[32 * 256], l1 = ex[33 * 256], mn = fmaxf(m_run, m1);
                // every query sees key 0, which is lane 0's (of split 0)
                wa = SPLIT && m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - mn);
                wb = m1 == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m1 - mn);
                if constexpr (SPLIT) {
                    l_run = l_run * wa + l1 * wb;
                    m_run = mn;
                } else {
                    const float il = 1.0f / (l_run * wa + l1 * wb);
                    wa *= il;
                    wb *= il;
                }
            }
#pragma unroll
            for (int d = 0; d < 2; d++)
#pragma unroll
                for (int i = 0; i < 16; i++) o[d0 + d][i] = o[d0 + d][i] * wa + ex[(16 * d + i) * 256] * wb;
        }
        __syncthreads();
    }
    if (b == 1 || !live) return;
    if ((SPLIT || a.out) && t < a.M) {
        float *op = (SPLIT ? a.part + (size_t)ks * a.M * a.qstride : a.out) + (size_t)t * a.qstride + head * D;
#pragma unroll
        for (int d = 0; d < DT; d++)
#pragma unroll
            for (int g = 0; g < 4; g++)
                *(v4f_t *)(op + 32 * d + 8 * g + 4 * h) =
                    v4f_t{o[d][4 * g], o[d][4 * g + 1], o[d][4 * g + 2], o[d][4 * g + 3]};
    }
    if constexpr (SPLIT) {
        if (h == 0 && t < a.M) {
            float *ml = a.ml + (((size_t)ks * a.M + t) * a.nkv * a.group + head) * 2;
            ml[0] = m_run;
            ml[1] = l_run;
        }
        return;
    }
    if (a.xp) {
        // quantize_input_q8_0_into (model.rs:5534-5571) of the row, per 32 channels
#pragma unroll
        for (int d = 0; d < DT; d++) {
            float amax = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; i++) amax = fmaxf(amax, fabsf(o[d][i]));
            amax = fmaxf(amax, attw_other(amax));
            const float qd = amax / 127.0f, id = (qd != 0.0f) ? 127.0f / amax : 0.0f;
            const int blk = head * DT + d;
            char *rec = a.xp + ((size_t)tile * a.nst + (blk >> 3)) * kPackRec;
            int sum = 0;
#pragma unroll
            for (int g = 0; g < 4; g++) {
                int q[4];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    q[i] = q8_code(o[d][4 * g + i] * id);
                    sum += q[i];
                }
                pack_codes4(rec, l31, (blk & 7) * 32 + 8 * g + 4 * h, q[0], q[1], q[2], q[3]);
            }
            sum += __shfl_xor(sum, 32, 64);
            if (h == 0) pack_scale(rec, l31, blk & 7, qd, sum);
        }
    }
    if constexpr (!CAREFUL) {
        float n[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int d = 0; d < DT; d++)
#pragma unroll
            for (int i = 0; i < 16; i++) n[i & 3] = __builtin_fmaf(o[d][i], 0.0f, n[i & 3]);
        if ((n[0] + n[1]) + (n[2] + n[3]) != 0.0f)  // 0 * Inf and 0 * NaN are NaN
            __hip_atomic_store(a.flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// The splits' (max, sum, O) into the result: 1024 channels of a token per
// workgroup, 4 a thread (workgroups mapped as pack_wg says).
template <int D>
__global__ __launch_bounds__(256) void k_attw_merge(AttwArgs a) {
    int t, chunk;
    pack_wg((a.qstride + 1023) >> 10, t, chunk);
    if (t >= a.M) return;
    const int e = chunk * 1024 + 4 * threadIdx.x, ec = min(e, a.qstride - 4), nh = a.nkv * a.group;
    // splits that hold a key which some query of the token's tile sees
    const int last = a.pos0 + min(a.M, (t & ~31) + 32) - 1, n = min(a.ksplit, (last >> 6) / a.chunk + 1);
    // batches of U splits, so that their loads are in flight together (one at a
    // time 11.5 us for 64 tokens of 16 heads x 64 and 22 splits, so 9.2)
    constexpr int U = 8;
    const size_t mls = (size_t)a.M * nh * 2, ps = (size_t)a.M * a.qstride;
    const float *ml = a.ml + ((size_t)t * nh + ec / D) * 2, *part = a.part + (size_t)t * a.qstride + ec;
    float m = -INFINITY, l = 0.0f;
    for (int k = 0; k < n; k += U) {
        float mk[U];
#pragma unroll
        for (int u = 0; u < U; u++) mk[u] = ml[min(k + u, n - 1) * mls];
#pragma unroll
        for (int u = 0; u < U; u++) m = fmaxf(m, mk[u]);
    }
    v4f_t o = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int k = 0; k < n; k += U) {
        float mk[U], lk[U];
        v4f_t p[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i = min(k + u, n - 1);
            mk[u] = ml[i * mls];
            lk[u] = ml[i * mls + 1];
            p[u] = *(const v4f_t *)(part + i * ps);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (k + u >= n) break;
            const float wk = mk[u] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mk[u] - m);
            l = __builtin_fmaf(lk[u], wk, l);
#pragma unroll
            for (int j = 0; j < 4; j++) o[j] = __builtin_fmaf(p[u][j], wk, o[j]);
        }
    }
    const float il = 1.0f / l;
    float y[4], nan = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        y[j] = o[j] * il;
        nan = __builtin_fmaf(y[j], 0.0f, nan);
    }
    if (a.flag && nan != 0.0f) __hip_atomic_store(a.flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (a.out && e < a.qstride) *(v4f_t *)(a.out + (size_t)t * a.qstride + e) = v4f_t{y[0], y[1], y[2], y[3]};
    if (a.xp) pack_block8(y, e < a.qstride, a.xp + ((size_t)(t >> 5) * a.nst + (ec >> 8)) * kPackRec, t, e & 255);
}

// f32 rows (FMT 0) or a Q8 cache (FMT 1) into three bfloat16 planes; slots
// T .. the next multiple of 32 become zeros.  CAREFUL: Inf and NaN in the first
// plane alone.  grid (32-slot blocks, kv heads)
template <int FMT, int D, bool CAREFUL>
__global__ __launch_bounds__(256) void k_attw_split(AttwSplitArgs a) {
    __shared__ float lv[32][D + 1];
    const int blk = blockIdx.x, kvh = blockIdx.y;
    auto value = [&](const void *p, const uint16_t *sc, int r, int d, bool tblk) -> float {
        const int s = 32 * blk + r;
        if (s >= a.T) return 0.0f;
        if constexpr (FMT == 0) {
            return ((const float *)p)[(size_t)kvh * a.head_stride + (size_t)s * a.tok_stride + d];
        } else {  // V in transposed blocks [slot / 32][D][32]
            const size_t e = (size_t)kvh * a.head_stride + (tblk ? ((size_t)blk * D + d) * 32 + r : (size_t)s * D + d);
            return (float)((const int8_t *)p)[e] * h2f(sc[((size_t)kvh * a.S + s) * (D / 32) + (d >> 5)]);
        }
    };
    auto put = [&](uint16_t *o, size_t at, float v) {
        if (CAREFUL && v != v) v = __uint_as_float(0x7FC00000u);
        const bool fin = !CAREFUL || fabsf(v) < INFINITY;
#pragma unroll
        for (int p = 0; p < 3; p++) {
            const uint32_t u = attw_part(__float_as_uint(v), p);
            o[p * a.plane + at] = (uint16_t)(u >> 16);
            v = fin ? v - __uint_as_float(u & 0xFFFF0000u) : 0.0f;
        }
    };
    const size_t base = (size_t)kvh * a.out_stride + (size_t)blk * 32 * D;
    for (int i = threadIdx.x; i < 32 * D; i += 256) {
        const int r = i / D, d = i % D;
        put(a.ko, base + i, value(a.k, a.ks, r, d, false));
        if (FMT == 0) lv[r][d] = value(a.v, a.vs, r, d, false);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 32 * D; i += 256) {
        const int d = i >> 5, r = i & 31;
        put(a.vo, base + i, FMT == 1 ? value(a.v, a.vs, r, d, true) : lv[r][d]);
    }
}

}  // namespace fl

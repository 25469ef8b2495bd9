// Large-batch quantized GEMM (more than 16 tokens): the projections of
// prefill passes and of batched_dequant_matmul (flare-core/src/model.rs:
// 740-1036, one quantized matvec per token there).
//
// The work is a contraction with per-32-block scales: out[t][r] = sum over
// blocks of s[t] * d[r] * dot(q_x[t], q_w[r]).  The dots go to the f16 matrix
// cores with exact operands: activation codes are integers below 128 and
// weight codes (Q4_K: less 8, times their 6-bit sub-block scale) integers below
// 1024, so one v_mfma_f32_32x32x16_f16 pair holds sc * dot of a block exactly
// (< 2^24) and what is left for the vector units is one fused multiply-add
// per output and block (the token's scale; a token is a lane of the MFMA's
// result, so that scale is one register).
#pragma once

#include "bgemm_pack.h"
#include "verify_args.h"

namespace fl {

__device__ __forceinline__ h8x_t as_h8(u4x_t v) { return __builtin_bit_cast(h8x_t, v); }
__device__ __forceinline__ uint32_t h2_bits(h2x_t v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ h2x_t bits_h2(uint32_t v) { return __builtin_bit_cast(h2x_t, v); }
__device__ __forceinline__ h2x_t h2_both(float v) { return h2x_t{(_Float16)v, (_Float16)v}; }

// 8 nibbles (LOW / high ones of two dwords) less 8, times the sub-block scale,
// as binary16, order 0 2 1 3 4 6 5 7.  A nibble n in bits 4..7 under 0x5400 is
// 64 + n, so fma(v, sc, -72 sc) is sc * (n - 8), exact (72 sc < 2^13 has at
// most 10 significant bits).  Less 8: the codes' mean would otherwise double
// the sums, and with them their rounding, before the min terms take it out
// again.
template <bool LOW>
__device__ __forceinline__ void q4_pairs(uint32_t w0, uint32_t w1, h2x_t mul, h2x_t add, uint32_t (&o)[4]) {
    constexpr uint32_t m = 0x00F000F0u;
    uint32_t e = 0x54005400u;
    asm("" : "+v"(e));  // in a register: v_and_or_b32 takes one constant
    const uint32_t v[4] = {((LOW ? w0 << 4 : w0) & m) | e, ((w0 >> (LOW ? 4 : 8)) & m) | e,
                           ((LOW ? w1 << 4 : w1) & m) | e, ((w1 >> (LOW ? 4 : 8)) & m) | e};
#pragma unroll
    for (int i = 0; i < 4; i++) o[i] = h2_bits(__builtin_elementwise_fma(bits_h2(v[i]), mul, add));
}

// 8 int8 codes of two dwords as binary16 in the same order: (q ^ 0x80) is
// q + 128, 0x6400 | that is 1152 + q.
__device__ __forceinline__ void i8_pairs(uint32_t w0, uint32_t w1, uint32_t (&o)[4]) {
    const h2x_t bias = {(_Float16)1152.0f, (_Float16)1152.0f};
    const uint32_t a = w0 ^ 0x80808080u, b = w1 ^ 0x80808080u;
    const uint32_t v[4] = {__builtin_amdgcn_perm(0x64646464u, a, 0x04020400u),
                           __builtin_amdgcn_perm(0x64646464u, a, 0x04030401u),
                           __builtin_amdgcn_perm(0x64646464u, b, 0x04020400u),
                           __builtin_amdgcn_perm(0x64646464u, b, 0x04030401u)};
#pragma unroll
    for (int i = 0; i < 4; i++) o[i] = h2_bits(bits_h2(v[i]) - bias);
}

// quantize_input_q8_0_into (model.rs:5534-5571) of M f32 rows into packed
// records: one wave per (tile, block), a lane holds half a block of a token.
__global__ __launch_bounds__(256) void k_quant_pack(const float *x, int M, int K, int nst, char *xp) {
    const int lane = threadIdx.x & 63, blk = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (blk * 32 >= K) return;
    const int tile = blockIdx.x, l31 = lane & 31, h = lane >> 5;
    const int t = min(tile * kPackTile + l31, M - 1);
    const v4f_t *src = (const v4f_t *)(x + (size_t)t * K + blk * 32 + 16 * h);
    float v[16];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const v4f_t u = src[j];
        v[4 * j] = u.x; v[4 * j + 1] = u.y; v[4 * j + 2] = u.z; v[4 * j + 3] = u.w;
    }
    float amax = 0.0f;
#pragma unroll
    for (int j = 0; j < 16; j++) amax = fmaxf(amax, fabsf(v[j]));
    amax = fmaxf(amax, __shfl_xor(amax, 32, 64));
    const float d = amax / 127.0f;
    const float id = (d != 0.0f) ? 127.0f / amax : 0.0f;
    int sum = 0;
    h8x_t c[2];
#pragma unroll
    for (int j = 0; j < 16; j++) {
        const int8_t q = q8_code(v[j] * id);
        sum += q;
        const int e = (j & 4) | ((j & 1) << 1) | ((j >> 1) & 1);
        c[j >> 3][e] = (_Float16)(float)q;
    }
    sum += __shfl_xor(sum, 32, 64);
    char *rec = xp + ((size_t)tile * nst + (blk >> 3)) * kPackRec;
    char *o = rec + (blk & 7) * 2048 + lane * 16;
    *(h8x_t *)o = c[0];
    *(h8x_t *)(o + 1024) = c[1];
    if (h == 0) pack_scale(rec, l31, blk & 7, d, sum);
}

__device__ __forceinline__ v4f_t part_sum4(const float *part, int ksplit, size_t plane, size_t at) {
    v4f_t v = *(const v4f_t *)(part + at);
    for (int k = 1; k < ksplit; k++) v += *(const v4f_t *)(part + k * plane + at);
    return v;
}

// Residual add, RMSNorm and Q8_0 quantization of M tokens as k_v_resnorm
// (rmsnorm_quantize_q8_0 / rmsnorm_into + quantize, model.rs:5581-5640 /
// 7456-7477), the codes into packed records.  One workgroup per token.
template <int PRO>
__global__ __launch_bounds__(kResnormThreads) void k_b_resnorm(const float *part, int ksplit, int M, int H, float *x,
                                                                const float *w, float eps, int nst, char *xp) {
    __shared__ float red[kResnormThreads / 64];
    int t, chunk;
    pack_wg(1, t, chunk);
    if (t >= M) return;
    const int tid = threadIdx.x;
    float *xt = x + (size_t)t * H;
    v4f_t v[kResnormChunks], wv[kResnormChunks];
    float ss = 0.0f;
#pragma unroll
    for (int c = 0; c < kResnormChunks; c++) {
        const int e = 4 * (tid + c * kResnormThreads);
        v[c] = wv[c] = v4f_t{0.0f, 0.0f, 0.0f, 0.0f};
        if (e < H) {
            v[c] = *(const v4f_t *)(xt + e);
            wv[c] = *(const v4f_t *)(w + e);
            if (part) {
                v[c] += part_sum4(part, ksplit, (size_t)M * H, (size_t)t * H + e);
                *(v4f_t *)(xt + e) = v[c];
            }
        }
        ss += v[c].x * v[c].x + v[c].y * v[c].y + v[c].z * v[c].z + v[c].w * v[c].w;
    }
    ss = wave_sum(ss);
    if ((tid & 63) == 0) red[tid >> 6] = ss;
    __syncthreads();
    ss = 0.0f;
#pragma unroll
    for (int i = 0; i < kResnormThreads / 64; i++) ss += red[i];
    const float inv = 1.0f / sqrtf(ss / (float)H + eps);
#pragma unroll
    for (int c = 0; c < kResnormChunks; c++) {
        const int e = 4 * (tid + c * kResnormThreads);
        if (c * 4 * kResnormThreads >= H) break;  // uniform: shuffles below
        float y[4];
#pragma unroll
        for (int j = 0; j < 4; j++) y[j] = (PRO == PRO_NORMQ0) ? v[c][j] * wv[c][j] * inv : (v[c][j] * inv) * wv[c][j];
        pack_block8(y, e < H, xp + ((size_t)(t >> 5) * nst + (min(e, H - 4) >> 8)) * kPackRec, t, e & 255);
    }
}

// SiLU(g) * u (silu_mul_into, model.rs:9783-9796) of the gate/up partials and
// its Q8_0 quantization into packed records; 1024 hidden units of a token per
// workgroup.
__global__ __launch_bounds__(256) void k_b_silu(const float *part, int ksplit, int M, int F, int nst, char *xp) {
    int t, chunk;
    pack_wg((F + 1023) >> 10, t, chunk);
    if (t >= M) return;
    const int e = chunk * 1024 + 4 * threadIdx.x, ec = min(e, F - 4);  // F % 32 == 0
    const size_t plane = (size_t)M * 2 * F, at = (size_t)t * 2 * F + ec;
    const v4f_t g = part_sum4(part, ksplit, plane, at), u = part_sum4(part, ksplit, plane, at + F);
    float y[4];
#pragma unroll
    for (int j = 0; j < 4; j++) y[j] = (g[j] / (1.0f + fl_expf(-g[j]))) * u[j];
    pack_block8(y, e < F, xp + ((size_t)(t >> 5) * nst + (ec >> 8)) * kPackRec, t, e & 255);
}

// x[i] += partials of one row (part: that row of split 0; splits `plane` apart)
__global__ __launch_bounds__(256) void k_b_residual_row(const float *part, int ksplit, size_t plane, int H, float *x) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= H) return;
    float v = part[i];
    for (int k = 1; k < ksplit; k++) v += part[k * plane + i];
    x[i] += v;
}

// One workgroup: NW waves of 32 weight rows, TT tiles of 32 tokens; K in steps
// of 256 values.  Weights go from memory to registers (every row belongs to
// one wave; the next step's are in flight), activations through a
// double-buffered LDS slot that all waves share, copied there without
// registers while the step before is consumed.  Bound by vector issue (the
// multiply-adds of the block scales, the unpacking, the MFMAs' own issue), not
// by memory.  Measured on MI355X: 14336 x 4096 Q4_K, 1000 rows 188 us (624
// TFLOP/s; the call 4100 -> 213 us against 16 rows a launch).
template <int FMT, int TT, int NW>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_bgemm(BgArgs a) {
    extern __shared__ __align__(16) char smem[];  // [2][TT][kPackRec], then [NW][32] floats
    constexpr int RC = FMT == F_Q4K ? kPackRec / 1024 : kPackMin / 1024;  // KiB copied per record
    const WDesc &W = a.W;
    const int lane = threadIdx.x & 63, l31 = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // workgroups of one XCD (blockIdx % 8) walk neighbouring tiles: 4 token
    // tiles of one row tile, then the next row tile, so both operands are
    // shared in that XCD's L2
    int wg = blockIdx.x;
    {
        const int n = gridDim.x, per = n >> 3, rem = n & 7, x = wg & 7, i = wg >> 3;
        wg = x * per + min(x, rem) + i;
    }
    const int per_split = a.nrt * a.ntt, ks = wg / per_split;
    int r = wg % per_split, rt, ct;
    {
        const int full = (a.ntt >> 2) * 4 * a.nrt;
        const int g = r < full ? r / (4 * a.nrt) : a.ntt >> 2, w4 = r < full ? 4 : a.ntt & 3;
        r -= g * 4 * a.nrt;
        rt = r / w4;
        ct = g * 4 + r % w4;
    }
    const int s0 = ks * a.chunk, s1 = min(a.nst, s0 + a.chunk);
    const int tile0 = ct * TT, ntile = (a.M + kPackTile - 1) / kPackTile;
    const int row0 = (rt * NW + wave) * 32;
    const size_t row = min(row0 + l31, W.rows - 1);

    const uint32_t lane16 = lane * 16;
    auto stage = [&](int buf, int st) {
#pragma unroll
        for (int c = 0; c < (TT * RC + NW - 1) / NW; c++) {
            const int p = wave + c * NW, tt = p / RC, kb = p % RC;
            if ((c + 1) * NW > TT * RC && p >= TT * RC) break;  // the last round may be partial
            // 32-bit scalar offset (packed activations are below 4 GiB): the
            // lanes' part of the address is then one register for all copies
            uint32_t off = (uint32_t)(min(tile0 + tt, ntile - 1) * a.nst + st) * kPackRec + kb * 1024;
            asm("" : "+s"(off));
            copy_to_lds(a.xp + off + lane16, smem + (buf * TT + tt) * kPackRec + kb * 1024);
        }
    };

    f16x_t acc[TT];
#pragma unroll
    for (int tt = 0; tt < TT; tt++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[tt][i] = 0.0f;
    const f16x_t zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

    if constexpr (FMT == F_Q4K) {
        float *dl = (float *)(smem + 2 * TT * kPackRec) + wave * 32;  // d of the wave's rows
        const uint8_t *qp = W.q + row * a.nst * 128 + 16 * h, *hp = W.h + row * a.nst * 16;
        // Weights: one step in registers; a piece is loaded again for the next
        // step as soon as its codes are unpacked.
        u4x_t w[4], hd;
        auto wload = [&](int st, int j) { w[j] = *(const u4x_t *)(qp + (size_t)st * 128 + 32 * j); };
        stage(0, s0);
        asm volatile("" ::: "memory");  // the copies first: the wait below counts the loads after them
#pragma unroll
        for (int j = 0; j < 4; j++) wload(s0, j);
        hd = *(const u4x_t *)(hp + (size_t)s0 * 16);
        for (int st = s0; st < s1; st++) {
            const int cur = (st - s0) & 1, nx = min(st + 1, s1 - 1);
            // this wave's copies have landed (loads complete in order, and the
            // five weight loads issued after them may be in flight) and its
            // reads of the other buffer are complete
            asm volatile("s_waitcnt vmcnt(5) lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            if (st + 1 < s1) stage(cur ^ 1, nx);
            asm volatile("" ::: "memory");
            const char *buf = smem + cur * TT * kPackRec;
            // unpack_q4k_scales (model.rs:8709-8719), flare packing
            const uint32_t sa = hd[1], sb = hd[2], sc = hd[3];
            if (h == 0) dl[l31] = h2f((uint16_t)(hd[0] & 0xFFFF));
            // Blocks in the order 0 4 1 5 2 6 3 7 (two share their bytes), TT
            // token tiles each: unit i = (block i / TT, tile i % TT).  The
            // multiply-adds of unit i - 1 are issued between the two MFMAs of
            // unit i and after them, so the matrix and the vector units of the
            // SIMD work at once (in the order the compiler chose, each unit's
            // MFMAs, a wait, then its multiply-adds, two 8B-shaped layers and
            // 4096 tokens took 7.85 ms against 6.85).  What bounds it then is
            // vector issue: ~1000 instructions and 76 MFMAs per wave and step,
            // two waves per SIMD, fill ~90 % of its slots.
            f16x_t C[TT], dd[2];
            h8x_t A[2], B[2][2];
            float s3[3];
            auto unpack = [&](int bi, int half) {  // half of block bi's weight operand
                const int j = bi >> 1, hi = bi & 1;
                const uint32_t s8 = (sa >> (8 * j)) & 0xFF;
                const uint32_t six = hi ? (s8 >> 6) | (((sc >> (8 * j)) & 0xF) << 2) : s8 & 63;
                const float fs = (float)six;
                const h2x_t mul = h2_both(fs), add = h2_both(fs * -72.0f);
                uint32_t o[4];
                if (hi) q4_pairs<false>(w[j][2 * half], w[j][2 * half + 1], mul, add, o);
                else q4_pairs<true>(w[j][2 * half], w[j][2 * half + 1], mul, add, o);
                A[half] = as_h8(u4x_t{o[0], o[1], o[2], o[3]});
                if (hi && half) wload(nx, j);
            };
            auto fetch = [&](int i) {  // unit i's activations
                const int bi = i / TT, blk = (bi >> 1) + 4 * (bi & 1);
                const char *rec = buf + (i % TT) * kPackRec;
                B[i & 1][0] = *(const h8x_t *)(rec + blk * 2048 + lane * 16);
                B[i & 1][1] = *(const h8x_t *)(rec + blk * 2048 + 1024 + lane * 16);
                s3[i % 3] = *(const float *)(rec + kPackScale + blk * 128 + l31 * 4);
            };
            auto madd = [&](int i, int half) {  // half of unit i's multiply-adds
                const int tt = i % TT;
                const float sv = s3[i % 3];
#pragma unroll
                for (int e = 8 * half; e < 8 * half + 8; e++)
                    C[tt][e] = i < TT ? sv * dd[i & 1][e] : __builtin_fmaf(sv, dd[i & 1][e], C[tt][e]);
            };
            unpack(0, 0);
            unpack(0, 1);
            fetch(0);
#pragma unroll
            for (int i = 0; i < 8 * TT; i++) {
                const int bi = i / TT, tt = i % TT;
                __builtin_amdgcn_sched_barrier(0);
                dd[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[0], B[i & 1][0], zero, 0, 0, 0);
                if (i + 1 < 8 * TT) fetch(i + 1);
                if (i > 0) madd(i - 1, 0);
                if (bi < 7 && tt == TT - 1) unpack(bi + 1, 0);  // its operand has just been read
                __builtin_amdgcn_sched_barrier(0);
                dd[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[1], B[i & 1][1], dd[i & 1], 0, 0, 0);
                if (i > 0) madd(i - 1, 1);
                if (bi < 7 && tt == TT - 1) unpack(bi + 1, 1);
            }
            __builtin_amdgcn_sched_barrier(0);
            madd(8 * TT - 1, 0);
            madd(8 * TT - 1, 1);
            // acc += d * C + sum_j c_j (s sum q)_j, c_j = 8 d sc_j - dmin mn_j
            // (C holds codes less 8): c_j and s sum q as three bfloat16 parts
            // each, the products of parts down to 2^-24 summed by the MFMA
            const float d8 = 8.0f * h2f((uint16_t)(hd[0] & 0xFFFF)), dmin = h2f((uint16_t)(hd[0] >> 16));
            uint32_t cp[3][4];
#pragma unroll
            for (int p = 0; p < 4; p++) {
                uint32_t part[2][3];
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const int j = 2 * p + e, jj = j & 3;
                    const uint32_t s8 = (sa >> (8 * jj)) & 0xFF, m8 = (sb >> (8 * jj)) & 0xFF, u8 = sc >> (8 * jj);
                    const uint32_t six = j >= 4 ? (s8 >> 6) | ((u8 & 0xF) << 2) : s8 & 63;
                    const uint32_t mn = j >= 4 ? (m8 >> 6) | (((u8 >> 4) & 0xF) << 2) : m8 & 63;
                    float v = __builtin_fmaf(d8, (float)six, -(dmin * (float)mn));
#pragma unroll
                    for (int k = 0; k < 3; k++) {
                        part[e][k] = __float_as_uint(v);
                        v -= __uint_as_float(part[e][k] & 0xFFFF0000u);
                    }
                }
#pragma unroll
                for (int k = 0; k < 3; k++) cp[k][p] = __builtin_amdgcn_perm(part[1][k], part[0][k], 0x07060302u);
            }
            hd = *(const u4x_t *)(hp + (size_t)nx * 16);
            const b8x_t c1 = __builtin_bit_cast(b8x_t, u4x_t{cp[0][0], cp[0][1], cp[0][2], cp[0][3]});
            const b8x_t c2 = __builtin_bit_cast(b8x_t, u4x_t{cp[1][0], cp[1][1], cp[1][2], cp[1][3]});
            const uint32_t hmask = 0u - (uint32_t)h;  // (a select here went through memory)
            u4x_t c13;
#pragma unroll
            for (int k = 0; k < 4; k++) c13[k] = (cp[2][k] & hmask) | (cp[0][k] & ~hmask);
            const b8x_t c3 = __builtin_bit_cast(b8x_t, c13);
#pragma unroll
            for (int tt = 0; tt < TT; tt++) {
                const char *rec = buf + tt * kPackRec + kPackMin;
                // planes: lane half 0 / 1 = parts 1 / 2, then parts 3 / 1
                const b8x_t b12 = *(const b8x_t *)(rec + lane * 16);
                const b8x_t b31 = *(const b8x_t *)(rec + (h ? 0 : 1024) + l31 * 16);
                f16x_t cm = __builtin_amdgcn_mfma_f32_32x32x16_bf16(c2, b12, zero, 0, 0, 0);
                cm = __builtin_amdgcn_mfma_f32_32x32x16_bf16(c3, b31, cm, 0, 0, 0);
                cm = __builtin_amdgcn_mfma_f32_32x32x16_bf16(c1, b12, cm, 0, 0, 0);
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const v4f_t d = *(const v4f_t *)(dl + 8 * g + 4 * h);
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        acc[tt][4 * g + i] += __builtin_fmaf(d[i], C[tt][4 * g + i], cm[4 * g + i]);
                }
            }
        }
    } else {
        const int nb = W.cols >> 5;
        const uint8_t *qp = W.q + row * W.cols + 16 * h;
        const uint16_t *sp = W.s + row * nb;
        // weights in half steps (4 blocks): the next half is in flight while
        // one is consumed
        u4x_t wn[4];
        uint16_t dn[2];
        auto wload = [&](int b0) {
#pragma unroll
            for (int b = 0; b < 4; b++) wn[b] = *(const u4x_t *)(qp + (size_t)min(b0 + b, nb - 1) * 32);
#pragma unroll
            for (int u = 0; u < 2; u++) dn[u] = sp[min(b0 + 2 * u + h, nb - 1)];
        };
        stage(0, s0);
        wload(8 * s0);
        for (int st = s0; st < s1; st++) {
            const int cur = (st - s0) & 1;
            const char *buf = smem + cur * TT * kPackRec;
#pragma unroll
            for (int half = 0; half < 2; half++) {
                u4x_t w[4];
                float d[2];
                if (half == 0) {
                    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's copies have landed
                    __syncthreads();
                    if (st + 1 < s1) stage(cur ^ 1, st + 1);
                }
#pragma unroll
                for (int b = 0; b < 4; b++) w[b] = wn[b];
#pragma unroll
                for (int u = 0; u < 2; u++) d[u] = h2f(dn[u]);
                const int b0 = 8 * st + 4 * half;
                wload(b0 + 4);
                auto block_pair = [&](int u, bool second) {
                    h8x_t a0[2], a1[2];
#pragma unroll
                    for (int e = 0; e < 2; e++) {
                        uint32_t o0[4], o1[4];
                        i8_pairs(w[2 * u + e][0], w[2 * u + e][1], o0);
                        i8_pairs(w[2 * u + e][2], w[2 * u + e][3], o1);
                        a0[e] = as_h8(u4x_t{o0[0], o0[1], o0[2], o0[3]});
                        a1[e] = as_h8(u4x_t{o1[0], o1[1], o1[2], o1[3]});
                    }
#pragma unroll
                    for (int tt = 0; tt < TT; tt++) {
                        const char *rec = buf + tt * kPackRec + 8192 * half;
                        // the products s * d of both blocks as one outer-product
                        // MFMA: lane half h supplies block 2u + h
                        const float s = *(const float *)(buf + tt * kPackRec + kPackScale + (4 * half + 2 * u + h) * 128 +
                                                         l31 * 4);
                        f32x_t sd;
#pragma unroll
                        for (int i = 0; i < 32; i++) sd[i] = 0.0f;
                        sd = __builtin_amdgcn_mfma_f32_32x32x1f32(d[u], s, sd, 0, 0, 0);
#pragma unroll
                        for (int e = 0; e < 2; e++) {
                            if (e == 1 && !second) break;
                            const h8x_t x0 = *(const h8x_t *)(rec + (2 * u + e) * 2048 + lane * 16);
                            const h8x_t x1 = *(const h8x_t *)(rec + (2 * u + e) * 2048 + 1024 + lane * 16);
                            f16x_t dd = __builtin_amdgcn_mfma_f32_32x32x16_f16(a0[e], x0, zero, 0, 0, 0);
                            dd = __builtin_amdgcn_mfma_f32_32x32x16_f16(a1[e], x1, dd, 0, 0, 0);
#pragma unroll
                            for (int i = 0; i < 16; i++) acc[tt][i] = __builtin_fmaf(sd[16 * e + i], dd[i], acc[tt][i]);
                        }
                    }
                };
                if (b0 + 4 <= nb) {
                    block_pair(0, true);
                    block_pair(1, true);
                } else {
#pragma unroll
                    for (int u = 0; u < 2; u++)
                        if (b0 + 2 * u < nb) block_pair(u, b0 + 2 * u + 1 < nb);
                }
            }
        }
    }
    // lane = token, registers = rows 8 g + 4 h + i
#pragma unroll
    for (int tt = 0; tt < TT; tt++) {
        const int t = (tile0 + tt) * kPackTile + l31;
        if (t >= a.M) continue;
        float *o = a.part + ((size_t)ks * a.M + t) * W.rows;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int n = row0 + 8 * g + 4 * h;
            const v4f_t v = {acc[tt][4 * g], acc[tt][4 * g + 1], acc[tt][4 * g + 2], acc[tt][4 * g + 3]};
            if ((W.rows & 3) == 0 && n + 4 <= W.rows) {
                *(v4f_t *)(o + n) = v;
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (n + i < W.rows) o[n + i] = v[i];
            }
        }
    }
}

}  // namespace fl

// Output projection with an f32 input on f16 MFMA (the logits path of
// forward_greedy, flare-core/src/model.rs:1917-1931: matvec_argmax_f32 over
// the dequantized Q6_K output / tied Q8_0 embedding, model.rs:8668-8689).
//
// The RMS-normed input of up to 8 tokens (rmsnorm_into, model.rs:7456-7477)
// sits in LDS as f16 high parts and f16 residuals (x = hi + lo to ~22 bits);
// weight codes are exact in f16 (Q6_K: q - 32 in -32..31; Q8_0: int8), so
// every MFMA product is exact in fp32 and the per-block scale (Q6_K d*sc per
// 16 values, Q8_0 d per 32) multiplies the block's MFMA sum in fp32.
//   Q6_K: v_mfma_f32_16x16x16_f16, one 16-value sub-block of 16 rows.
//   Q8_0: v_mfma_f32_16x16x32_f16, one 32-value block of 16 rows.
// Tile rows: lane l owns weight row l%16 of the tile; MFMA rows are
// (token, hi / lo), so lane group l/16 collects tokens 2(l/16), 2(l/16)+1.
// Epilogue: logits store, or first-max argmax per token (packed u64 max).
#pragma once

#include "mv_kernels.h"

namespace fl {

typedef _Float16 v4h_t __attribute__((ext_vector_type(4)));
typedef _Float16 v8h2_t __attribute__((ext_vector_type(8)));
typedef float v4fm_t __attribute__((ext_vector_type(4)));

constexpr int kMvoThreads = 512;  // 8 waves
constexpr int kMvoMaxTokens = 8;
// LDS rows lie K + 8 halves apart: 16 bytes beyond a multiple of the banks, so
// the 16 rows of an operand read (2 lane groups at a time) take every bank once
// (LONG rows, one token: 0)
constexpr int kMvoPad = 8;

struct MvoArgs {
    WDesc W;
    const float *x;   // [M][K] input rows (before the norm)
    const float *nw;  // norm weight [K] (nullptr: no norm, x used as is)
    float eps;
    int M;
    int epi;          // EPI_STORE or EPI_ARGMAX
    float *out;       // EPI_STORE: [M][rows]
    unsigned long long *slots;  // EPI_ARGMAX: [M] packed (value, index) keys
};

__device__ __forceinline__ v4fm_t mfma_k16(const v4h_t &a, const v4h_t &b, const v4fm_t &c) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ v4fm_t mfma_k32(const v8h2_t &a, const v8h2_t &b, const v4fm_t &c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// 4 six-bit Q6_K codes (bytes of w, 0..63) -> f16 (code - 32), exact:
// binary16 0x6400 | c is 1024 + c; subtracting 1056 leaves c - 32.
__device__ __forceinline__ v4h_t q6_codes_to_h4(uint32_t w) {
    const uint32_t lo = __builtin_amdgcn_perm(0x64646464u, w, 0x07010700u);  // bytes c0, 0x64, c1, 0x64
    const uint32_t hi = __builtin_amdgcn_perm(0x64646464u, w, 0x07030702u);  // bytes c2, 0x64, c3, 0x64
    v4h_t r;
    uint32_t u[2] = {lo, hi};
    __builtin_memcpy(&r, u, 8);
    const v4h_t bias = {(_Float16)1056.0f, (_Float16)1056.0f, (_Float16)1056.0f, (_Float16)1056.0f};
    return r - bias;
}

// 8 int8 codes -> f16, exact
__device__ __forceinline__ v8h2_t i8_codes_to_h8(uint32_t w0, uint32_t w1) {
    v8h2_t r;
#pragma unroll
    for (int i = 0; i < 8; i++) r[i] = (_Float16)(int8_t)(((i < 4 ? w0 : w1) >> (8 * (i & 3))) & 0xFFu);
    return r;
}

// 4 x 4 transpose over the four 16-lane rows: on entry lane row g holds dwords
// 0..3 of segment g; on return register s holds dword g of segment s.
__device__ __forceinline__ void rows_transpose(uint32_t (&d)[4]) {
    auto a = __builtin_amdgcn_permlane32_swap(d[0], d[2], false, false);
    auto b = __builtin_amdgcn_permlane32_swap(d[1], d[3], false, false);
    auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
    auto e = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    d[0] = c[0];
    d[1] = c[1];
    d[2] = e[0];
    d[3] = e[1];
}

// One unit (256 values) of a weight row as lane (row, kg) loads it: 16-byte
// pieces, the four lanes of a row taking neighbouring ones.
template <int FMT>
struct MvoUnit;

// Q6_K super-block.  Llama.cpp layout (quantize.rs:343-384): value
// e = 128 hf + 32 g + l: ql byte 64 hf + 32 (g & 1) + l (low nibble g < 2),
// qh byte 32 hf + l (bits 2g), scale sc[8 hf + l / 16 + 2 g].
template <>
struct MvoUnit<F_Q6K> {
    v4i_t ql[2], qh, sc;  // ql pieces kg and 4 + kg, qh piece kg, the row's 16 int8 scales
    uint16_t d;
    __device__ __forceinline__ void load(const WDesc &W, int row, int u, int kg) {
        const size_t rs = (size_t)row * (W.cols >> 8) + u;
        ql[0] = *(const v4i_t *)(W.q + rs * 128 + 16 * kg);
        ql[1] = *(const v4i_t *)(W.q + rs * 128 + 64 + 16 * kg);
        qh = *(const v4i_t *)(W.h + rs * 64 + 16 * kg);
        sc = *(const v4i_t *)(W.h2 + rs * 16);
        d = W.s[rs];
    }
};

// Q8_0: 8 blocks as 4 pairs of 64 bytes; past the row's end the last pair
// (blocks that do not exist are not used)
template <>
struct MvoUnit<F_Q8_0> {
    v4i_t q[4];
    uint16_t s[8];
    __device__ __forceinline__ void load(const WDesc &W, int row, int u, int kg) {
        const int nb = W.cols >> 5;
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const int blk = min(8 * u + 2 * p + (kg >> 1), nb - 1);
            q[p] = *(const v4i_t *)(W.q + (size_t)row * W.cols + 32 * blk + 16 * (kg & 1));
        }
#pragma unroll
        for (int b = 0; b < 8; b++) s[b] = W.s[(size_t)row * nb + min(8 * u + b, nb - 1)];
    }
};

// A tile of 16 rows costs ~245 vector ops per 256 values (51 us of the 107 us
// that 128256 x 4096 Q6_K, 8 tokens, takes on MI355X; its 431 MB alone take 60;
// 245 us with 4-byte loads, a branch around every activation read and a wave
// per tile).  The waves of a workgroup share a tile and split its K, unit by
// unit, so together they read KiBs of each row in a row: 16 rows in 256-byte
// pieces per wave ran the same loop 17 us slower.  KW waves per tile (mvo_waves),
// kMvoThreads / 64 / KW tiles per workgroup; the next unit's loads are in
// flight while one is consumed (a third unit in flight, or 16 waves, measured
// alike).  LONG: one token whose row leaves the LDS no room for the padding and
// both buffers of partial sums.
template <int FMT, int KW, bool LONG>
__global__ __launch_bounds__(kMvoThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_mvo(MvoArgs a) {
    extern __shared__ __align__(16) char smem[];
    const WDesc &W = a.W;
    const int K = W.cols, M = a.M;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, kg = lane >> 4, r16 = lane & 15;
    constexpr int NW = kMvoThreads / 64, TG = NW / KW;
    // LDS: rows m = 2t + (hi / lo) of the normed input as f16, [2*M][XS]
    const int XS = K + (LONG ? 0 : kMvoPad);
    _Float16 *xa = (_Float16 *)smem;
    // ---- prologue, a wave per token: rmsnorm_into, split into f16 hi / lo ----
    for (int t = wave; t < M; t += NW) {
        const float *x = a.x + (size_t)t * K;
        float inv = 1.0f;
        if (a.nw) {
            float ss = 0.0f;
            for (int i = 4 * lane; i < K; i += 256) {
                const v4f_t v = *(const v4f_t *)(x + i);
                ss += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
            }
            inv = 1.0f / sqrtf(wave_sum(ss) / (float)K + a.eps);
        }
        for (int i = 4 * lane; i < K; i += 256) {
            v4f_t v = *(const v4f_t *)(x + i);
            if (a.nw) v = (v * inv) * *(const v4f_t *)(a.nw + i);
            v4h_t hi, lo;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                // high part rounded toward zero by v_cvt_pkrtz (the compiler
                // cannot re-form it from the product, so hi and the residual
                // come from the same fp32 v)
                const auto h2 = __builtin_amdgcn_cvt_pkrtz(v[j], 0.0f);
                _Float16 h;
                __builtin_memcpy(&h, &h2, 2);
                hi[j] = h;
                lo[j] = (_Float16)(v[j] - (float)h);
            }
            *(v4h_t *)(xa + (size_t)(2 * t) * XS + i) = hi;
            *(v4h_t *)(xa + (size_t)(2 * t + 1) * XS + i) = lo;
        }
    }
    __syncthreads();
    // A operand row of this lane: m = r16 (token m/2, hi/lo m%2); past 2M the
    // last row again, into result rows that nothing reads
    const _Float16 *xrow = xa + (size_t)min(r16, 2 * M - 1) * XS;
    const v4fm_t zero = {0.f, 0.f, 0.f, 0.f};

    const int ntile = (W.rows + 15) / 16, nu = (K + 255) >> 8, upw = (nu + KW - 1) / KW;
    const int kw = wave % KW, tg = wave / KW;
    // partial sums of a tile, [2 buffers][wave][2][64]: a buffer is written
    // again two tiles later, past the barrier between.  LONG: [wave][16], written
    // again after a barrier of its own.
    __shared__ float part[LONG ? 1 : 2][NW][LONG ? 1 : 2][LONG ? 16 : 64];
    const int first = blockIdx.x * TG, step = gridDim.x * TG;
    const int niter = (ntile - first + step - 1) / step;  // the same for every wave (first < ntile)
    unsigned long long best[2] = {0ull, 0ull};  // KW 1: tokens 2kg, 2kg+1; else one
    float acc[2] = {0.0f, 0.0f};  // tokens 2kg, 2kg+1
    MvoUnit<FMT> ta, tb;
    auto load = [&](MvoUnit<FMT> &T, int f) {
        const int tile = min(first + (f / upw) * step + tg, ntile - 1);
        T.load(W, min(tile * 16 + r16, W.rows - 1), min(kw + (f % upw) * KW, nu - 1), kg);
    };
    auto consume = [&](MvoUnit<FMT> &T, int f) {
        const int it = f / upw, j = f % upw, u = kw + j * KW;
        const _Float16 *xu = xrow + u * 256;
        if (u < nu) {
            if constexpr (FMT == F_Q6K) {
                uint32_t ql[2][4], qh[4];
                float C[2] = {0.0f, 0.0f};
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    ql[0][i] = (uint32_t)T.ql[0][i];
                    ql[1][i] = (uint32_t)T.ql[1][i];
                    qh[i] = (uint32_t)T.qh[i];
                }
                rows_transpose(ql[0]);  // [hf][2 (g & 1) + l / 16]
                rows_transpose(ql[1]);
                rows_transpose(qh);     // [2 hf + l / 16]
#pragma unroll
                for (int hf = 0; hf < 2; hf++)
#pragma unroll
                    for (int g = 0; g < 4; g++)
#pragma unroll
                        for (int h16 = 0; h16 < 2; h16++) {
                            const v4h_t av = *(const v4h_t *)(xu + hf * 128 + g * 32 + h16 * 16 + 4 * kg);
                            const uint32_t lw = ql[hf][2 * (g & 1) + h16], hw = qh[2 * hf + h16];
                            const uint32_t codes = ((lw >> (4 * (g >> 1))) & 0x0F0F0F0Fu) |
                                                   ((g < 2 ? hw << (4 - 2 * g) : hw >> (2 * g - 4)) & 0x30303030u);
                            const v4fm_t dd = mfma_k16(av, q6_codes_to_h4(codes), zero);
                            const int si = hf * 8 + h16 + 2 * g;
                            const float s = (float)(int8_t)(((uint32_t)T.sc[si >> 2] >> (8 * (si & 3))) & 0xFFu);
                            C[0] = __builtin_fmaf(s, dd[0] + dd[1], C[0]);
                            C[1] = __builtin_fmaf(s, dd[2] + dd[3], C[1]);
                        }
                const float d = h2f(T.d);
                acc[0] = __builtin_fmaf(d, C[0], acc[0]);
                acc[1] = __builtin_fmaf(d, C[1], acc[1]);
            } else {
                const int nb = (K >> 5) - 8 * u;  // blocks from this unit on
                // after the swaps below lane group kg holds bytes 8 x
                // {0, 2, 1, 3}[kg] of a block
                const int off = 8 * (((kg & 1) << 1) | (kg >> 1));
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    if (2 * p >= nb) break;
                    auto x = __builtin_amdgcn_permlane32_swap((uint32_t)T.q[p][0], (uint32_t)T.q[p][2], false, false);
                    auto y = __builtin_amdgcn_permlane32_swap((uint32_t)T.q[p][1], (uint32_t)T.q[p][3], false, false);
#pragma unroll
                    for (int e = 0; e < 2; e++) {  // block 2p + e: dwords x[e], y[e]
                        if (2 * p + e >= nb) break;
                        const v8h2_t av = *(const v8h2_t *)(xu + 64 * p + 32 * e + off);
                        const v4fm_t dd = mfma_k32(av, i8_codes_to_h8(x[e], y[e]), zero);
                        const float s = h2f(T.s[2 * p + e]);
                        acc[0] = __builtin_fmaf(s, dd[0] + dd[1], acc[0]);
                        acc[1] = __builtin_fmaf(s, dd[2] + dd[3], acc[1]);
                    }
                }
            }
        }
        if (j < upw - 1) return;
        if constexpr (KW == 1) {  // a wave's own tile
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const int tile = first + it * step + tg, n = tile * 16 + r16, t = 2 * kg + e;
                if (tile < ntile && t < M && n < W.rows) {
                    if (a.epi == EPI_STORE) a.out[(size_t)t * W.rows + n] = acc[e];
                    else best[e] = umax64(best[e], argmax_key(acc[e], (uint32_t)n));
                }
                acc[e] = 0.0f;
            }
            return;
        }
        // the tile's KW partial sums: (row, token) per thread, summed in order.
        // Only LDS is waited for: the next unit's loads stay in flight.
        if constexpr (LONG) {
            __syncthreads();
            if (lane < 16) part[0][wave][0][lane] = acc[0];
        } else {
            part[it & 1][wave][0][lane] = acc[0];
            part[it & 1][wave][1][lane] = acc[1];
        }
        acc[0] = acc[1] = 0.0f;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const int g = threadIdx.x >> 7, e = (threadIdx.x >> 6) & 1;  // tile of the group, token parity
        if (LONG ? threadIdx.x < 16 : g < TG) {
            const int buf = LONG ? 0 : it & 1;
            float v = part[buf][g * KW][e][lane];
#pragma unroll
            for (int k = 1; k < KW; k++) v += part[buf][g * KW + k][e][lane];
            const int tile = first + it * step + g, n = tile * 16 + r16, t = 2 * kg + e;
            if (tile < ntile && t < M && n < W.rows) {
                if (a.epi == EPI_STORE) a.out[(size_t)t * W.rows + n] = v;
                else best[0] = umax64(best[0], argmax_key(v, (uint32_t)n));
            }
        }
    };
    load(ta, 0);
    pingpong(niter * upw, ta, tb, load, consume);
    if (a.epi == EPI_ARGMAX) {
        // per token: max over the 16 rows (lanes of one kg group), then the
        // workgroup's tiles, then one device atomic per token
        __shared__ unsigned long long lb[TG][kMvoMaxTokens];
#pragma unroll
        for (int e = 0; e < (KW == 1 ? 2 : 1); e++) {
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) best[e] = umax64(best[e], __shfl_xor(best[e], o, 64));
            const int g = KW == 1 ? wave : threadIdx.x >> 7, t = 2 * kg + (KW == 1 ? e : (threadIdx.x >> 6) & 1);
            if (g < TG && r16 == 0) lb[g][t] = best[e];
        }
        __syncthreads();
        if (threadIdx.x < M) {
            unsigned long long b = lb[0][threadIdx.x];
            for (int i = 1; i < TG; i++) b = umax64(b, lb[i][threadIdx.x]);
            atomicMax(a.slots + threadIdx.x, b);
        }
    }
}

}  // namespace fl

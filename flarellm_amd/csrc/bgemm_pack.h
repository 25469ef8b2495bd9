// Device helpers of the packed activations (layout in bgemm_args.h).
#pragma once

#include "bgemm_args.h"

namespace fl {

typedef _Float16 h8x_t __attribute__((ext_vector_type(8)));
typedef _Float16 h4x_t __attribute__((ext_vector_type(4)));
typedef _Float16 h2x_t __attribute__((ext_vector_type(2)));
typedef __bf16 b8x_t __attribute__((ext_vector_type(8)));
typedef float f16x_t __attribute__((ext_vector_type(16)));
typedef float f32x_t __attribute__((ext_vector_type(32)));
typedef uint32_t u4x_t __attribute__((ext_vector_type(4)));

// 16 bytes per lane from memory to LDS at lds + 16 * lane (lds wave-uniform)
__device__ __forceinline__ void copy_to_lds(const char *g, char *lds) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)g,
                                     (__attribute__((address_space(3))) void *)lds, 16, 0, 0);
}

// 4 consecutive codes k .. k + 3 (k % 4 == 0, within the step) of token t into
// a record: 8 bytes in the layout's value order.
__device__ __forceinline__ void pack_codes4(char *rec, int t, int k, int q0, int q1, int q2, int q3) {
    char *o = rec + (k >> 5) * 2048 + ((k >> 3) & 1) * 1024 + ((t & 31) + 32 * ((k >> 4) & 1)) * 16 + 2 * (k & 4);
    *(h4x_t *)o = h4x_t{(_Float16)(float)q0, (_Float16)(float)q2, (_Float16)(float)q1, (_Float16)(float)q3};
}

// A block's scale and s * sum q in a record (blk within the step).
__device__ __forceinline__ void pack_scale(char *rec, int t, int blk, float s, int sum) {
    *(float *)(rec + kPackScale + blk * 128 + (t & 31) * 4) = s;
    // three bfloat16 parts, each the truncated rest of the one before: 24 bits
    float v = s * (float)sum;
    uint16_t *m = (uint16_t *)(rec + kPackMin) + (t & 31) * 8 + blk;
#pragma unroll
    for (int p = 0; p < 3; p++) {
        const uint32_t b = __float_as_uint(v) & 0xFFFF0000u;
        m[p * 256] = (uint16_t)(b >> 16);
        v -= __uint_as_float(b);
    }
}

// Workgroup -> (token, chunk): the 32 tokens of a tile share a record, so they
// run on one XCD (blockIdx % 8) in a row and its L2 merges their 8-byte pieces.
__device__ __forceinline__ void pack_wg(int nchunk, int &t, int &chunk) {
    const int i = blockIdx.x >> 3;
    chunk = (i >> 5) % nchunk;
    t = (((i >> 5) / nchunk) * 8 + (blockIdx.x & 7)) * kPackTile + (i & 31);
}

// workgroups of kernels that map them with pack_wg: tiles in groups of 8
inline unsigned pack_grid(int M, int nchunk) {
    return (unsigned)((M + 8 * kPackTile - 1) / (8 * kPackTile) * 8 * kPackTile * nchunk);
}

// The Q8_0 block of 32 values held 4 a thread by 8 neighbouring threads, into a
// record (quantize_input_q8_0_into arithmetic); k = the first value's index
// within the step.
__device__ __forceinline__ void pack_block8(const float (&y)[4], bool in, char *rec, int t, int k) {
    float amax = fmaxf(fmaxf(fabsf(y[0]), fabsf(y[1])), fmaxf(fabsf(y[2]), fabsf(y[3])));
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
    const float d = amax / 127.0f;
    const float id = (d != 0.0f) ? 127.0f / amax : 0.0f;
    int q[4], sum = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        q[j] = q8_code(y[j] * id);
        sum += q[j];
    }
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) sum += __shfl_xor(sum, o, 64);
    if (!in) return;
    pack_codes4(rec, t, k, q[0], q[1], q[2], q[3]);
    if ((k & 31) == 0) pack_scale(rec, t, k >> 5, d, sum);
}

}  // namespace fl

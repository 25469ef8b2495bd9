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

}  // namespace fl

// Arguments of the many-query attention (kernels in attw_kernels.h, included
// by attw.hip only).
#pragma once

#include "kernels.h"

namespace fl {

// Keys and values of one layer as matrix-core operands, per plane
//   K [kv head][slot][D], V [kv head][slot / 32][D][32]
// One binary16 plane (the fp16 model cache itself) or three bfloat16 planes
// (f32 values split exactly into 3 x 8 bits; AttwPlanes in a workspace).
struct AttwArgs {
    const float *q;         // [M][qstride] f32, RoPE applied; head h at h * D
    const uint16_t *k, *v;  // plane 0
    size_t plane;           // elements between planes (k and v alike)
    size_t head_stride;     // elements between kv heads
    int slots;              // readable slots per kv head (a multiple of 32)
    int M, pos0;            // queries; query t attends slots 0 .. pos0 + t
    int nkv, group;         // kv heads, query heads per kv head
    int qstride;
    float *out;             // [M][qstride] f32, or
    char *xp;               // Q8_0 rows in packed records (bgemm_args.h) of
    int nst;                // nst steps
    int ksplit, chunk;      // workgroups over the keys of an item, 64-key tiles of each (ksplit 0 or 1: whole)
    float *part, *ml;       // split: [ksplit][M][qstride] f32, [ksplit][M][heads][2] (attw_split_floats)
    int *flag;              // host memory: set if some output is not finite; nullptr: the careful form
};

// f32 rows or cache slots -> three bfloat16 planes
struct AttwSplitArgs {
    const void *k, *v;          // f32 values, or Q8 codes (V in 32-slot transposed blocks) with ks / vs
    const uint16_t *ks, *vs;    // Q8: binary16 scales [kv head][S][D / 32]
    long long tok_stride, head_stride;  // elements between slots / kv heads
    int S;                      // slots per kv head of the source
    int T, nkv;                 // slots to split, kv heads
    uint16_t *ko, *vo;          // planes out
    size_t plane, out_stride;   // elements between planes / kv heads
    bool careful;               // for the careful form of the attention
};

}  // namespace fl

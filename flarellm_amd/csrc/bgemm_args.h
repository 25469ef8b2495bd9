// Arguments of the large-batch quantized GEMM (kernels in bgemm_kernels.h,
// included by bgemm.hip only) and the layout of its packed activations.
#pragma once

#include "kernels.h"

namespace fl {

// Packed Q8_0 activations: one record per (tile of 32 tokens, step of 256
// values), tiles outermost, in the order the GEMM's lanes read them, so a
// record goes from memory to LDS unchanged and every operand read is one
// conflict-free 16-byte read per lane.
//   [0, 16384)      codes as binary16 (exact), [block 8][m 2][lane 64][8]:
//                   lane = token + 32 h holds values 16 h + 8 m + order[0..8)
//                   of the block, order = 0 2 1 3 4 6 5 7 (the order the
//                   weight codes unpack in)
//   [16384, 17408)  block scales f32, [block 8][token 32]
//   [17408, 18944)  s * sum q as three bfloat16 parts (24 bits),
//                   [part 3][token 32][block 8] (the Q4_K min term); to 19456 unused
constexpr int kPackRec = 19456, kPackScale = 16384, kPackMin = 17408;
constexpr int kPackTile = 32;  // tokens per record

inline size_t pack_bytes(int tokens, int cols) {
    return (size_t)((tokens + kPackTile - 1) / kPackTile) * ((cols + 255) / 256) * kPackRec;
}

struct BgArgs {
    WDesc W;
    const char *xp;  // packed activations [tile][step] records
    int M;           // tokens
    int nst;         // 256-value steps per row (the last may be partial: Q8_0)
    int ksplit;      // K splits (steps [k * chunk, (k + 1) * chunk))
    int chunk;
    float *part;     // [ksplit][M][rows] partial sums (ksplit 1: the result)
    int nrt, ntt;    // workgroup tiles over rows and tokens
};

}  // namespace fl

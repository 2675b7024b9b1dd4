// Matrix-core helpers of the whole-layer kernels (gfx950).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "sru_scan.h"

namespace sru_amd {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x2 __attribute__((aligned(4))) u32x2_a4;
typedef u32x4 __attribute__((aligned(4))) u32x4_a4;

constexpr int kStepK = 32;      // inner indices per matrix instruction

// c += a b for 16 x 32 times 32 x 16: lane (q, m) = (lane / 16, lane % 16) holds row m of a and column
// m of b, inner indices 8q .. 8q + 7, and rows 4q .. 4q + 3 of column m of c.
template <typename T> __device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c);
template <> __device__ __forceinline__ f32x4 mfma<bf16_bits>(u32x4 a, u32x4 b, f32x4 c) {
    typedef __bf16 v8 __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
}
template <> __device__ __forceinline__ f32x4 mfma<half_bits>(u32x4 a, u32x4 b, f32x4 c) {
    typedef _Float16 v8 __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
}

// The weights of one cell (its K streams) for inner indices k0 .. k0 + 7 as K matrix operands, operand
// s holding stream s. `column` is the cell's first column, `cols` the row pitch (both in elements, cols
// even, the weight 4-byte aligned). Three streams start at an odd element every other cell: those
// load from one element earlier, so that every load is 8 bytes from a 4-byte boundary and the last
// one ends with its row.
template <int K>
__device__ __forceinline__ void load_cell_weights(const uint16_t *weight, int64_t cols, int64_t column, int64_t k0, u32x4 (&out)[K]) {
    const int odd = K == 3 ? (int)(column & 1) : 0;
    const uint16_t *p = weight + k0 * cols + (column - odd);
    u32x2 w[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) w[r] = *reinterpret_cast<const u32x2_a4 *>(p + r * cols);
    if constexpr (K == 3) {
        const uint32_t sh = odd * 16;
#pragma unroll
        for (int r = 0; r < 8; ++r) w[r] = u32x2{__builtin_amdgcn_alignbit(w[r][1], w[r][0], sh), w[r][1] >> sh};
    }
#pragma unroll
    for (int s = 0; s < K; ++s)
#pragma unroll
        for (int h = 0; h < 4; ++h)   // the low or high halves of two dwords
            out[s][h] = __builtin_amdgcn_perm(w[2 * h + 1][s / 2], w[2 * h][s / 2], (s & 1) ? 0x07060302u : 0x05040100u);
}

}  // namespace sru_amd

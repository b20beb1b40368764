// Small device helpers of the matrix-core and staging kernels.
#pragma once

#include <hip/hip_runtime.h>

namespace feq {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

// D = A B + C, 16 x 16 x 4 in float32: lane (c = l % 16, g = l / 16) holds A[c][g], B[g][c]
// and, in register r, C and D[4 g + r][c].
__device__ __forceinline__ v4f mfma4(float a, float b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// q / d for 0 <= q < 2^22, inv = 1 / d: q + 1/2 is exact and the two roundings of the
// product stay under the 1 / (2 d) that separates it from the next integer.
__device__ __forceinline__ int quotient(int q, float inv) {
    return static_cast<int>((static_cast<float>(q) + 0.5f) * inv);
}

}  // namespace
}  // namespace feq

// The factor of an RMS norm that a product's rows still lack.
#pragma once
#include "common.h"

// Parts of a row's sum of squares: one for each block of the product that made the row (gemm_residual.hip).
constexpr int SQUARE_PARTS = 256;

struct RowNorm {
  const float* squares;  // [rows, SQUARE_PARTS]
  float inv_width, eps;
  // 1 / sqrt(mean of squares + eps) of the row whose parts 4 lane .. 4 lane + 3 a wave's lane holds
  __device__ __forceinline__ float factor(f32x4_t parts) const {
    return rsqrtf(wave_sum((parts[0] + parts[1]) + (parts[2] + parts[3])) * inv_width + eps);
  }
};

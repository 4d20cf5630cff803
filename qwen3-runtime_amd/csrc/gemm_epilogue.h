// What the bfloat16 products do with their float32 sums.
#pragma once
#include "common.h"

// What the gated products do with a gate and an up value (their template's GATED: 0 no gate, 1 SwiGLU and
// nothing else, 2 what is given here): an activation of common.h, times a factor per row of the
// activations (null: 1).
#define QRT_ACT_RELU2 2  // of a product without a gate: the square of relu
struct GatedEpilogue {
  int kind;
  float limit;
  const float* row_scale;
  template <int GATED>
  __device__ __forceinline__ float apply(float g, float u, int m) const {
    if (GATED == 1) return gated_act(g, u, QRT_ACT_SWIGLU, 0.f);
    const float v = gated_act(g, u, kind, limit);
    return row_scale ? v * row_scale[m] : v;
  }
  // a sum without a gate; the activation is of the sum rounded to bfloat16, as a kernel behind the product sees it
  __device__ __forceinline__ float whole(float x) const {
    if (kind != QRT_ACT_RELU2) return x;
    const float v = fmaxf((float)(bf16_t)x, 0.f);
    return v * v;
  }
};

__device__ __forceinline__ void store4(float* p, const float (&o)[4]) {
  *(f32x4_t*)p = (f32x4_t){o[0], o[1], o[2], o[3]};
}
__device__ __forceinline__ void store4(bf16_t* p, const float (&o)[4]) {
  typedef bf16_t bf16x4_t __attribute__((ext_vector_type(4)));
  *(bf16x4_t*)p = (bf16x4_t){(bf16_t)o[0], (bf16_t)o[1], (bf16_t)o[2], (bf16_t)o[3]};
}

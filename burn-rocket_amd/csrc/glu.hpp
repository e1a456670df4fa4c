// MLP glue of a gate|up product (host.rs:12-39), shared by the GEMM epilogues.
#pragma once

#include "common.hpp"

// silu(g)·u or gelu_tanh(g)·u in f32, in the reference's operation order with
// no FMA contraction.
enum { GLU_NONE = 0, GLU_SILU = 1, GLU_GELU = 2 };
template <int GLU>
__device__ __forceinline__ float glu_apply(float g, float u) {
#pragma clang fp contract(off)
  if constexpr (GLU == GLU_SILU) {
    const float sigmoid = 1.0f / (1.0f + expf(-g));
    return g * sigmoid * u;
  } else {
    constexpr float k = (float)(1.12837916709551257390 * 0.70710678118654752440);  // sqrt(2/pi)
    const float inner = (g + g * g * g * 0.044715f) * k;
    return ((g * (tanhf(inner) + 1.0f)) * 0.5f) * u;
  }
}

// Device helpers of the attention kernels: masks as key intervals, cross-lane
// reductions over the lanes that hold one query, and the fp16 split of P.
#pragma once

#include "common.hpp"
#include "kernels.hpp"

namespace {
constexpr float LOG2E = 1.4426950408889634f;
constexpr float MASKED_SCORE = -30000.0f;  // fa_score clamp (attn/softmax.rs:59)

// Visible absolute key interval [lo, hi] of query t (hi may exceed the keys).
__device__ __forceinline__ void vis_range(int mode, int64_t w, int64_t t, int64_t &lo,
                                          int64_t &hi) {
  const int64_t INF = (int64_t)1 << 60;
  switch (mode) {
    case RK_MASK_CAUSAL:
      lo = -INF;
      hi = t;
      break;
    case RK_MASK_WINDOW:
      lo = t - w;
      hi = t + w;
      break;
    case RK_MASK_CAUSAL_WINDOW:
      lo = t - w + 1;
      hi = t;
      break;
    default:
      lo = -INF;
      hi = INF;
  }
}

// x - f32(h) for the low / high fp16 half of h in one v_fma_mix_f32 (the f16
// operand is widened exactly and the difference of a value and its
// truncation to fp16 is exact in f32), instead of a convert and a subtract.
__device__ __forceinline__ float minus_half_lo(unsigned h, float x) {
  float r;
  asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(x));
  return r;
}
__device__ __forceinline__ float minus_half_hi(unsigned h, float x) {
  float r;
  asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(x));
  return r;
}

// max over lanes l, l^16, l^32, l^48 (the four lane groups holding one query).
__device__ __forceinline__ float max4groups(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float sum4groups(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Key tiles (of TK keys) that queries q_lo..q_hi read: their rows
// see absolute keys in per-row intervals whose ends never decrease with the
// query position, so the union of the rows' intervals and "some row sees no
// key at all" (degenerate: then every key tile is swept) follow from the first
// and the last query. full_lo..full_hi: relative keys every row of the tile
// sees.
struct TileKeys {
  int kt_begin, kt_end, full_lo, full_hi;
  bool degenerate;
};
template <int TK>
__device__ __forceinline__ TileKeys tile_keys(const AttnArgs &a, int q_lo, int q_hi) {
  const int n_kt = (a.n_kv + TK - 1) / TK;
  const int64_t t_min = a.q0 + q_lo, t_max = a.q0 + q_hi;
  const int64_t kabs0 = a.k0, kabs1 = a.k0 + a.n_kv - 1;
  int64_t lo_a, hi_a, lo_b, hi_b;
  vis_range(a.mask_mode, a.window, t_min, lo_a, hi_a);
  vis_range(a.mask_mode, a.window, t_max, lo_b, hi_b);
  TileKeys t;
  // a row t sees no key iff lo(t) > kabs1, hi(t) < kabs0 or lo(t) > hi(t);
  // lo - hi is the same for every row
  t.degenerate = hi_a < kabs0 || lo_b > kabs1 || lo_a > hi_a;
  t.full_lo = (int)min(max(lo_b - a.k0, (int64_t)0), (int64_t)a.n_kv);
  t.full_hi = (int)max(min(hi_a - a.k0, (int64_t)a.n_kv - 1), (int64_t)-1);
  t.kt_begin = 0;
  t.kt_end = n_kt;
  if (!t.degenerate) {
    const int64_t any_lo = max(lo_a, kabs0) - a.k0;  // relative key indices
    const int64_t any_hi = min(hi_b, kabs1) - a.k0;
    t.kt_begin = (int)(max(any_lo, (int64_t)0) / TK);
    t.kt_end = (int)min((any_hi / TK) + 1, (int64_t)n_kt);
  }
  return t;
}
}  // namespace

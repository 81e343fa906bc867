// Activations: what a feed-forward makes of its gate and up columns, or (kinds from kGluKinds on) of its up columns alone.  The kind is
// the same for a whole launch.
#pragma once

#include "common.hpp"

namespace sgl_amd {

enum : int { kGluNone = 0, kGluSilu = 1, kGluGeluTanh = 2, kGluClampedSwish = 3, kGluKinds = 4, kActSquaredRelu = 4, kActKinds = 5 };

struct GluParams {
  int kind;
  float limit, alpha;          // of kGluClampedSwish
};

// gelu_tanh(g) * u: 0.5 (1 + tanh y) = 1 / (1 + exp(-2 y))
__device__ __forceinline__ float gelu_tanh_glu(float g, float u) {
  const float y = 0.7978845608028654f * (g + 0.044715f * g * g * g);
  return g / (1.0f + expf(-2.0f * y)) * u;
}
// g = min(g, limit), u in [-limit, limit]:  g sigmoid(alpha g) (u + 1)
__device__ __forceinline__ float clamped_swish_glu(const GluParams& p, float g, float u) {
  g = fminf(g, p.limit);
  u = fminf(fmaxf(u, -p.limit), p.limit);
  return g / (1.0f + expf(-p.alpha * g)) * (u + 1.0f);
}

__device__ __host__ __forceinline__ bool act_gated(int kind) { return kind > kGluNone && kind < kGluKinds; }
__device__ __host__ __forceinline__ bool act_pointwise(int kind) { return kind >= kGluKinds; }

// the one activation without a gate: relu(v)^2
__device__ __forceinline__ float squared_relu(float v) {
  v = fmaxf(v, 0.f);
  return v * v;
}

// silu(g) of a g that is a bf16 value.  Up to |g| = 80 nothing over- or underflows, and a gate costs 12 instructions in the place of the 60 of
// expf and a division for all cases: log2 e in two parts (Cody and Waite), the first of 16 bits, so that its product with the 8 bits of g is exact
// and v_exp_f32 takes it as it is; the reciprocal's quotient once corrected.  Rounded to bf16 it has silu_any()'s bits for all 65 536 g, -0 among them
// (compared on the device; of a g that is no number the sign may differ).
// us: 3000 tokens over 8 experts (64 outputs a lane at the end of a tile) 2243 -> 2194, a decode step of four layers 720 -> 716; 48 tokens the same.
__device__ __forceinline__ float silu_near(float g) {                      // |g| <= 80, or no number
  const float e = fast_exp2(g * -0x1.7154p+0f);
  const float d = 1.0f + __builtin_fmaf(e, g * -0x1.480fb6p-18f, e);
  const float r = __builtin_amdgcn_rcpf(d);
  const float q = g * r;
  return __builtin_fmaf(-__builtin_fmaf(d, q, -g), r, q);                  // (this way round a gate of -0 keeps its sign)
}
__device__ __forceinline__ float silu_any(float g) { return g / (1.0f + expf(-g)); }

// kRound: silu keeps the rounding points of 16-bit activations (projection -> bf16, silu -> bf16); the other kinds stay in fp32
template <bool kRound>
__device__ __forceinline__ float glu(const GluParams& p, float g, float u) {
  if (p.kind == kGluGeluTanh) return gelu_tanh_glu(g, u);
  if (p.kind == kGluClampedSwish) return clamped_swish_glu(p, g, u);
  if (!kRound) return silu_any(g) * u;
  const float gb = rbf(g);
  return rbf(fabsf(gb) > 80.f ? silu_any(gb) : silu_near(gb)) * rbf(u);
}
// four outputs of glu<true>, the kind and the range looked at once
__device__ __forceinline__ void glu4(const GluParams& p, const float (&g)[4], const float (&u)[4], float (&o)[4]) {
  if (p.kind != kGluSilu) {
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = glu<true>(p, g[r], u[r]);
    return;
  }
  float gb[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) gb[r] = rbf(g[r]);
  if (fmaxf(fmaxf(fabsf(gb[0]), fabsf(gb[1])), fmaxf(fabsf(gb[2]), fabsf(gb[3]))) > 80.f) {
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = silu_any(gb[r]);
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = silu_near(gb[r]);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) o[r] = rbf(o[r]) * rbf(u[r]);
}

}  // namespace sgl_amd

// The experts' activations (moe.hip, moe_pingpong.hip).
#pragma once
#include "common.h"

namespace dlia {

// An expert's activation from its gate and up pre-activations.
__device__ __forceinline__ float expert_act_limited(float g, float u, float limit) {
  const float gv = fminf(g, limit), uv = fminf(fmaxf(u, -limit), limit);
  return gv / (1.f + expf(-1.702f * gv)) * (uv + 1.f);
}
__device__ __forceinline__ float expert_act_free(float g, float u) { return g / (1.f + expf(-g)) * u; }

__device__ __forceinline__ float expert_act(float g, float u, float limit) {
  if (limit > 0.f) return expert_act_limited(g, u, limit);
  return expert_act_free(g, u);
}

__device__ __forceinline__ float relu2(float u) { const float r = fmaxf(u, 0.f); return r * r; }

}  // namespace dlia

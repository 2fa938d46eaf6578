// Activations in the epilogues of the bf16 products (kinds as in stream32.hip's act_kernel: gated 0 gelu_tanh(g) u, 1 g'
// sigmoid(alpha g') (u' + 1) with g' = min(g, limit) and u' = clamp(u, +-limit) where limit > 0, 5 relu(g) u; elementwise 7
// relu(x)^2), on the hardware's exponential and reciprocal: a sigmoid of x is off by about (|x| + 4) 2^-24 relative (the
// exponent x log2 e is rounded to fp32), the result is then rounded to bf16.
#pragma once

#include "common.h"

namespace k8sllm {

struct EpiAct {
  int kind = -1;         // -1: none
  float limit = 0.f, alpha = 1.f;
};
__device__ __forceinline__ float epi_sigmoid(float x) { return __builtin_amdgcn_rcpf(1.f + __expf(-x)); }
template <int KIND>
__device__ __forceinline__ float epi_pair(float g, float u, float limit, float alpha) {
  if constexpr (KIND == 0) return g * epi_sigmoid(1.5957691216057308f * (g + 0.044715f * g * g * g)) * u;
  if constexpr (KIND == 5) return fmaxf(g, 0.f) * u;
  if (limit > 0.f) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
  }
  return g * epi_sigmoid(alpha * g) * (u + 1.f);
}
// The kind of a launch, for epilogues of a few elements per lane.
__device__ __forceinline__ float epi_gated(float g, float u, const EpiAct& a) {
  if (a.kind == 0) return epi_pair<0>(g, u, a.limit, a.alpha);
  if (a.kind == 5) return epi_pair<5>(g, u, a.limit, a.alpha);
  return epi_pair<1>(g, u, a.limit, a.alpha);
}
__device__ __forceinline__ float epi_elem(float v, const EpiAct&) { return v > 0.f ? v * v : 0.f; }

}  // namespace k8sllm

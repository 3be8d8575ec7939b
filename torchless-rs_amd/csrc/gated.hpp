// The gate of a gated feed-forward: act(gate) * up.
#pragma once
#include "common.hpp"

namespace tl {

// ---- the function of a gated feed-forward's gate ---------------------------------
// 0: silu(g) = g / (1 + exp(-g)); 1: the tanh form of gelu,
// 0.5 g (1 + tanh(sqrt(2/pi) (g + 0.044715 g^3)))
constexpr int ACT_SILU = 0;
constexpr int ACT_GELU_TANH = 1;
constexpr int ACT_SWISH_CLAMPED = 2;   // g' = min(g, limit), u' = clamp(u, -limit, limit): g' logistic(alpha g') (u' + shift)
constexpr int ACT_RELU = 3;            // max(g, 0)
__device__ __forceinline__ float gate_act(float g, int act) {
  if (act == ACT_RELU) return fmaxf(g, 0.f);
  if (act == ACT_GELU_TANH) return 0.5f * g * (1.0f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g)));
  return g / (1.0f + expf(-g));
}
// act(gate) * up with the constants of the functions that have some
struct ActConstants {
  float alpha, limit, shift;
};
__device__ __forceinline__ float gate_times_up(float g, float u, int act, ActConstants k) {
  if (act == ACT_SWISH_CLAMPED) {
    g = fminf(g, k.limit);
    u = fminf(fmaxf(u, -k.limit), k.limit);
    return (g / (1.0f + expf(-k.alpha * g))) * (u + k.shift);
  }
  return gate_act(g, act) * u;
}

}  // namespace tl

// The activations of routed experts, for the kernels that apply them to sums they have in registers and for those
// that read the sums from memory.
#pragma once
#include "common.hpp"

namespace tl {

// act = the square of max(., 0) (code 0), max(., 0) (code 1), or xIELU (code 2) with two numbers a and b:
// a z^2 + z/2 where z > 0, b (exp(z) - 1 - z) + z/2 elsewhere
struct UnaryAct {
  int code;
  float a, b;
};
__device__ __forceinline__ float unary_act(float z, const UnaryAct& k) {
  if (k.code == 2) return z > 0.f ? fmaf(k.a * z, z, 0.5f * z) : fmaf(k.b, expm1f(z) - z, 0.5f * z);
  const float r = fmaxf(z, 0.f);
  return k.code == 0 ? r * r : r;
}

// An expert with a gate: down(act(g, u)) with g = W_gate t, u = W_up t and
//     act(g, u) = g' logistic(alpha g') (u' + shift) ,  g' = min(g, limit) ,  u' = clamp(u, -limit, limit).
// The stacked matrix holds, expert after expert, the rows [gate (ff) | up (ff)], and behind the last expert
// the shared one's [gate (shared) | up (shared)], which has a limit of its own.  The router's weight s
// multiplies the expert's INPUT t = s y (`on_input`: g and u are linear in t, so s multiplies both before
// the clamps) or its output (the activation times s).  An expert with weight 0 adds nothing either way.
struct GateTerms {
  float limit, limit_shared, alpha, shift;
  int on_input;
};

__device__ __forceinline__ float gated_value(float g, float u, float s, float limit, const GateTerms& k) {
  if (k.on_input) {
    g *= s;
    u *= s;
  }
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  const float a = g / (1.0f + expf(-k.alpha * g)) * (u + k.shift);
  return k.on_input ? a : a * s;
}

}  // namespace tl

// What the bfloat16 products do with their sums.
#pragma once
#include "common.hpp"

namespace tl {

// what happens to the product
constexpr int EPI_STORE = 0;        // C = product (float)
constexpr int EPI_ACCUMULATE = 1;   // C += product (float; the residual stream)
constexpr int EPI_SILU_PAIR = 2;    // W's rows come in groups of 64 (32 gate rows, their 32 up rows):
                                    // C is bfloat16 [M, N/2] = silu(gate) * up
constexpr int EPI_GELU_PAIR = 3;    // the same pairs with the tanh form of gelu on the gate:
                                    // 0.5 g (1 + tanh(sqrt(2/pi) (g + 0.044715 g^3)))
constexpr int EPI_SWISH_CLAMPED_PAIR = 4;   // the same pairs with g' = min(g, limit), u' = clamp(u, -limit, limit):
                                            // g' / (1 + exp(-alpha g')) * (u' + shift)
constexpr int EPI_RELU_PAIR = 5;    // the same pairs with max(g, 0) on the gate
__host__ __device__ __forceinline__ bool is_pair(int epilogue) {
  return epilogue == EPI_SILU_PAIR || epilogue == EPI_GELU_PAIR || epilogue == EPI_SWISH_CLAMPED_PAIR ||
         epilogue == EPI_RELU_PAIR;
}
// What happens to the product as the kernels take it: the code, and the constants of a paired epilogue
// whose function has some.  It reads as its code wherever a plain number is asked for.
struct Epi {
  int code;
  float alpha, limit, shift;
  __host__ __device__ Epi(int c = EPI_STORE, float a = 1.f, float l = 0.f, float s = 0.f) : code(c), alpha(a), limit(l), shift(s) {}
  __host__ __device__ __forceinline__ operator int() const { return code; }
};
// act(gate) * up of a paired epilogue, on the float sums
__device__ __forceinline__ float pair_value(float g, float u, const Epi& e) {
  if (e.code == EPI_SWISH_CLAMPED_PAIR) {
    g = fminf(g, e.limit);
    u = fminf(fmaxf(u, -e.limit), e.limit);
    return (g / (1.0f + expf(-e.alpha * g))) * (u + e.shift);
  }
  if (e.code == EPI_RELU_PAIR) return fmaxf(g, 0.f) * u;
  if (e.code == EPI_GELU_PAIR) return 0.5f * g * (1.0f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g))) * u;
  return (g / (1.0f + expf(-g))) * u;
}

// The same where the result is rounded to bfloat16 (up to 2^-8 of it) and a lane has many: the logistic function by the exponential and
// reciprocal instructions.  The exponent's product is rounded before the exponential, so that the error grows with a negative g:
// within (8 + 1.5 |g|) 2^-24 of the value (2^-20.7 near 0, 2^-18.5 at -22, 2^-16.9 at -87), and below -87.3, where the reciprocal's
// sum passes 2^126, the result may be 0 for a value under 2^-119 |u|.  A product of the library's that is stored in bfloat16 ahead of
// the activation rounds g and u to 2^-8 of themselves besides.  A tile of 256 x 256 sums takes 2 us of them, 6 with the functions above.
__device__ __forceinline__ float pair_value_near(float g, float u, const Epi& e) {
  if (e.code == EPI_SILU_PAIR) return g * __builtin_amdgcn_rcpf(1.0f + __expf(-g)) * u;
  return pair_value(g, u, e);
}

// the code with the constants that the next calls of this thread are to use (gemm_bf16.hip, tl_pair_constants)
Epi epi_of(int epilogue);

}  // namespace tl

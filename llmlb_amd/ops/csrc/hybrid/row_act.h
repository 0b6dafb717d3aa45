// What becomes of a product's sums before they are stored: a launch less
// than a kernel of its own, and a pass over memory less.  The sum is rounded
// to bf16 first, as where it is stored for that kernel.  With two matrices,
// gate and up, the rows of up begin at row ``up`` of the weight.
#pragma once
#include "mfma.h"

enum RowKind { PLAIN, RELU2, GELU, SWIGLU, CLAMPED, CAPPED };
struct RowAct {
  int kind;
  int up;      // SWIGLU, CLAMPED: the first row of up
  float a, b;  // CLAMPED: limit, sharpness; CAPPED: cap (0: none)
};
// n / d by the reciprocal, 1.5 units in a float's last place: results are
// bf16, and of 16384 x 7168 none differed.  What divides exactly takes ten
// instructions more of an epilogue that nothing hides.
__device__ __forceinline__ float row_ratio(float n, float d) {
  return n * __builtin_amdgcn_rcpf(d);
}
// gelu, its tanh form: z / (1 + exp(-2 k (z + c z^3))), k = sqrt(2 / pi)
__device__ __forceinline__ float row_gelu(float z) {
  constexpr float k = -2.f * 0.7978845608028654f * LOG2E;
  const float t = z * (k + k * 0.044715f * (z * z));
  return row_ratio(z, 1.f + __builtin_amdgcn_exp2f(t));
}
__device__ __forceinline__ float row_act(const RowAct& act, float z) {
  if (act.kind == RELU2) {
    z = fmaxf(z, 0.f);
    return z * z;
  }
  if (act.kind == GELU) return row_gelu(z);
  if (act.kind == CAPPED && act.a > 0.f) return act.a * tanhf(z / act.a);
  return z;
}
__device__ __forceinline__ float row_gate(const RowAct& act, float g,
                                          float u) {
  if (act.kind == SWIGLU) return row_ratio(g, 1.f + __expf(-g)) * u;
  g = fminf(g, act.a);
  u = fminf(fmaxf(u, -act.a), act.a);
  return row_ratio(g, 1.f + __expf(-act.b * g)) * (u + 1.f);
}
